"""Supports that most or all rows meet, in blocks whose row pass runs on listed rows.

Above a share of the rows every row is listed and the column pass projects without
updating any row itself. One individual on each side of that bound, one at it, one
with every row and a sparse one share the launches; results against the FP64 oracle,
as close as the FP32 oracle is within 4x, with the single-step bar of 1e-5 as floor.

The update accepts a pixel or not by whether a phase is pi. Where the FP64 value is
nearer to the negative real axis than four times the FP32 oracle's error, either
decision is right, and the iteration that took the other one ends up to 1e-3 apart
(at 768^2, ER, one pixel of 615 rows does: the same in the form that stores the
state). So a result beyond the bar has to meet it after up to three such decisions,
each the one that brings the FP64 iteration nearest, are taken the other way.
"""
import numpy as np
import pytest

from conftest import rel_l2
from helpers import case

pytestmark = pytest.mark.gpu


def listed_max(n):
    return n - n // 5 if n == 768 else n - n // 8


def iterate64(orc, alg, beta, rho, supp, amp, flips=(), near=None):
    """Two FP64 iterations and the trailing projection, with the decisions (iteration,
    flat pixel) of `flips` taken the other way; `near` collects the undecided ones."""
    b, a64 = rho.astype(np.complex128), amp.astype(np.float64)
    for it in range(2):
        d = orc.ift(orc.project(orc.ft(b), a64))
        z = 2 * d - b if alg == "RAAR" else d
        accept = (supp != 0) & ~((z.real < 0) & (z.imag == 0))
        if near is not None:
            err = np.abs(orc.ift(orc.project(orc.ft(b.astype(np.complex64)), amp)) - d).max()
            close = (supp != 0) & (z.real < 0) & (np.abs(z.imag) <= (12 if alg == "RAAR" else 4) * err)
            near += [(it, i) for i in np.flatnonzero(close)]
        for at, i in flips:
            if at == it:
                accept.flat[i] = not accept.flat[i]
        b = np.where(accept, d, {"ER": 0 * d, "HIO": b - beta * d, "RAAR": beta * b + (1 - 2 * beta) * d}[alg])
    return orc.ift(orc.project(orc.ft(b), a64))


def nearest_decisions(orc, alg, beta, rho, supp, amp, got, bar):
    """Relative L2 to the FP64 iteration after up to three undecided pixels, and these."""
    near, flips = [], []
    e = rel_l2(got, iterate64(orc, alg, beta, rho, supp, amp, near=near))
    while e >= bar and len(flips) < 3:
        tried = [(rel_l2(got, iterate64(orc, alg, beta, rho, supp, amp, flips + [f])), f) for f in near if f not in flips]
        if not tried or min(tried)[0] >= e:
            break
        e, f = min(tried)
        flips.append(f)
    return e, flips


@pytest.mark.parametrize("n", [256, 384, 512, 768, 1024, 2048])
@pytest.mark.parametrize("alg,beta", [("HIO", 0.9), ("RAAR", 0.87), ("ER", 0.0)])
def test_two_iterations(hip, orc, n, alg, beta):
    rows = [listed_max(n) - 1, listed_max(n), listed_max(n) + 1, n, n // 4]
    if n == 2048:
        rows = rows[1:4]
    amp, rho, _ = case(n, len(rows), seed=71)
    supp = np.zeros(rho.shape, np.int32)
    rng = np.random.default_rng(72)
    for i, k in enumerate(rows):
        supp[i, rng.permutation(n)[:k], n // 3:2 * n // 3] = 1
    be = hip.Backend(amp, capacity=len(rows))
    be.set_population(rho, supp)
    be.iterate(alg, 2, beta, 0.0)
    got, s = be.get_population()
    be.close()
    assert np.array_equal(s, supp)
    for i, k in enumerate(rows):
        want = orc.iterate(alg, rho[i:i + 1].astype(np.complex128), supp[i:i + 1], amp.astype(np.float64), 2, beta, 0.0)
        ref32 = orc.iterate(alg, rho[i:i + 1], supp[i:i + 1], amp, 2, beta, 0.0)
        e, e32 = rel_l2(got[i], want[0]), rel_l2(ref32[0], want[0])
        bar = max(1e-5, 4 * e32)
        flips = []
        if e >= bar:
            e, flips = nearest_decisions(orc, alg, beta, rho[i], supp[i], amp, got[i], bar)
        print(f"{alg} n={n} {k} rows: rel-L2 vs fp64 oracle {e:.2e}, fp32 oracle {e32:.2e}, other decisions {flips}", flush=True)
        assert e < bar
