"""The projection pass of the listed-row iteration (k_col_step) in every column variant.

Each column variant runs with a row variant that recomputes the state, two iterations
on supports of every kind (a full row and a corner pixel, the last pixel, rows apart
from each other, every row), against the FP64 oracle: as close as the FP32 oracle is
within 4x, with the single-step bar of 1e-5 as floor; pixels whose acceptance is
within rounding may go either way (decisions.py). One individual alone, in whatever
strips such a launch takes, has the bits it has among the others.
"""
import numpy as np
import pytest

from conftest import rel_l2
from decisions import nearest_decisions
from helpers import case
from s_spi_spring_amd import hipcore

pytestmark = pytest.mark.gpu

SIZES = [256, 384, 512, 768, 1024, 2048]


def supports(n, P):
    s = np.zeros((4, n, n), np.int32)
    s[0, 0, n // 3] = 1
    s[0, n // 2, :] = 1
    s[1, 2:n:7, n // 4:3 * n // 4] = 1
    s[1, n - 1, n - 1] = 1
    s[2, n // 3:n // 3 + n // 4, n // 3:2 * n // 3] = 1
    s[3, :, n // 2:n // 2 + 9] = 1
    return s[[1, 3]] if P == 2 else s


def recomputing(n):
    return [r for r in range(hipcore.variant_counts(n)[1]) if hipcore.row_variant_recomputes_state(n, r)]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("alg,beta", [("HIO", 0.9), ("RAAR", 0.87), ("ER", 0.0)])
def test_every_column_variant(hip, orc, n, alg, beta):
    P = 4 if n < 2048 else 2
    amp, rho, _ = case(n, P, seed=91)
    supp = supports(n, P)
    want = orc.iterate(alg, rho.astype(np.complex128), supp, amp.astype(np.float64), 2, beta, 0.0)
    ref32 = orc.iterate(alg, rho, supp, amp, 2, beta, 0.0)
    row = recomputing(n)[0]
    for col in range(hipcore.variant_counts(n)[0]):
        out = []
        for sl in (slice(0, P), slice(0, 1)):
            be = hip.Backend(amp, capacity=P)
            be.set_variants(col, row)
            be.set_population(rho[sl], supp[sl])
            be.iterate(alg, 2, beta, 0.0)
            out.append(be.get_population(support=False))
            be.close()
        assert np.array_equal(out[0][:1], out[1]), (n, col)
        for i in range(P):
            e, e32 = rel_l2(out[0][i], want[i]), rel_l2(ref32[i], want[i])
            bar, flips = max(1e-5, 4 * e32), []
            if e >= bar:
                e, flips = nearest_decisions(orc, alg, beta, rho[i], supp[i], amp, out[0][i], bar)
            print(f"{alg} n={n} column variant {col} individual {i}: rel-L2 vs fp64 oracle {e:.2e}, fp32 oracle "
                  f"{e32:.2e}, other decisions {flips}", flush=True)
            assert e < bar


@pytest.mark.parametrize("n", SIZES)
def test_every_row_variant_with_the_compiled_column_variant(hip, orc, n):
    amp, rho, _ = case(n, 2, seed=92)
    supp = supports(n, 2)
    want = orc.iterate("RAAR", rho.astype(np.complex128), supp, amp.astype(np.float64), 2, 0.87, 0.0)
    ref32 = orc.iterate("RAAR", rho, supp, amp, 2, 0.87, 0.0)
    col = hipcore.default_variants(n)[0]
    for row in recomputing(n):
        be = hip.Backend(amp, capacity=2)
        be.set_variants(col, row)
        be.set_population(rho, supp)
        be.iterate("RAAR", 2, 0.87, 0.0)
        got = be.get_population(support=False)
        be.close()
        for i in range(2):
            e, e32 = rel_l2(got[i], want[i]), rel_l2(ref32[i], want[i])
            bar, flips = max(1e-5, 4 * e32), []
            if e >= bar:
                e, flips = nearest_decisions(orc, "RAAR", 0.87, rho[i], supp[i], amp, got[i], bar)
            print(f"n={n} row variant {row} individual {i}: rel-L2 {e:.2e}, fp32 oracle {e32:.2e}, other decisions {flips}",
                  flush=True)
            assert e < bar
