"""Iteration blocks whose row pass visits only the rows that meet the support.

A population with a different support in every individual: one full row and one
pixel in the first row, a pixel in the last row, rows that are not adjacent, and
every row. Bar: that of the multi-iteration tests, as close to the FP64 oracle as
the FP32 oracle is within 4x, with the single-step bar of 1e-5 as its floor.
"""
import numpy as np
import pytest

from conftest import rel_l2
from helpers import case

pytestmark = pytest.mark.gpu


def supports(n, disk):
    s = np.zeros((4, n, n), np.int32)
    s[0, 0, n // 3] = 1
    s[0, n // 2, :] = 1
    s[1, n - 1, n - 1] = 1
    s[1, 5, 3:n // 2] = 1
    s[2, 3:n:7, n // 4:3 * n // 4] = 1
    s[3] = disk
    s[3, :, n // 2] = 1
    return s


@pytest.mark.parametrize("n", [64, 128, 256, 384, 512, 768, 1024])
@pytest.mark.parametrize("alg,beta", [("HIO", 0.9), ("RAAR", 0.87), ("ER", 0.0)])
def test_two_iterations_by_rows(hip, orc, n, alg, beta):
    amp, rho, disk = case(n, 4, seed=17)
    supp = supports(n, disk[0])
    be = hip.Backend(amp, capacity=4)
    if n <= 128:
        be.set_fused(1)     # on chip: wavefronts of eight (128^2) or sixteen (64^2) rows
    be.set_population(rho, supp)
    be.iterate(alg, 2, beta, 0.0)
    got, s = be.get_population()
    be.close()
    assert np.array_equal(s, supp)
    want = orc.iterate(alg, rho.astype(np.complex128), supp, amp.astype(np.float64), 2, beta, 0.0)
    ref32 = orc.iterate(alg, rho, supp, amp, 2, beta, 0.0)
    for i in range(4):
        e, e32 = rel_l2(got[i], want[i]), rel_l2(ref32[i], want[i])
        print(f"{alg} n={n} individual {i}: rel-L2 vs fp64 oracle {e:.2e}, fp32 oracle {e32:.2e}")
        assert e < max(1e-5, 4 * e32)


@pytest.mark.parametrize("n,stored", [(256, 2), (512, 0), (1024, 0)])
def test_empty_support_as_the_stored_state(hip, n, stored):
    """ER empties a density whose support is empty, and the projection of the
    vanishing spectrum takes its phases from the signs of its zeros: both forms
    run the same transforms on the same zeros."""
    amp, rho, _ = case(n, 1, seed=18)
    out = []
    for row in (None, stored):
        be = hip.Backend(amp, capacity=1)
        if row is not None:
            be.set_variants(0, row)
        be.set_population(rho, np.zeros((1, n, n), np.int32))
        be.iterate("ER", 1, 0.0, 0.0)
        out.append(be.get_population(support=False))
        be.close()
    assert rel_l2(out[0], out[1]) < 1e-6
