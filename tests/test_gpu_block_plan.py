"""What a block of the listed-row iteration prepares from the supports, per block.

The lists are made by the first row pass of every block, so that a handle whose
supports change between two blocks runs the second as a fresh handle would, bit for
bit; in chunks and lanes each part lists its own individuals' rows. A block without
iterations needs no lists and is one projection.
"""
import numpy as np
import pytest

from conftest import rel_l2
from helpers import case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [256, 384, 512, 768, 1024])
@pytest.mark.parametrize("alg,beta", [("HIO", 0.9), ("RAAR", 0.87), ("ER", 0.0)])
def test_supports_that_change_between_blocks(hip, n, alg, beta):
    P = 3
    amp, rho, disk = case(n, P, seed=81)
    other = np.zeros_like(disk)
    other[0, n // 2:n // 2 + 9, :] = 1
    other[1, ::3, ::2] = 1
    other[2, :, n // 3] = 1
    be = hip.Backend(amp, capacity=P)
    be.set_population(rho, disk)
    be.iterate(alg, 2, beta, 0.0)
    mid = be.get_population(support=False)
    be.set_population(mid, other)
    be.iterate(alg, 0, beta, 0.0)
    be.set_population(mid, other)
    be.iterate(alg, 2, beta, 0.0)
    got = be.get_population(support=False)
    be.close()
    fresh = hip.Backend(amp, capacity=P)
    fresh.set_chunk(17 * n * n)
    fresh.set_population(mid, other)
    fresh.iterate(alg, 2, beta, 0.0)
    assert np.array_equal(fresh.get_population(support=False), got)
    fresh.close()


@pytest.mark.parametrize("n", [256, 512, 768, 1024, 2048])
@pytest.mark.parametrize("alg,beta", [("HIO", 0.9), ("RAAR", 0.87), ("ER", 0.0)])
def test_no_iterations_is_one_projection(hip, orc, n, alg, beta):
    amp, rho, supp = case(n, 1, seed=82)
    be = hip.Backend(amp, capacity=1)
    be.set_population(rho, supp)
    be.iterate(alg, 0, beta, 0.0)
    got, s = be.get_population()
    be.close()
    assert np.array_equal(s, supp)
    want = orc.ift(orc.project(orc.ft(rho[0].astype(np.complex128)), amp.astype(np.float64)))
    assert rel_l2(got[0], want) < 1e-5


@pytest.mark.parametrize("n", [256, 512])
def test_lanes_list_their_own_rows(hip, monkeypatch, n):
    amp, rho, _ = case(n, 4, seed=83)
    supp = np.zeros(rho.shape, np.int32)
    for i in range(4):
        supp[i, 5 + 11 * i:n // 2 + 7 * i, n // 4:n // 2] = 1
    out = []
    for lanes in ("1", "2"):
        monkeypatch.setenv("SPR_ITERATE_LANES", lanes)
        be = hip.Backend(amp, capacity=4)
        be.set_population(rho, supp)
        be.iterate("RAAR", 3, 0.87, 0.0)
        be.iterate("ER", 2, 0.0, 0.0)
        out.append(be.get_population(support=False))
        be.close()
    assert np.array_equal(out[0], out[1])
