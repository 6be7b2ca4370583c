"""An individual's iteration does not depend on who shares its launches.

The projection pass takes narrower strips for few individuals per launch. With
P individuals in one launch it uses the wide strips, with `part` the narrow ones
(up to 4 individuals at 256^2, 2 at 384^2 and 512^2; larger grids always take the
wide ones).
Chunks, lanes, handles of one individual and batches of several patterns have to
give every individual the same bits as the whole population in one launch.
"""
import numpy as np
import pytest

from helpers import case
from s_spi_spring_amd import hipcore

pytestmark = pytest.mark.gpu

SIZES = [(256, 9, 2), (384, 8, 2), (512, 5, 2), (768, 4, 1), (1024, 3, 1), (2048, 2, 1)]
ALGS = [("HIO", 0.9), ("RAAR", 0.87), ("ER", 0.0)]


def iterate(hip, amp, rho, supp, alg, beta, chunk=0):
    be = hip.Backend(amp, capacity=len(rho))
    be.set_chunk(chunk * 17 * amp.size)
    be.set_population(rho, supp)
    be.iterate(alg, 3, beta, 0.0)
    out = be.get_population(support=False)
    be.close()
    return out


@pytest.mark.parametrize("n,P,part", SIZES)
@pytest.mark.parametrize("alg,beta", ALGS)
def test_chunks_and_single_handles(hip, n, P, part, alg, beta):
    amp, rho, supp = case(n, P, seed=51)
    whole = iterate(hip, amp, rho, supp, alg, beta)
    assert np.array_equal(iterate(hip, amp, rho, supp, alg, beta, chunk=part), whole)
    for i in (0, P - 1):
        assert np.array_equal(iterate(hip, amp, rho[i:i + 1], supp[i:i + 1], alg, beta)[0], whole[i]), i


@pytest.mark.parametrize("n,P,part", [(384, 3, 2), (384, 8, 4), (512, 3, 2)])
def test_lanes(hip, monkeypatch, n, P, part):
    amp, rho, supp = case(n, P, seed=52)
    out = []
    for lanes in ("1", "2"):
        monkeypatch.setenv("SPR_ITERATE_LANES", lanes)
        out.append(iterate(hip, amp, rho, supp, "RAAR", 0.87))
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("n,pops", [(384, (2, 1)), (384, (4, 4)), (512, (3, 2))])
def test_batch_of_patterns(hip, n, pops):
    cs = [case(n, P, seed=53 + k) for k, P in enumerate(pops)]
    b = hipcore.Batch([c[0] for c in cs], list(pops))
    for k, (_, rho, supp) in enumerate(cs):
        b.set_population(k, rho, supp)
    b.run([("HIO", [3, 0.9]), ("RAAR", [3, 0.87]), ("ER", [2])])
    for k, (amp, rho, supp) in enumerate(cs):
        one = hip.Backend(amp, capacity=len(rho))
        one.set_population(rho, supp)
        one.run([("HIO", [3, 0.9]), ("RAAR", [3, 0.87]), ("ER", [2])])
        assert np.array_equal(b.get_population(k)[0], one.get_population(support=False)), k
        one.close()
    b.close()
