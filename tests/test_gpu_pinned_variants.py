"""A column variant that the caller sets, or the autotuner picks, runs as itself.

A handle with the compiled choice may run its plain projections (the trailing one
of a block, shrink-wrap) in another variant than its iterations; a handle whose
variants were set must not, else a variant's tests and timings are another's.
"""
import pytest

from helpers import case
from s_spi_spring_amd import hipcore

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [128, 256, 512])
def test_set_variants_run_as_they_are(hip, n):
    amp, rho, supp = case(n, 1, seed=61)
    be = hip.Backend(amp, capacity=1)
    nc, _ = hipcore.variant_counts(n)
    assert be.variants() == hipcore.default_variants(n)
    for col in range(nc):
        be.set_variants(col, be.variants()[1])
        assert be.variants()[0] == col and be.plain_variant() == col
    be.close()


def test_process_defaults_and_autotune_run_as_they_are(hip):
    n = 512
    before = hipcore.default_variants(n)
    amp, rho, supp = case(n, 1, seed=62)
    hipcore.set_default_variants(n, *before)
    be = hip.Backend(amp, capacity=1)
    assert be.variants() == before and be.plain_variant() == before[0]
    be.set_population(rho, supp)
    be.autotune(reps=1)
    assert be.plain_variant() == be.variants()[0]
    be.close()
    hipcore.set_default_variants(n, *before)
