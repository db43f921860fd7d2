"""Loci whose minor allele has frequency 0 or 1: one of the allele log-frequencies
is infinite there.  Where nobody is genotyped, or every genotype is of the allele
that exists, the locus's founder-allele likelihood is 1 and the M-sampler goes
through it as through any other."""
import dataclasses

import numpy as np
import pytest

from family_cases import family_case
from oracle_lib import Oracle
from swiftlink_amd import linkage, native
from test_gpu_msweep_order import WIDE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graphs", (0, native.SL_MSAMPLER_LDS_GRAPHS))
@pytest.mark.parametrize("mode,chains", ((native.SL_MSAMPLER_SPECULATIVE, 2), (native.SL_MSAMPLER_TWO_LAUNCH, 3),
                                         (native.SL_MSAMPLER_AUTO, 70)))
def test_loci_of_one_allele(mode, chains, graphs):
    M = 65
    minor = np.full(M, 0.3)
    minor[10:20], minor[30:40] = 0.0, 1.0
    case, g0 = family_case(markers=M, missing=0.3, seed=5, minor=minor, **WIDE)
    assert set(case.geno[:, 10:20].ravel()) == {linkage.UNTYPED, linkage.HOMOZ_A}
    assert set(case.geno[:, 30:40].ravel()) == {linkage.UNTYPED, linkage.HOMOZ_B}
    geno = case.geno.copy()
    geno[:, 15:20] = geno[:, 35:40] = linkage.UNTYPED
    case = dataclasses.replace(case, geno=geno, legal=linkage.eliminate(geno, case.mother, case.father, case.F),
                               geno_prob=linkage.sampler_cache(geno, minor))
    o = Oracle(case)
    order = o.meioses()
    with native.Context(case, native.SL_FP64, msampler_mode=mode | graphs) as ctx:
        ctx.mcmc_init(np.repeat(g0[None], chains, axis=0))
        lik = ctx.mcmc_likelihood()
        for sweep in range(2):
            ctx.msweep(9, sweep, order)
        out = ctx.mcmc_graphs()
        assert np.all(ctx.mcmc_status() == 0)
        assert ctx.mcmc_near_edge()[0] == 0
    assert np.all(lik[:, 10:20] == 1.0) and np.all(lik[:, 30:40] == 1.0)
    for c in (0, chains - 1):
        g = g0
        for sweep in range(2):
            g = o.msweep(g, order, 9, c, sweep)
        assert np.array_equal(out[c], g), c
