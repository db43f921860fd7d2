"""Families whose workgroups come within a few hundred bytes of the 160 KiB of LDS:
a kernel's own arrays count besides what its launch asks for, and where both do
not fit the steps take the form that needs less."""
import dataclasses

import numpy as np
import pytest

from family_cases import family_case, line_family
from oracle_lib import Oracle
from swiftlink_amd import linkage, native
from test_gpu_lsampler import _check_fp32_sweep, oracle_lsweep

pytestmark = pytest.mark.gpu

KIB160 = 160 * 1024


def likelihood_lds(N, F, threads):
    """Dynamic LDS of the likelihood jobs (msampler_lds_bytes)."""
    in_registers = max(N, 2 * F) <= 1024
    wave = 4 * (-(-2 * (N - F) // 32)) + 16 * F + 4 * N + 4 * (N if in_registers else N - F)
    return -(-8 * (N - F) // 16) * 16 + threads // 64 * (-(-wave // 16) * 16)


@pytest.mark.parametrize("people,founders,threads,chains", ((819, 200, 1024, 700), (1978, 200, 512, 1)))
def test_passes_beside_jobs_near_the_limit(people, founders, threads, chains):
    assert KIB160 - threads // 64 * 40 < likelihood_lds(people, founders, threads) <= KIB160
    M = 6
    case, g0 = family_case(markers=M, missing=0.0, seed=3, minor=np.full(M, 0.02), tries=1,
                           **line_family(people, founders))
    o = Oracle(case)
    order = np.random.default_rng(people).choice(o.meioses(), 40, replace=False).astype(np.int32)
    parent = np.where(order % 2, case.father[founders + order // 2], case.mother[founders + order // 2])
    jobs = ((case.legal[parent] & 12) != 0).sum() / len(order)  # at most: a parent that may be heterozygous
    if chains > 1:  # the sizes for which the pass runs beside the jobs
        assert 0 < jobs * chains * 16 <= 12288 and 2 * chains * M > 8192
    out = []
    for mode in (native.SL_MSAMPLER_AUTO, native.SL_MSAMPLER_TWO_LAUNCH):
        with native.Context(case, native.SL_FP64, msampler_mode=mode) as ctx:
            ctx.mcmc_init(np.repeat(g0[None], chains, axis=0))
            ctx.profile(True)
            ctx.msweep(31, 0, order)
            assert ctx.profile_read(native.SL_KERNEL_MSAMPLER_FB)[1] == len(order)  # two launches a step
            ctx.profile(False)
            assert np.all(ctx.mcmc_status() == 0)
            assert ctx.mcmc_near_edge()[0] == 0
            out.append(ctx.mcmc_graphs())
    assert np.array_equal(out[0], out[1])
    assert np.array_equal(out[0][0], o.msweep(g0, order, 31, 0, 0))


def test_kept_products_at_the_limit():
    """A locus whose tables and kept products leave an L-sampler workgroup not one
    byte: 6952 cells of five FP32 entries and the rest of its arrays."""
    N, F, at, cells = 497, 133, 553, 6952
    case, g = family_case(markers=2000, missing=0.95, seed=1, tries=1, **line_family(N, F))
    minor = case.minor[[at] * 4]
    geno = np.ascontiguousarray(case.geno[:, [at] * 4])
    case = dataclasses.replace(case, M=4, geno=geno, minor=minor, theta=case.theta[:3], partial_theta=case.partial_theta[:3],
                               geno_prob=linkage.sampler_cache(geno, minor),
                               legal=linkage.eliminate(geno, case.mother, case.father, F))
    g0 = np.ascontiguousarray(g[[at] * 4])
    legal = np.array([bin(x & 15).count("1") for x in case.legal[:, 0]])
    tables = sum(int(np.prod(legal[case.ops.cutset(o)], dtype=int)) for o in range(case.ops.n))
    assert -(-tables // 8) * 8 == cells
    rest = 8 * (N + 2 * (N - F) + 4) + 4 * (8 * (N - F) + 20) + 4 * (N + 4) + N + 2 * (N - F)
    assert KIB160 - 16 < 4 * 5 * cells + rest <= KIB160
    o = Oracle(case)
    with native.Context(case, native.SL_FP32_RESCALED) as ctx:
        ctx.mcmc_init(np.stack([g0, g0]))
        ctx.lsweep(77, 0, 0)
        out = ctx.mcmc_graphs()
        near = ctx.mcmc_near_edge_loci()
        assert np.all(ctx.mcmc_status() == 0)
    for c in range(2):
        _check_fp32_sweep(case, out[c], oracle_lsweep(o, g0, case.M, 77, c, 0, 0), near[c], 0)
