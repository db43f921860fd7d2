"""Families whose workgroups come within a few hundred bytes of the 160 KiB of LDS:
a kernel's own arrays count besides what its launch asks for, and where both do
not fit the steps take the form that needs less."""
import numpy as np
import pytest

from family_cases import family_case, line_family
from oracle_lib import Oracle
from swiftlink_amd import native

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
            ctx.msweep(31, 0, order)
            assert np.all(ctx.mcmc_status() == 0)
            assert ctx.mcmc_near_edge()[0] == 0
            out.append(ctx.mcmc_graphs())
    assert np.array_equal(out[0], out[1])
    assert np.array_equal(out[0][0], o.msweep(g0, order, 31, 0, 0))
