"""M-sweeps of several chains over maps whose forward-backward passes take two and
four loci a thread, and past 4096 loci, where they draw their own uniforms: beside
the next step's jobs where they fit, and after them."""
import numpy as np
import pytest

from oracle_lib import Oracle
from swiftlink_amd import native, synth
from test_gpu_msampler import shuffled_order

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("markers", (1025, 2048, 2049, 4096, 4097))
def test_maps_past_a_thread_per_locus(tmp_path, markers):
    case, data = synth.make_case("ped30_snp100", str(tmp_path), n_markers=markers)
    g0 = synth.true_graph(data, case)
    o = Oracle(case)
    chains = 5
    assert 2 * chains * markers > 8192
    out = {}
    for precision in (native.SL_FP64, native.SL_FP32_RESCALED):
        for mode in (native.SL_MSAMPLER_AUTO, native.SL_MSAMPLER_TWO_LAUNCH):
            with native.Context(case, precision, msampler_mode=mode) as ctx:
                ctx.mcmc_init(np.repeat(g0[None], chains, axis=0))
                ctx.profile(True)
                ctx.msweep(61, 4)
                passes = ctx.profile_read(native.SL_KERNEL_MSAMPLER_FB)[1]
                ctx.profile(False)
                # launches of a pass alone: none where the passes run beside the jobs
                beside = mode == native.SL_MSAMPLER_AUTO and markers <= 4096
                assert passes == (0 if beside else len(o.meioses()))
                assert np.all(ctx.mcmc_status() == 0)
                near = ctx.mcmc_near_edge()
                out[precision, mode] = ctx.mcmc_graphs(), near
        a, b = (out[precision, m] for m in (native.SL_MSAMPLER_AUTO, native.SL_MSAMPLER_TWO_LAUNCH))
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    graphs, near = out[native.SL_FP64, native.SL_MSAMPLER_AUTO]
    for c in (0, chains - 1):
        assert near[c] == 0
        assert np.array_equal(graphs[c], o.msweep(g0, shuffled_order(o, 61, c, 4), 61, c, 4)), c
