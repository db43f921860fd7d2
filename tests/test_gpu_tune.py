"""The autotuner does not leave a context on a shape that is slower than the
library's own choice."""
import numpy as np
import pytest

from swiftlink_amd import native, synth, tune

LOD = {(64, 1, native.SL_LOD_WORKGROUP): 2.0, (64, 4, native.SL_LOD_WORKGROUP): 1.0}
AUTO = (64, 1, native.SL_LOD_AUTO)


@pytest.mark.parametrize("auto_ms,picks", ((0.5, True), (1.0, True), (1.02, True), (1.1, False)))
def test_an_explicit_shape_has_to_be_faster(auto_ms, picks):
    assert (tune._fastest({**LOD, AUTO: auto_ms}, AUTO) == AUTO) is picks


def test_without_the_librarys_choice():
    assert tune._fastest(LOD, AUTO) == (64, 4, native.SL_LOD_WORKGROUP)


@pytest.mark.gpu
def test_autotune_keeps_the_lane_peel(tmp_path):
    """64 FP64 chains of 150 people: one evaluation per lane scores them several
    times faster than any shape of the workgroup kernel."""
    case, data = synth.make_case("ped150_snp1000", str(tmp_path), n_markers=300)
    starts = np.repeat(synth.true_graph(data, case)[None], 64, axis=0)
    with native.Context(case, native.SL_FP64) as ctx:
        ctx.mcmc_init(starts)
        tu = tune.autotune(ctx, blocks=(128, 256), gpws=(1, 4))
        print(tu)
        assert tu["lod_kernel"] == native.SL_LOD_AUTO and ctx.options["lod_kernel"] == native.SL_LOD_AUTO
        assert tu["lod_ms"]["auto"] < 0.5 * min(v for k, v in tu["lod_ms"].items() if k != "auto")
        assert native.SL_MSAMPLER_AUTO in tu["msweep_ms"]
        limit = (1.0 + tune.AUTO_MARGIN) * min(tu["msweep_ms"].values())
        assert tu["msweep_ms"][tu["msampler_mode"]] <= limit
        assert np.array_equal(ctx.mcmc_graphs(), starts)
