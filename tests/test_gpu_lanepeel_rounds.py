"""The lane peel in more evaluations than one round of its wavefronts takes (3072
of them in FP64, 4096 in FP32, 2048 in the adjoint, 64 evaluations each), by numbers
that leave a last wavefront partly empty, against the kernels it stands in for:
each wavefront goes through its table slot and columns again."""
import numpy as np
import pytest

from swiftlink_amd import native, synth
from test_gpu_lanepeel import MODEL, _graphs

pytestmark = pytest.mark.gpu


def _terms(case, g, precision, kernel):
    with native.Context(case, precision, lod_kernel=kernel) as ctx:
        terms = ctx.lod_terms(g)
        ctx.lod_accumulate(g)
        return terms, ctx.lod_results()[0]


@pytest.mark.parametrize("config,markers,nlod,graphs", (("ped30_snp100", 1094, 3, 61), ("ped200_snp2000", 401, 5, 99)))
def test_fp64_rounds(tmp_path, config, markers, nlod, graphs):
    case, data = synth.make_case(config, str(tmp_path), nlod=nlod, n_markers=markers)
    E = graphs * (markers - 1) * nlod
    assert E > 3072 * 64 and E % 64
    g = _graphs(case, data, graphs)
    for a, b in zip(_terms(case, g, native.SL_FP64, native.SL_LOD_AUTO),
                    _terms(case, g, native.SL_FP64, native.SL_LOD_WORKGROUP)):
        assert np.array_equal(a, b)


# the workgroup kernel's order: equal bits; the lane kernel's: to the rounding of
# ln L + E ln 2 (|ln L| below 1e3)
@pytest.mark.parametrize("markers,nlod,graphs,kernel", (
    (2906, 5, 19, native.SL_LOD_WORKGROUP), (3002, 3, 64, native.SL_LOD_LANES), (3002, 3, 59, native.SL_LOD_LANES)))
def test_fp32_rounds(tmp_path, markers, nlod, graphs, kernel):
    case, data = synth.make_case("ped30_snp100", str(tmp_path), nlod=nlod, n_markers=markers)
    if kernel == native.SL_LOD_WORKGROUP:
        pairs = 64 // nlod
        assert graphs * (markers - 1) > 4096 * pairs and graphs * (markers - 1) % pairs
    else:
        assert (markers - 1) * nlod > 2 * 4096 and (markers - 1) * nlod * graphs % (4096 * 64)
    g = _graphs(case, data, graphs)
    with native.Context(case, native.SL_FP32_RESCALED) as ctx:
        assert ctx.lod_kernel_for(graphs) == kernel
    for a, b in zip(_terms(case, g, native.SL_FP32_RESCALED, native.SL_LOD_AUTO),
                    _terms(case, g, native.SL_FP32_RESCALED, kernel)):
        assert np.array_equal(a, b) if kernel == native.SL_LOD_WORKGROUP else np.abs(a - b).max() < 1e-12


def test_adjoint_rounds(tmp_path):
    """The workgroup kernel serves a graph at a time (its sums of at most some 1e4
    terms: 1e-11 of the largest)."""
    case, data = synth.make_case("ped30_snp100", str(tmp_path), nlod=3, n_markers=1094)
    g = _graphs(case, data, 41)
    per = (case.M - 1) * 3
    assert 41 * per > 2048 * 64 and 41 * per % 64 and per < 6144
    with native.Context(case, native.SL_FP64) as ctx:
        ctx.set_trait_model(*MODEL)
        got = ctx.trait_grad(g)
        ref = np.concatenate([ctx.trait_grad(x[None]) for x in g])
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    ok = np.isfinite(ref[..., 0])
    np.testing.assert_allclose(got[..., 0][ok], ref[..., 0][ok], rtol=1e-14)
    for k in range(1, 7):
        assert np.abs(got[..., k] - ref[..., k]).max() <= 1e-11 * np.abs(ref[..., k]).max()
