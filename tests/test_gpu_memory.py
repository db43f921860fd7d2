"""Device memory of a context: what its optional buffers take, and that calls give
the same results as these come and go."""
import numpy as np
import pytest

from swiftlink_amd import native, synth
from test_gpu_lanepeel import MODEL, _graphs

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def test_scoring_before_and_after_a_gradient(tmp_path):
    """Scoring and the adjoint, both one evaluation per lane, have table slots of
    their own: a gradient leaves scoring's as they are."""
    case, data = synth.make_case("ped30_snp100", str(tmp_path))
    g = _graphs(case, data, 40)
    with native.Context(case, native.SL_FP64) as ctx:
        ctx.set_trait_model(*MODEL)
        before = ctx.lod_terms(g)
        grad = ctx.trait_grad(g)
        assert np.array_equal(ctx.lod_terms(g), before)
        assert np.array_equal(ctx.trait_grad(g), grad)
    ok = np.isfinite(before)
    assert ok.any()
    np.testing.assert_allclose(grad[..., 0][ok], before[ok], rtol=1e-14)
