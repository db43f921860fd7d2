"""Device memory of a context: what its optional buffers take, and that calls give
the same results as these come and go."""
import numpy as np
import pytest

from family_cases import family_case, line_family, locus_cells
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


def test_terms_of_a_long_map_take_no_array(tmp_path):
    """400 graphs of 100000 positions: 320 MB of terms, which the wavefronts sum
    themselves, as the FP32 lane kernel's do (equal to the rounding of ln L + E ln 2,
    |ln L| below 1e3)."""
    import torch
    from swiftlink_amd.case import pack_graphs
    case, data = synth.make_case("ped30_snp100", str(tmp_path), n_markers=20001)
    n = 400
    g = _graphs(case, data, 20)
    dev = torch.from_numpy(pack_graphs(case, g).reshape(20, -1).view(np.int32)).cuda()
    dev = dev[torch.arange(n, device="cuda") % 20].contiguous()
    torch.cuda.synchronize()
    out = []
    for kernel in (native.SL_LOD_AUTO, native.SL_LOD_LANES):
        with native.Context(case, native.SL_FP32_RESCALED, lod_kernel=kernel) as ctx:
            free = torch.cuda.mem_get_info()[0]
            ctx.lod_accumulate_packed(dev.data_ptr(), n)
            out.append(ctx.lod_results()[0])
            assert free - torch.cuda.mem_get_info()[0] < 64 * MIB
    assert np.abs(out[0] - out[1]).max() < 1e-12


def test_batches_allocate_the_tables_they_use():
    """300 people, hardly typed, in FP64: tables and kept products pass LDS, so the
    decoding L-sampler would keep both in 2048 slots of global memory (at least
    5 x 8 bytes x 3500 cells each, 286 MB); the record form that runs has no slots."""
    import torch
    case, g0 = family_case(markers=50, missing=0.95, seed=1, tries=1, **line_family(300, 80))
    legal = np.array([bin(x).count("1") for x in range(16)])[case.legal & 15]
    cells = sum(np.prod(legal[case.ops.cutset(o)], axis=0, dtype=int) for o in range(case.ops.n))
    assert 5 * 8 * cells.max() > 160 * 1024
    with native.Context(case, native.SL_FP64) as ctx:
        ctx.mcmc_init(np.stack([g0, g0]))
        ctx.lod_reset()
        with native.Batch([ctx]) as b:
            free = torch.cuda.mem_get_info()[0]
            b.run(4, 0, 2, 0.5, 7)
            assert free - torch.cuda.mem_get_info()[0] < 128 * MIB
        out = ctx.mcmc_graphs()
        assert np.all(ctx.mcmc_status() == 0)
    with native.Context(case, native.SL_FP64) as ctx:
        ctx.mcmc_init(np.stack([g0, g0]))
        ctx.lod_reset()
        ctx.mcmc_run(4, 0, 2, 0.5, 7)
        assert np.array_equal(out, ctx.mcmc_graphs())


def test_sampler_tables_come_with_the_chains():
    """4000 cells of 128 bytes of records at each of 400 loci, 200 MB, and the flip
    classes: a context that only scores has none of them; the first chains, or the
    first replicates, bring them."""
    import torch
    case, g0 = family_case(markers=400, missing=0.95, seed=1, tries=1, **line_family(300, 80))
    records = 128 * int(locus_cells(case).sum())
    assert records > 128 * MIB
    free = lambda: torch.cuda.mem_get_info()[0]
    for first in ("chains", "replicates"):
        with native.Context(case, native.SL_FP32_RESCALED) as ctx:
            ctx.lod_terms(g0[None])
            before = free()
            if first == "chains":
                ctx.mcmc_init(g0[None])
            else:
                ctx.sequential_imputation(1, 1)
            after = free()
            assert before - after >= records
            ctx.sequential_imputation(1, 1)  # there already
            ctx.mcmc_init(g0[None])
            assert after - free() < 32 * MIB
