"""The peel with one evaluation per lane (scoring from 16384 evaluations,
the adjoint from 6144) against the workgroup kernels that serve smaller
launches and explicit requests: scoring terms and accumulators bit for bit,
the adjoint's value bit for bit up to the final subtraction and its derivatives
to FP64 rounding of their sums (at most some 1e4 terms of one sign pattern per
parameter: 1e-11 of the largest)."""
import numpy as np
import pytest

from conftest import load_golden, GOLDEN_CASES
from swiftlink_amd import native, synth

pytestmark = pytest.mark.gpu

MODEL = ((0.05, 0.3, 0.85), 0.12)


def _graphs(case, data, n, seed=3):
    rng = np.random.default_rng(seed)
    g = np.repeat(synth.true_graph(data, case)[None], n, axis=0)
    nm = 2 * (case.N - case.F)
    for x in g[1:]:
        x[rng.integers(0, case.M, 40), 2 * case.F + rng.integers(0, nm, 40)] ^= 1
    return g


# evaluations: just over the threshold, a last wavefront of one lane, of 63,
# one position, sixteen positions, more graphs than a wavefront, one graph
@pytest.mark.parametrize("markers,nlod,graphs", ((100, 5, 34), (66, 16, 17), (65, 1, 257), (1094, 3, 5),
                                                 (3279, 5, 1)))
def test_scoring_equals_the_workgroup_kernel(tmp_path, markers, nlod, graphs):
    case, data = synth.make_case("ped30_snp100", str(tmp_path), nlod=nlod, n_markers=markers)
    assert graphs * (markers - 1) * nlod >= 16384
    g = _graphs(case, data, graphs)
    out = []
    for kernel in (native.SL_LOD_AUTO, native.SL_LOD_WORKGROUP):
        with native.Context(case, native.SL_FP64, lod_kernel=kernel) as ctx:
            terms = ctx.lod_terms(g)
            ctx.lod_accumulate(g)
            out.append((terms,) + ctx.lod_results())
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("name", GOLDEN_CASES)
def test_scoring_on_golden_pedigrees(name):
    """Loops and half-sib ships put every kind of op through the kernel."""
    case, fx = load_golden(name)
    n = -(-20000 // ((case.M - 1) * case.nlod))
    g = np.concatenate([fx["graphs"]] * -(-n // len(fx["graphs"])))[:n]
    with native.Context(case, native.SL_FP64) as a, \
            native.Context(case, native.SL_FP64, lod_kernel=native.SL_LOD_WORKGROUP) as b:
        ta, tb = a.lod_terms(g), b.lod_terms(g)
    assert np.array_equal(ta, tb)
    np.testing.assert_allclose(ta[:len(fx["graphs"])], fx["lod_terms"], rtol=1e-12, atol=1e-10)


@pytest.mark.parametrize("config,markers,nlod,graphs", (("ped30_snp100", 100, 5, 13), ("ped30_snp100", 65, 16, 6),
                                                        ("ped150_snp1000", 42, 5, 31), ("ped200_snp2000", 70, 1, 90)))
def test_adjoint_equals_the_workgroup_kernel(tmp_path, config, markers, nlod, graphs):
    case, data = synth.make_case(config, str(tmp_path), nlod=nlod, n_markers=markers)
    assert graphs * (markers - 1) * nlod >= 6144 > (markers - 1) * nlod
    g = _graphs(case, data, graphs)
    with native.Context(case, native.SL_FP64) as ctx:
        for pen, freq in (MODEL, ((0.0, 0.0, 1.0), 0.01)):  # a second model on the same programs
            ctx.set_trait_model(pen, freq)
            got = ctx.trait_grad(g)
            ref = np.concatenate([ctx.trait_grad(x[None]) for x in g])
            assert np.array_equal(np.isfinite(got), np.isfinite(ref))
            ok = np.isfinite(ref[..., 0])
            np.testing.assert_allclose(got[..., 0][ok], ref[..., 0][ok], rtol=1e-14)
            for k in range(1, 7):
                scale = np.abs(ref[..., k]).max()
                assert np.abs(got[..., k] - ref[..., k]).max() <= 1e-11 * scale


def test_captured_scoring(tmp_path):
    """A batch's captured sweep scores its chains in the same kernel."""
    case, data = synth.make_case("ped30_snp100", str(tmp_path))
    g = np.repeat(synth.true_graph(data, case)[None], 36, axis=0)
    accs = []
    for batched in (False, True):
        with native.Context(case, native.SL_FP64) as ctx:
            ctx.mcmc_init(g)
            if batched:
                with native.Batch([ctx]) as b:
                    b.run(6, 0, 2, 0.5, 11)
            else:
                ctx.mcmc_run(6, 0, 2, 0.5, 11)
            accs.append(ctx.lod_results()[0])
    assert np.array_equal(accs[0], accs[1])


# FP32: in the workgroup kernel's arithmetic and exponents (fewer than 32
# graphs): equal bit for bit; and in the FP32 lane kernel's (whole wavefronts of
# graphs, and evaluations in a row), whose tables may take their powers of two
# elsewhere, which moves the rounding of ln L + E ln 2 (|ln L| below 1e3: 1e-12)
@pytest.mark.parametrize("config,markers,nlod,graphs,kernel", (
    ("ped30_snp100", 200, 5, 20, native.SL_LOD_WORKGROUP), ("ped150_snp1000", 66, 16, 17, native.SL_LOD_WORKGROUP),
    ("ped150_snp1000", 300, 5, 64, native.SL_LOD_LANES), ("ped150_snp1000", 300, 5, 63, native.SL_LOD_LANES),
    ("ped150_snp1000", 150, 5, 129, native.SL_LOD_LANES), ("ped150_snp1000", 300, 5, 33, native.SL_LOD_LANES)))
def test_fp32_scoring_is_the_other_kernels(tmp_path, config, markers, nlod, graphs, kernel):
    case, data = synth.make_case(config, str(tmp_path), nlod=nlod, n_markers=markers)
    assert graphs * (markers - 1) * nlod >= 16384
    g = _graphs(case, data, graphs)
    out = []
    for k in (native.SL_LOD_AUTO, kernel):
        with native.Context(case, native.SL_FP32_RESCALED, lod_kernel=k) as ctx:
            assert ctx.lod_kernel_for(graphs) == kernel
            terms = ctx.lod_terms(g)
            ctx.lod_accumulate(g)
            out.append((terms, ctx.lod_results()[0]))
    for a, b in zip(*out):
        assert np.array_equal(a, b) if kernel == native.SL_LOD_WORKGROUP else np.abs(a - b).max() < 1e-12


def test_allocation_free_sums_are_the_same(tmp_path):
    """96 graphs: summed in the wavefronts without an array for the terms."""
    import torch
    from swiftlink_amd.case import pack_graphs
    case, data = synth.make_case("ped150_snp1000", str(tmp_path), n_markers=300)
    g = _graphs(case, data, 96)
    dev = torch.from_numpy(pack_graphs(case, g).reshape(-1).view(np.int32)).cuda()
    with native.Context(case, native.SL_FP32_RESCALED) as ctx:
        ctx.lod_accumulate_packed(dev.data_ptr(), 96)
        a = ctx.lod_results()[0]
        ctx.lod_reset()
        ctx.lod_accumulate_packed_noalloc(dev.data_ptr(), 96)
        assert np.array_equal(a, ctx.lod_results()[0])
