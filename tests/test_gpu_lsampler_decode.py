"""The L-sampler's decoding kernel, which serves families the task records do not
hold (here an op that consumes five or six tables: a couple's children peeled side
by side), with its tables in LDS and in global memory, against the oracle; and the
record form's two ways of sampling, whose graphs are the same bit for bit."""
import numpy as np
import pytest

from family_cases import family_case, line_family, locus_cells, unchained
from oracle_lib import Oracle
from swiftlink_amd import native
from test_gpu_lsampler import _check_fp32_sweep, oracle_lsweep

pytestmark = pytest.mark.gpu

KIB160 = 160 * 1024


def _decoded(people, founders, markers, missing, seed=1):
    case, g0 = family_case(markers=markers, missing=missing, seed=seed, tries=4, **line_family(people, founders))
    case = unchained(case)
    assert max(len(case.ops.prevs(o)) for o in range(case.ops.n)) > 3  # past a task record
    return case, g0, Oracle(case)


def _sweep(case, graphs, precision, seed, sweep, parity):
    with native.Context(case, precision) as ctx:
        ctx.mcmc_init(graphs)
        ctx.lsweep(seed, sweep, parity)
        assert np.all(ctx.mcmc_status() == 0)
        return ctx.mcmc_graphs(), ctx.mcmc_near_edge_loci()


def test_many_consumed_tables():
    case, g0, o = _decoded(40, 8, 41, 0.2)
    out, near = _sweep(case, np.stack([g0] * 3), native.SL_FP64, 8, 1, 1)
    assert not near.any()
    for c in range(3):
        assert np.array_equal(out[c], oracle_lsweep(o, g0, case.M, 8, c, 1, 1)), c
    with native.Context(case, native.SL_FP64) as ctx:
        best, weights, index, graphs = ctx.sequential_imputation(3, 4, all_graphs=True)
    for r in range(4):
        g, w = o.impute(3, r)
        assert np.array_equal(graphs[r], g) and abs(weights[r] / w - 1.0) < 1e-12, r


def test_narrow_shape_matches_wide():
    """One FP32 chain of 1000 loci makes 500 workgroups of 512 threads, two make
    1000 of 256: chain 0 draws the same stream in both."""
    case, g0, o = _decoded(150, 30, 1000, 0.1)
    assert locus_cells(case).max() < 8 * case.ops.n
    one, _ = _sweep(case, g0[None], native.SL_FP32_RESCALED, 91, 2, 1)
    two, near = _sweep(case, np.stack([g0, g0]), native.SL_FP32_RESCALED, 91, 2, 1)
    assert np.array_equal(two[0], one[0])
    assert np.any(two[1] != two[0])
    _check_fp32_sweep(case, two[1], oracle_lsweep(o, g0, case.M, 91, 1, 2, 1), near[1], 1)


@pytest.mark.parametrize("precision,people,founders,chains", ((native.SL_FP64, 330, 60, 700),
                                                              (native.SL_FP32_RESCALED, 640, 116, 2)))
def test_tables_in_global_memory(precision, people, founders, chains):
    """Hardly typed families whose tables and products pass LDS; 700 chains take
    more workgroups than there are slots."""
    case, g0, o = _decoded(people, founders, 6, 0.95)
    esz = 8 if precision == native.SL_FP64 else 4
    assert 5 * esz * locus_cells(case).max() > KIB160
    out, near = _sweep(case, np.repeat(g0[None], chains, axis=0), precision, 13, 0, 0)
    for c in sorted({0, 1, chains - 1}):
        ref = oracle_lsweep(o, g0, case.M, 13, c, 0, 0)
        if precision == native.SL_FP64:
            assert not near[c].any() and np.array_equal(out[c], ref), c
        else:
            _check_fp32_sweep(case, out[c], ref, near[c], 0)


@pytest.mark.parametrize("precision,people,founders", ((native.SL_FP64, 200, 55), (native.SL_FP32_RESCALED, 320, 80)))
def test_products_kept_and_formed_again(precision, people, founders):
    """Kept products leave one workgroup to a CU, so a launch of more than 256
    forms them again; two chains keep them."""
    case, g0 = family_case(markers=6, missing=0.95, seed=1, tries=1, **line_family(people, founders))
    esz = 8 if precision == native.SL_FP64 else 4
    assert KIB160 // 2 < 5 * esz * locus_cells(case).max() < KIB160 - 12000
    few, few_near = _sweep(case, np.repeat(g0[None], 2, axis=0), precision, 21, 3, 0)
    many, near = _sweep(case, np.repeat(g0[None], 120, axis=0), precision, 21, 3, 0)
    assert np.array_equal(many[:2], few) and np.array_equal(near[:2], few_near)
    ref = oracle_lsweep(Oracle(case), g0, case.M, 21, 119, 3, 0)
    if precision == native.SL_FP64:
        assert not near.any() and np.array_equal(many[119], ref)
    else:
        _check_fp32_sweep(case, many[119], ref, near[119], 0)
