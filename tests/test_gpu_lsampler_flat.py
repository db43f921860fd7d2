"""L-sweeps through the per-locus task records at the sizes where the workgroup
of 256 runs out: meioses just below, at and above its 256 threads, levels of
more tasks than threads (sparsely typed), reverse levels wider than a wavefront;
and a family with an op of four consumed tables, which keeps the decoding
kernel.  FP64 graphs equal the oracle's."""
import numpy as np
import pytest

from oracle_lib import Oracle
from swiftlink_amd import linkage, native, synth
from test_gpu_lsampler import oracle_lsweep

pytestmark = pytest.mark.gpu


def _case(tmp_path, people, missing, seed, loops=2, markers=6):
    spec = synth.SynthSpec(people, 4 + people // 100, loops, markers, 0.25, missing=missing, seed=seed)
    data = synth.generate(spec, max_drops=2)
    return linkage.load(*synth.write_linkage(data, str(tmp_path))), data


def _with_meioses(tmp_path, lo, hi, missing):
    """A family whose meiosis count lies in [lo, hi]."""
    for people in range(150, 185):
        for seed in range(3000, 3004):
            try:
                case, data = _case(tmp_path, people, missing, seed)
            except RuntimeError:
                continue
            if lo <= 2 * (case.N - case.F) <= hi:
                return case, data
    raise AssertionError(f"no family with {lo}..{hi} meioses")


def _check(case, data, chains=2):
    o = Oracle(case)
    g = synth.true_graph(data, case)
    with native.Context(case, native.SL_FP64) as ctx:
        ctx.mcmc_init(np.repeat(g[None], chains, axis=0))
        ctx.lsweep(5, 0, 0)
        ctx.lsweep(5, 1, 1)
        out = ctx.mcmc_graphs()
        assert np.all(ctx.mcmc_status() == 0)
        assert np.all(ctx.mcmc_near_edge() == 0)
    for c in range(chains):
        ref = oracle_lsweep(o, g, case.M, 5, c, 0, 0)
        assert np.array_equal(out[c], oracle_lsweep(o, ref, case.M, 5, c, 1, 1)), c


@pytest.mark.parametrize("lo,hi", ((252, 254), (256, 256), (258, 262)))
def test_meioses_around_the_workgroup(tmp_path, lo, hi):
    _check(*_with_meioses(tmp_path, lo, hi, 0.1))


@pytest.mark.parametrize("people,missing", ((30, 0.95), (150, 0.8), (400, 0.3)))
def test_wide_levels(tmp_path, people, missing):
    for seed in range(3100, 3110):
        try:
            case, data = _case(tmp_path, people, missing, seed, loops=1)
        except RuntimeError:
            continue
        return _check(case, data)
    raise AssertionError("no family")


@pytest.mark.parametrize("people", (4, 6, 9))
def test_fewer_levels_than_chunks_in_flight(tmp_path, people):
    """Nuclear families: one to a few levels, fewer than the records' look-ahead."""
    spec = synth.SynthSpec(people, 2, 0, 6, 0.25, missing=0.3, seed=3200 + people)
    data = synth.generate(spec, max_drops=2)
    _check(linkage.load(*synth.write_linkage(data, str(tmp_path))), data)


@pytest.mark.parametrize("people,missing,chains,markers", ((150, 0.97, 300, 4), (300, 0.97, 3, 4)))
def test_products_formed_again(tmp_path, people, missing, chains, markers):
    """Sparsely typed families: kept products of one workgroup fill a CU and the
    launch has more than fit at once (91 KB, 600 workgroups); they do not fit."""
    for seed in range(3300, 3330):
        try:
            case, data = _case(tmp_path, people, missing, seed, loops=1, markers=markers)
        except RuntimeError:
            continue
        return _check(case, data, chains)
    raise AssertionError("no family")


def test_op_of_four_tables():
    from family_cases import family_case, line_family, unchained
    case, g = family_case(markers=9, missing=0.2, seed=6, tries=4, **line_family(26, 8))
    case = unchained(case)
    assert max(len(case.ops.prevs(o)) for o in range(case.ops.n)) == 4
    o = Oracle(case)
    with native.Context(case, native.SL_FP64) as ctx:
        ctx.mcmc_init(np.stack([g, g]))
        ctx.lsweep(5, 0, 0)
        out = ctx.mcmc_graphs()
        assert np.all(ctx.mcmc_status() == 0)
        assert np.all(ctx.mcmc_near_edge() == 0)
    for c in range(2):
        assert np.array_equal(out[c], oracle_lsweep(o, g, case.M, 5, c, 0, 0)), c
