"""M-sweeps over families and maps where the flip classes and the founder-allele
components take every form: fully typed (most flips need no graph), sparsely
typed (components no homozygous person reaches), map lengths around the 64 loci
of a job list's chunk, one and several chains (job index = locus, and job
lists)."""
import numpy as np
import pytest

from oracle_lib import Oracle
from swiftlink_amd import linkage, native, synth
from test_gpu_msampler import assert_likelihoods, shuffled_order

@pytest.mark.gpu
@pytest.mark.parametrize("mode", (native.SL_MSAMPLER_AUTO, native.SL_MSAMPLER_TWO_LAUNCH,
                                  native.SL_MSAMPLER_TWO_LAUNCH | native.SL_MSAMPLER_LDS_GRAPHS))
@pytest.mark.parametrize("markers,missing", ((63, 0.0), (64, 0.3), (65, 0.7), (130, 0.95)))
def test_msweep_over_missing_genotypes(tmp_path, markers, missing, mode):
    case, data = synth.make_case("ped30_snp100", str(tmp_path), n_markers=markers, missing=missing)
    o = Oracle(case)
    starts = np.repeat(synth.true_graph(data, case)[None], 3, axis=0)
    with native.Context(case, native.SL_FP64, msampler_mode=mode) as ctx:
        ctx.mcmc_init(starts)
        ctx.msweep(99, 0)
        ctx.msweep(99, 1)
        out = ctx.mcmc_graphs()
        assert np.all(ctx.mcmc_status() == 0)
        assert np.all(ctx.mcmc_near_edge() == 0)
        lik = ctx.mcmc_likelihood()
    for c in range(3):
        g = o.msweep(starts[c], shuffled_order(o, 99, c, 0), 99, c, 0)
        g = o.msweep(g, shuffled_order(o, 99, c, 1), 99, c, 1)
        assert np.array_equal(out[c], g), c
        ref = np.array([o.fag(g, l) for l in range(case.M)])
        assert np.all(ref > 0) and np.all(np.abs(lik[c] / ref - 1.0) <= 1e-12)


def test_classes_hold_for_every_flip(tmp_path):
    """The rule itself, on the CPU side: with the family's possible phased
    genotypes, a parent that cannot be heterozygous makes a flip change
    nothing, and a parent of known phase with a known transmitted allele makes
    it illegal."""
    case, data = synth.make_case("ped30_snp100", str(tmp_path), n_markers=20, missing=0.2)
    o = Oracle(case)
    g = synth.true_graph(data, case)
    het = 0b1100  # AU, UA
    seen = [0, 0]
    for l in range(case.M):
        cur = o.fag(g, l)
        for p in range(case.F, case.N):
            for side in range(2):
                q = int((case.father if side else case.mother)[p])
                mq, mp = int(case.legal[q, l]), int(case.legal[p, l])
                got = {(0, 1, 0, 1)[t] if side else (0, 1, 1, 0)[t] for t in range(4) if mp >> t & 1}
                f = g.copy()
                f[l, 2 * p + side] ^= 1
                if not mq & het:
                    seen[0] += 1
                    assert abs(o.fag(f, l) / cur - 1.0) < 1e-12
                elif mq in (0b0100, 0b1000) and len(got) == 1:
                    seen[1] += 1
                    assert o.fag(f, l) == 0.0
    assert min(seen) > 20


def _open_edges_case(tmp_path, people, markers, seed):
    """A family whose typed people are nearly all heterozygous: founders carry
    both alleles and homozygous people are untyped, but for one of them at every
    other locus.  Few founder alleles are fixed, so most edges stay open after a
    pass over them, or for several."""
    spec = synth.SynthSpec(people, 4 + people // 100, 1, markers, 0.25, missing=0.0, seed=seed)
    data = synth.generate(spec, max_drops=2)
    case = linkage.load(*synth.write_linkage(data, str(tmp_path / "a")))
    g = synth.true_graph(data, case)
    order = [data["ped"].ids.index(i) for i in case.ids]  # case person -> data person
    rng = np.random.default_rng(seed)
    for l in range(markers):
        al = np.empty((case.N, 2), int)
        for p in range(case.N):
            if p < case.F:
                al[p] = rng.permutation([1, 2])
            else:
                al[p] = [al[case.mother[p], g[l, 2 * p]], al[case.father[p], g[l, 2 * p + 1]]]
        homo = [p for p in range(case.N) if al[p, 0] == al[p, 1]]
        keep = homo[len(homo) // 2] if l % 2 and homo else -1
        for p in range(case.N):
            data["alleles"][order[p]][:, l] = al[p]
            data["missing"][order[p], l] = p in homo and p != keep
    return linkage.load(*synth.write_linkage(data, str(tmp_path / "b"))), g


@pytest.mark.gpu
@pytest.mark.parametrize("people", (30, 150, 180, 400))
def test_many_open_edges(tmp_path, people):
    """More than 64 edges without a fixed allele, below and above the size where
    the rounds leave the registers; legal graphs and flipped ones."""
    case, g = _open_edges_case(tmp_path, people, 8, 4100 + people)
    o = Oracle(case)
    rng = np.random.default_rng(people)
    gs = [g]
    for n in (1, 1, 2, 3):
        f = g.copy()
        for l in range(case.M):
            for b in rng.integers(2 * case.F, 2 * case.N, n):
                f[l, b] ^= 1
        gs.append(f)
    gs = np.stack(gs)
    lik = []
    for graphs in (native.SL_MSAMPLER_AUTO, native.SL_MSAMPLER_LDS_GRAPHS):
        with native.Context(case, native.SL_FP64, msampler_mode=graphs) as ctx:
            ctx.mcmc_init(gs)
            lik.append(ctx.mcmc_likelihood())
    ref = np.array([[o.fag(x, l) for l in range(case.M)] for x in gs])
    assert np.all(ref[0] > 0.0) and (ref == 0.0).any()
    assert_likelihoods(lik[0], ref)
    assert np.array_equal(lik[0], lik[1])


@pytest.mark.gpu
@pytest.mark.parametrize("mode", (native.SL_MSAMPLER_AUTO, native.SL_MSAMPLER_TWO_LAUNCH))
@pytest.mark.parametrize("chains,markers,missing", ((64, 65, 0.1), (70, 65, 0.7), (1100, 5, 0.3), (4200, 3, 0.1)))
def test_planned_steps(tmp_path, chains, markers, missing, mode):
    """Enough chains for planned launches, around the 64 candidates of a job's
    search for its chain (one, two and three rounds), the forward-backward pass
    beside the next step's jobs or before them."""
    case, data = synth.make_case("ped30_snp100", str(tmp_path), n_markers=markers, missing=missing)
    o = Oracle(case)
    g0 = synth.true_graph(data, case)
    with native.Context(case, native.SL_FP64, msampler_mode=mode) as ctx:
        ctx.mcmc_init(np.repeat(g0[None], chains, axis=0))
        ctx.msweep(41, 0)
        ctx.msweep(41, 1)
        out = ctx.mcmc_graphs()
        assert np.all(ctx.mcmc_status() == 0)
        near = ctx.mcmc_near_edge()
    for c in sorted({0, 1, 63, 64 % chains, 65 % chains, chains // 2, chains - 2, chains - 1}):
        assert near[c] == 0
        g = o.msweep(g0, shuffled_order(o, 41, c, 0), 41, c, 0)
        g = o.msweep(g, shuffled_order(o, 41, c, 1), 41, c, 1)
        assert np.array_equal(out[c], g), c
