"""Performance cases: the work a linkage analysis has this library do.

A case is one call (or one short run of calls) through the public entry points
of swiftlink_amd.native, on seeded synthetic pedigrees of the shapes this
repository's benchmark and tests use: 30 to 600 people over 4 to 10
generations with 1 to 10 consanguineous loops, 100 to 5000 SNPs at 0.1 to
0.5 cM, 5 to 20% missing genotypes.  The pedigree of a case is fixed by its
sizes; genotypes, affection, descent graphs and random streams come from the
seed.

kinds of case
  chain   sl_mcmc_run on one context: `chains` replicate chains through the
          L/M sweep schedule, a scored graph every `period`-th sweep, then the
          LOD results and the chains' graphs.  Every pass continues the run.
  batch   sl_batch_run over several uneven pedigrees, 4 chains each
  lod     sl_lod_accumulate_packed over device-resident descent graphs, then
          the LOD results
  terms   sl_lod_terms on graphs in the host layout
  grad    sl_lod_grad (one evaluation of a MOD-score ascent)
  impute  sl_sequential_imputation (the chains' starting graph)
  elod    sl_elod (expected LOD before genotyping)
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from swiftlink_amd import elod as elod_setup
from swiftlink_amd import linkage, native, peelseq, synth
from swiftlink_amd.case import Case

FREQ, PENETRANCE = 1e-4, (0.0, 0.0, 1.0)    # the recessive model the chains score
MOD_MODEL = ((0.05, 0.3, 0.85), 0.12)       # a model a MOD-score ascent passes through
PERIOD, LPROB = 10, 0.5
BATCH_CHAINS = 4


def listed():
    return [
        # a small family, one chain: every call is latency and launches
        dict(name="chain_small", kind="chain", people=30, markers=100, spacing=0.5, missing=0.05, nlod=5,
             fp32=False, chains=1, sweeps=20),
        # the benchmark's headline: one FP32-rescaled chain
        dict(name="chain_fp32", kind="chain", people=150, markers=1000, spacing=0.25, missing=0.10, nlod=5,
             fp32=True, chains=1, sweeps=40),
        # the reference's arithmetic on the larger of the two ordinary pedigrees
        dict(name="chain_fp64", kind="chain", people=200, markers=2000, spacing=0.25, missing=0.10, nlod=5,
             fp32=False, chains=1, sweeps=20),
        # replicate chains of one pedigree in one context
        dict(name="chains_64", kind="chain", people=150, markers=1000, spacing=0.25, missing=0.10, nlod=5,
             fp32=True, chains=64, sweeps=40),
        # the largest pedigree shape, a tenth of its map and an eighth of its chains
        dict(name="chains_large", kind="chain", people=600, markers=2000, spacing=0.1, missing=0.20, nlod=5,
             fp32=True, chains=32, sweeps=4),
        # uneven pedigrees swept side by side
        dict(name="batch_uneven", kind="batch", people=40, people_to=232, count=5, markers=500, markers_to=1700,
             spacing=0.2, missing=0.10, nlod=5, fp32=True, sweeps=10),
        # a few graphs of a small family, host to host: the smallest scoring call
        dict(name="terms_small", kind="terms", people=30, markers=100, spacing=0.5, missing=0.05, nlod=5,
             fp32=False, graphs=3),
        # scoring a batch of sampled graphs, FP32-rescaled and FP64
        dict(name="lod_fp32", kind="lod", people=150, markers=1000, spacing=0.25, missing=0.10, nlod=5,
             fp32=True, graphs=64),
        dict(name="lod_fp64", kind="lod", people=200, markers=2000, spacing=0.25, missing=0.10, nlod=5,
             fp32=False, graphs=50),
        # one MOD-score evaluation: the LOD's backward direction
        dict(name="grad", kind="grad", people=200, markers=2000, spacing=0.25, missing=0.10, nlod=5,
             fp32=False, graphs=32),
        # the default number of imputation replicates
        dict(name="impute_1000", kind="impute", people=150, markers=1000, spacing=0.25, missing=0.10, nlod=5,
             fp32=True, replicates=1000),
        # ELOD in its default precision
        dict(name="elod", kind="elod", people=150, fp32=False, replicates=200000),
    ]


def draw(rng):
    def span(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("chain", "chain", "chain", "batch", "lod", "lod", "terms", "grad", "impute", "elod"))
    c = dict(kind=kind, people=span(30, 400), fp32=rng.random() < 0.5)
    if kind == "elod":
        c["people"] = span(30, 150)
        c["replicates"] = span(1000, 150000)
        return c
    c.update(markers=span(100, 2500), spacing=rng.choice((0.1, 0.2, 0.25, 0.5)),
             missing=rng.choice((0.05, 0.10, 0.20)), nlod=rng.choice((1, 3, 5, 5, 5, 8)))
    if kind == "chain":
        c["people"] = span(30, 600)
        c["chains"] = rng.choice((1, 1, 2, 4, 8, span(2, 100), span(16, 100)))
        c["sweeps"] = rng.randint(4, 40)
        # at most the work of chains_large and chains_64
        while c["sweeps"] * c["chains"] * c["markers"] * c["people"] ** 2 > 4e10:
            if c["chains"] > 1 and c["chains"] >= c["sweeps"]:
                c["chains"] = c["chains"] * 2 // 3
            elif c["sweeps"] > 4:
                c["sweeps"] -= 1
            else:
                c["markers"] = c["markers"] * 2 // 3
    elif kind == "batch":
        c.update(people=span(30, 80), people_to=span(90, 200), count=rng.randint(2, 5), markers=span(100, 500),
                 markers_to=span(500, 1500), sweeps=rng.randint(4, 10))
    elif kind == "impute":
        c["people"] = span(30, 200)
        c["replicates"] = rng.choice((0, 1, span(2, 100), span(100, 1000), span(100, 1000)))
    else:
        c["people"] = span(30, 250)
        if kind == "terms":
            c["graphs"] = span(1, 32)
        else:
            c["graphs"] = span(1, 300)
        cost = {"grad": 1.2e9, "lod": 1.2e10, "terms": 2e9}[kind]
        while c["graphs"] * c["people"] * c["markers"] * c["nlod"] > cost / 16:
            c["graphs"] = max(1, c["graphs"] * 2 // 3)
            if c["graphs"] == 1:
                c["markers"] = max(100, c["markers"] * 2 // 3)
        if kind == "grad":
            c["fp32"] = False
    return c


# ---- inputs ----

@functools.lru_cache(maxsize=None)
def _family(people):
    """(pedigree, file position of each internal person, founders, mother, father, peel table) of a pedigree
    of `people` members in the generators' usual proportions."""
    gens = 4 if people < 100 else 4 + people // 75 if people < 500 else 8
    loops = max(1, people // 60)
    for s in range(1, 400):
        spec = synth.SynthSpec(people, gens, loops, 2, seed=s)
        try:
            ped = synth.make_pedigree(spec, np.random.default_rng(s))
        except RuntimeError:
            continue
        order = sorted(range(people), key=lambda i: ped.father[i] >= 0)
        F = sum(1 for f in ped.father if f < 0)
        at = {i: j for j, i in enumerate(order)}
        mother = np.array([at.get(ped.mother[i], -1) for i in order], np.int32)
        father = np.array([at.get(ped.father[i], -1) for i in order], np.int32)
        ops = peelseq.build(people, F, mother, father, seed=1, tries=16)
        if max(len(ops.cutset(o)) for o in range(ops.n)) <= 5:
            return ped, order, F, mother, father, ops
    raise RuntimeError(f"no pedigree of {people} people")


def _inputs(people, markers, spacing, missing, nlod, seed):
    """A Case with genotypes and affection dropped from `seed`, and the drop's descent graph [M][2N]."""
    ped, order, F, mother, father, ops = _family(people)
    rng = np.random.default_rng([seed, people, markers])
    pos = 10.0 + spacing * np.arange(markers)
    maf = rng.uniform(0.1, 0.5, size=markers)
    best = None
    for _ in range(8):
        alleles, carry, inherit = synth.gene_drop(ped, pos, maf, markers // 2, int(rng.integers(4)), rng)
        affected = carry[:, 0] & carry[:, 1]
        if best is None or affected.sum() > best[1].sum():
            best = alleles, affected, inherit
        if affected.sum() >= 2:
            break
    alleles, affected, inherit = (x[order] for x in best)
    geno = np.where(alleles[:, 0] != alleles[:, 1], linkage.HETERO,
                    np.where(alleles[:, 0] == 1, linkage.HOMOZ_A, linkage.HOMOZ_B)).astype(np.uint8)
    geno[rng.random(geno.shape) < missing] = linkage.UNTYPED
    theta = 0.5 * (1.0 - np.exp(-2.0 * np.diff(pos) / 100.0))
    partial = 0.5 * (1.0 - np.exp(-2.0 * (-0.5 * np.log(1.0 - 2.0 * theta)) / (nlod + 1)))
    aff = np.where(affected, 2, 1).astype(np.int32)
    dprob = np.array([linkage.disease_probs(int(a), i < F, FREQ, list(PENETRANCE)) for i, a in enumerate(aff)])
    case = Case(N=people, F=F, M=markers, nlod=nlod, mother=mother, father=father,
                sex=np.array([ped.sex[i] for i in order], np.int32), affection=aff,
                typed=(geno != 0).any(axis=1).astype(np.int32), geno=geno, disease_prob=dprob,
                geno_prob=linkage.sampler_cache(geno, maf), legal=linkage.eliminate(geno, mother, father, F),
                theta=theta, partial_theta=partial, minor=maf, ops=ops)
    graph = np.zeros((markers, 2 * people), np.int32)
    graph[:, 2 * F:] = inherit[F:].reshape(2 * (people - F), markers).T
    return case, graph


def _case_of(c, seed):
    return _inputs(c["people"], c["markers"], c["spacing"], c["missing"], c["nlod"], seed)


def _graph_bits(case, G, seed):
    """G descent graphs [G][M][2(N-F)]: fair meioses with Haldane crossovers."""
    rng = np.random.default_rng([seed, 77])
    nm = 2 * (case.N - case.F)
    x = np.empty((G, case.M, nm), np.uint8)
    x[:, 0] = rng.random((G, nm), dtype=np.float32) < 0.5
    x[:, 1:] = rng.random((G, case.M - 1, nm), dtype=np.float32) < case.theta[None, :, None].astype(np.float32)
    return np.bitwise_xor.accumulate(x, axis=1)


def _packed(bits):
    """Bits [G][M][nm] as the device layout uint32 [G][M][W], in an int32 tensor on the GPU."""
    W = (bits.shape[2] + 31) // 32
    pad = np.zeros(bits.shape[:2] + (4 * W,), np.uint8)
    by = np.packbits(bits, axis=2, bitorder="little")
    pad[:, :, :by.shape[2]] = by
    return torch.from_numpy(pad.view(np.int32).reshape(bits.shape[0], bits.shape[1], W)).cuda()


def _precision(c):
    return native.SL_FP32_RESCALED if c["fp32"] else native.SL_FP64


def _batch_cases(c, seed):
    n = c["count"]
    between = lambda a, b, i: int(round(a + (b - a) * i / max(n - 1, 1)))
    # the larger pedigrees do not have the longer maps
    return [_inputs(between(c["people"], c["people_to"], i), between(c["markers"], c["markers_to"], (3 * i) % n),
                    c["spacing"], c["missing"], c["nlod"], seed + 1000 * i) for i in range(n)]


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = {"c": c, "seed": seed}
    if kind == "chain":
        cs, g0 = _case_of(c, seed)
        s["ctx"] = ctx = native.Context(cs, _precision(c))
        ctx.mcmc_init(np.repeat(g0[None], c["chains"], axis=0))
        ctx.lod_reset()
        s["sweep"] = 0
    elif kind == "batch":
        s["ctxs"] = []
        for cs, g0 in _batch_cases(c, seed):
            ctx = native.Context(cs, _precision(c))
            ctx.mcmc_init(np.repeat(g0[None], BATCH_CHAINS, axis=0))
            ctx.lod_reset()
            s["ctxs"].append(ctx)
        s["batch"] = native.Batch(s["ctxs"])
        s["sweep"] = 0
    elif kind in ("lod", "grad"):
        cs, _ = _case_of(c, seed)
        s["graphs"] = _packed(_graph_bits(cs, c["graphs"], seed))
        s["ctx"] = native.Context(cs, _precision(c))
        if kind == "grad":
            s["ctx"].set_trait_model(*MOD_MODEL)
        torch.cuda.synchronize()
    elif kind == "terms":
        cs, _ = _case_of(c, seed)
        s["graphs"] = np.zeros((c["graphs"], cs.M, 2 * cs.N), np.int32)
        s["graphs"][:, :, 2 * cs.F:] = _graph_bits(cs, c["graphs"], seed)
        s["ctx"] = native.Context(cs, _precision(c))
    elif kind == "impute":
        s["ctx"] = native.Context(_case_of(c, seed)[0], _precision(c))
    elif kind == "elod":
        base, _ = _inputs(c["people"], 2, 0.25, 0.1, 1, seed)
        c3, c2 = elod_setup.elod_cases(base)
        s["ctx"] = native.Context(c3, _precision(c))
        s["scorer"] = native.Context(c2, native.SL_FP64)
    return s


def run(state):
    c, kind = state["c"], state["c"]["kind"]
    if kind == "chain":
        ctx = state["ctx"]
        st = ctx.mcmc_run(c["sweeps"], 0, PERIOD, LPROB, state["seed"], first_sweep=state["sweep"])
        state["sweep"] += c["sweeps"]
        acc, count, lod = ctx.lod_results()
        return {"stats": st, "acc": acc, "count": count, "lod": lod, "graphs": ctx.mcmc_graphs()}
    if kind == "batch":
        st = state["batch"].run(c["sweeps"], 0, PERIOD, LPROB, state["seed"], first_sweep=state["sweep"])
        state["sweep"] += c["sweeps"]
        out = []
        for ctx, x in zip(state["ctxs"], st):
            acc, count, lod = ctx.lod_results()
            out.append({"stats": x, "acc": acc, "count": count, "lod": lod, "graphs": ctx.mcmc_graphs()})
        return out
    if kind == "lod":
        ctx = state["ctx"]
        ctx.lod_reset()
        ctx.lod_accumulate_packed(state["graphs"].data_ptr(), c["graphs"])
        acc, count, lod = ctx.lod_results()
        return {"acc": acc, "count": count, "lod": lod}
    if kind == "terms":
        return state["ctx"].lod_terms(state["graphs"])
    if kind == "grad":
        lod, dlod = state["ctx"].lod_grad_packed(state["graphs"].data_ptr(), c["graphs"])
        return {"lod": lod, "dlod": dlod}
    if kind == "impute":
        best, weights, index, _ = state["ctx"].sequential_imputation(state["seed"], c["replicates"])
        return {"best": best, "weights": weights, "index": index}
    value = native.run_elod(state["ctx"], state["scorer"], state["seed"], c["replicates"])
    acc, count, _ = state["scorer"].lod_results()
    return {"elod": value, "acc": acc, "count": count}


# ---- what a pass cannot do without ----

def _peel_terms(ops, values):
    """Summed terms (4 per cell) and multiply-adds of one peel whose person p has values[p] possible traits."""
    terms = flops = 0.0
    for o in range(ops.n):
        t = 4.0 * float(np.prod([values[p] for p in ops.cutset(o)]))
        terms += t
        flops += t * (len(ops.prevs(o)) + 2 + len(ops.children(o)))
    return terms, flops


def _sweep_work(people, markers, chains, sweeps, missing):
    """Half L-sweeps, half M-sweeps: an L-step peels the legal cells of a locus and samples every meiosis; an
    M-step labels, joins and counts the founder alleles of every typed person per meiosis and locus."""
    _, _, F, mother, father, ops = _family(people)
    NF = people - F
    legal = np.full(people, 1.5 + 2.5 * missing)
    _, fl = _peel_terms(ops, legal)
    meioses = Case.meioses(_Shape(people, F, mother, father)).size
    col = 2 * NF / 8.0
    l_flops, l_bytes = fl + 20.0 * NF, 4 * col + 16.0 * people / 8
    m_flops, m_bytes = meioses * 8.0 * people, 2 * col + 2.0 * people / 8 + meioses * 16.0
    n = 0.5 * sweeps * chains * markers
    return {"bytes": n * (l_bytes + m_bytes), "flops": n * (l_flops + m_flops)}


class _Shape:
    def __init__(self, N, F, mother, father):
        self.N, self.F, self.mother, self.father = N, F, mother, father


def _plus(a, b):
    return {k: a[k] + b[k] for k in a}


def work(case):
    c, kind = case, case["kind"]

    def lod_work(people, markers, nlod, graphs, backward=False):
        _, _, F, _, _, ops = _family(people)
        values = np.full(people, 4.0 if backward else 3.0)  # unaffected: every trait but AA
        _, fl = _peel_terms(ops, values)
        W = (2 * (people - F) + 31) // 32
        return {"bytes": graphs * markers * 4.0 * W + 8.0 * (markers - 1) * nlod * (7 if backward else 2),
                "flops": graphs * (markers - 1.0) * nlod * fl * (3 if backward else 1)}

    if kind == "chain":
        w = _sweep_work(c["people"], c["markers"], c["chains"], c["sweeps"], c["missing"])
        return _plus(w, lod_work(c["people"], c["markers"], c["nlod"], c["chains"] * max(1, c["sweeps"] // PERIOD)))
    if kind == "batch":
        w = {"bytes": 0.0, "flops": 0.0}
        for i in range(c["count"]):
            t = i / max(c["count"] - 1, 1)
            p = int(round(c["people"] + (c["people_to"] - c["people"]) * t))
            m = (c["markers"] + c["markers_to"]) // 2
            w = _plus(w, _sweep_work(p, m, BATCH_CHAINS, c["sweeps"], c["missing"]))
            w = _plus(w, lod_work(p, m, c["nlod"], BATCH_CHAINS * max(1, c["sweeps"] // PERIOD)))
        return w
    if kind in ("lod", "terms", "grad"):
        return lod_work(c["people"], c["markers"], c["nlod"], c["graphs"], kind == "grad")
    _, _, F, _, _, ops = _family(c["people"])
    R = max(1, c["replicates"])
    if kind == "impute":
        _, fl = _peel_terms(ops, np.full(c["people"], 1.5 + 2.5 * c["missing"]))
        col = 2 * (c["people"] - F) / 8.0
        return {"bytes": R * c["markers"] * 2 * col, "flops": R * c["markers"] * (fl + 20.0 * (c["people"] - F))}
    _, fl = _peel_terms(ops, np.full(c["people"], 4.0))
    _, fd = _peel_terms(ops, np.full(c["people"], 3.0))
    # the trait locus is peeled once for all replicates; the markers and the score once for each
    return {"bytes": R * 8.0, "flops": fd + R * (2 * fl + fd)}


# ---- the same values in 64 bits ----

#: alleles a phased trait UU, AA, AU, UA carries on its maternal and paternal side (1: disease allele)
_ALLELES = ((0, 0), (1, 1), (1, 0), (0, 1))


def _transmission(f, g):
    """P(child trait | mother's, father's) [E][4 mother][4 father][4 child]; f, g [E][2]: probabilities that
    the mother transmits her maternal or paternal allele, and the father his."""
    pick = torch.zeros(4, 4, 4, 2, 2, dtype=torch.float64, device=f.device)
    for m in range(4):
        for p in range(4):
            for i in range(2):
                for j in range(2):
                    pick[m, p, _ALLELES.index((_ALLELES[m][i], _ALLELES[p][j])), i, j] = 1.0
    out = 0.0
    for i in range(2):
        for j in range(2):
            out = out + (f[:, i] * g[:, j]).reshape(-1, 1, 1, 1) * pick[:, :, :, i, j]
    return out


def _peel(cs, trait, trans):
    """The peel's likelihood [E]; trait(p) [E or 1][4], trans(p) as _transmission."""
    ops, tables = cs.ops, {}
    for o in range(ops.n):
        peel = int(ops.peel[o])
        people = ops.cutset(o) + [peel]

        def lay(t, who):
            # t [E][4]... with axes of `who` -> axes of `people`
            perm = sorted(range(len(who)), key=lambda a: people.index(who[a]))
            t = t.permute(0, *[1 + a for a in perm])
            shape = [t.shape[0]] + [4 if p in who else 1 for p in people]
            return t.reshape(shape)

        x = lay(trait(peel), [peel])
        for q in ops.prevs(o):
            x = x * lay(tables[q], ops.cutset(q))
            del tables[q]
        kind = int(ops.type[o])
        if kind == 1:      # CHILD: the peeled person's own transmission
            x = x * lay(trans(peel), [int(cs.mother[peel]), int(cs.father[peel]), peel])
        elif kind == 2:    # PARENT: those of its children in the cutset
            for ch in ops.cutset(o):
                if peel in (int(cs.mother[ch]), int(cs.father[ch])):
                    x = x * lay(trans(ch), [int(cs.mother[ch]), int(cs.father[ch]), ch])
        x = x.expand([x.shape[0]] + [4] * len(people))
        tables[o] = x.sum(dim=-1)
    return tables[ops.n - 1]


def _model(pen, freq, cs, p):
    """Person p's trait probabilities [E][4] under penetrances pen [E][3] and disease frequency freq [E]."""
    aff, out = int(cs.affection[p]), []
    for a, b in _ALLELES:
        k = a + b
        pn = pen[:, k]
        w = pn if aff == 2 else 1.0 - pn
        if p < cs.F:
            w = w * (freq * freq if k == 2 else freq * (1.0 - freq) if k == 1 else (1.0 - freq) * (1.0 - freq))
        out.append(w)
    return torch.stack(out, dim=1)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind not in ("lod", "terms", "grad"):
        return None  # sampled: whole numbers, and sums that depend on every draw
    cs, _ = _case_of(c, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f64 = dict(dtype=torch.float64, device=dev)
    G, nl, n = c["graphs"], cs.M - 1, cs.nlod
    if G * nl * n * cs.N > 2.5e8:
        return None
    bits = torch.from_numpy(_graph_bits(cs, G, seed)).to(dev)
    nm = bits.shape[2]
    ptheta = torch.tensor(cs.partial_theta, **f64)
    k = torch.arange(n, **f64)
    grad = kind == "grad"
    pen, freq = MOD_MODEL if grad else (PENETRANCE, FREQ)
    half = torch.full((1, 2), 0.5, **f64)

    # P(T): every meiosis fair and unlinked
    mp = torch.tensor([list(pen)], **f64).requires_grad_(grad)
    mf = torch.tensor([freq], **f64).requires_grad_(grad)
    pt = _peel(cs, lambda p: _model(mp, mf, cs, p), lambda p: _transmission(half, half)).log()
    dpt = None
    if grad:
        a, b = torch.autograd.grad(pt.sum(), (mp, mf))
        dpt = torch.cat([a[0], b])
    pt = float(pt.detach())

    terms = torch.empty(G, nl, n, **f64)
    d = torch.empty(G, nl, n, 6, **f64) if grad else None
    lt, la = torch.tensor(np.log(cs.theta), **f64), torch.tensor(np.log(1.0 - cs.theta), **f64)
    step = max(1, (16000 if grad else 40000) // (G * n))
    for l0 in range(0, nl, step):
        l1 = min(nl, l0 + step)
        m = l1 - l0
        tl = (ptheta[l0:l1, None] * (k + 1)).expand(G, m, n).reshape(-1)
        tr = (ptheta[l0:l1, None] * (n - k)).expand(G, m, n).reshape(-1)
        x0 = bits[:, l0:l1, None, :].expand(G, m, n, nm).reshape(-1, nm).bool()
        x1 = bits[:, l0 + 1:l1 + 1, None, :].expand(G, m, n, nm).reshape(-1, nm).bool()
        if grad:
            tl, tr = tl.clone().requires_grad_(), tr.clone().requires_grad_()
            E = tl.shape[0]
            mp = torch.tensor([list(pen)], **f64).expand(E, 3).clone().requires_grad_()
            mf = torch.full((E,), freq, **f64).requires_grad_()
        else:
            mp, mf = torch.tensor([list(pen)], **f64), torch.tensor([freq], **f64)

        def side(b):
            return torch.stack([torch.where(x0[:, b] == bool(i), 1.0 - tl, tl) *
                                torch.where(x1[:, b] == bool(i), 1.0 - tr, tr) for i in range(2)], dim=1)

        def trans(p):
            b = 2 * (p - cs.F)
            return 0.25 * _transmission(side(b), side(b + 1))

        like = _peel(cs, lambda p: _model(mp, mf, cs, p), trans)
        if grad:
            g4, gf, gl, gr = torch.autograd.grad(like.sum(), (mp, mf, tl, tr))
            dl = torch.cat([g4, gf[:, None], gl[:, None], gr[:, None]], dim=1) / like.detach()[:, None]
            d[:, l0:l1] = dl.reshape(G, m, n, 6)
        cross = (x0 != x1).sum(dim=1).to(torch.float64).reshape(G, m, n)
        rec = cross * lt[l0:l1, None] + (nm - cross) * la[l0:l1, None]
        terms[:, l0:l1] = like.detach().log().reshape(G, m, n) - rec - nm * math.log(0.5)
    if kind == "terms":
        return terms.cpu().numpy()
    acc = torch.logsumexp(terms, dim=0)
    lod = (acc - math.log(G) - pt) / math.log(10.0)
    if kind == "lod":
        return {"acc": acc.reshape(-1).cpu().numpy(), "count": None, "lod": lod.reshape(-1).cpu().numpy()}
    w = torch.exp(terms - acc)
    dlod = (w[..., None] * d).sum(dim=0)
    dlod[..., :4] -= dpt
    return {"lod": lod.cpu().numpy(), "dlod": (dlod / math.log(10.0)).cpu().numpy()}
