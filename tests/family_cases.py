"""Cases from a pedigree given as parent arrays, without going through files."""
import dataclasses

import numpy as np

from swiftlink_amd import linkage, peelseq
from swiftlink_amd.case import OP_CHILD, Case, PeelOps


def family_case(mother, father, founders, markers, missing, seed, minor=None, spacing=0.5, nlod=2, untyped=(),
                tries=16):
    """(Case, descent graph [M][2N]) of genotypes dropped from `seed` down the
    pedigree (internal order, founders first), a share `missing` of them and all
    of the people `untyped` left out."""
    mother, father = np.asarray(mother, np.int32), np.asarray(father, np.int32)
    N, F, M = len(mother), founders, markers
    rng = np.random.default_rng(seed)
    maf = rng.uniform(0.1, 0.5, M) if minor is None else np.asarray(minor, float)
    theta = np.full(M - 1, 0.5 * (1.0 - np.exp(-2.0 * spacing / 100.0)))
    partial = 0.5 * (1.0 - np.exp(-2.0 * (-0.5 * np.log(1.0 - 2.0 * theta)) / (nlod + 1)))
    graph = np.zeros((M, 2 * N), np.int32)
    graph[0, 2 * F:] = rng.integers(0, 2, 2 * (N - F))
    for l in range(1, M):
        graph[l, 2 * F:] = graph[l - 1, 2 * F:] ^ (rng.random(2 * (N - F)) < theta[l - 1])
    alleles = np.zeros((N, 2, M), np.int8)
    alleles[:F] = rng.random((F, 2, M)) < maf
    for p in range(F, N):  # parents come before children
        for side, q in enumerate((mother[p], father[p])):
            alleles[p, side] = np.where(graph[:, 2 * p + side] == 0, alleles[q, 0], alleles[q, 1])
    geno = np.where(alleles[:, 0] != alleles[:, 1], linkage.HETERO,
                    np.where(alleles[:, 0] == 0, linkage.HOMOZ_A, linkage.HOMOZ_B)).astype(np.uint8)
    geno[rng.random((N, M)) < missing] = linkage.UNTYPED
    geno[list(untyped)] = linkage.UNTYPED
    aff = np.where(np.arange(N) >= F, 1 + rng.integers(0, 2, N), 1).astype(np.int32)
    dprob = np.array([linkage.disease_probs(int(a), i < F, 0.05, [0.1, 0.4, 0.9]) for i, a in enumerate(aff)])
    case = Case(N=N, F=F, M=M, nlod=nlod, mother=mother, father=father, sex=np.zeros(N, np.int32), affection=aff,
                typed=(geno != 0).any(axis=1).astype(np.int32), geno=geno, disease_prob=dprob,
                geno_prob=linkage.sampler_cache(geno, maf), legal=linkage.eliminate(geno, mother, father, F),
                theta=theta, partial_theta=partial, minor=maf,
                ops=peelseq.build(N, F, mother, father, seed=1, tries=tries))
    return case, graph


def line_family(people, founders):
    """A line of couples: each one's first child marries the next founder.
    `people - founders` children in all, spread evenly."""
    mother, father = [-1] * founders, [-1] * founders
    couples, kids = founders - 1, people - founders
    ma, pa = 0, 1
    for c in range(couples):
        first = len(mother)
        for _ in range(kids // couples + (c < kids % couples)):
            mother.append(ma)
            father.append(pa)
        ma, pa = first, c + 2
    return dict(mother=mother, father=father, founders=founders)


def unchained(case):
    """The case with a peel table in which a couple's children are peeled side by
    side: a CHILD op that consumes another over the same parents leaves that table to
    its own consumer, whose op then consumes as many tables as the couple has
    children."""
    ops = case.ops
    prevs = [ops.prevs(o) for o in range(ops.n)]
    for o in range(ops.n - 1, -1, -1):
        for q in list(prevs[o]):
            if ops.type[o] == OP_CHILD == ops.type[q] and set(ops.cutset(o)) == set(ops.cutset(q)):
                up = next(u for u in range(o + 1, ops.n) if o in prevs[u])
                prevs[o].remove(q)
                prevs[up].append(q)
                break
    return dataclasses.replace(case, ops=PeelOps.from_lists(
        ops.type, ops.peel, [ops.cutset(o) for o in range(ops.n)], prevs, [ops.children(o) for o in range(ops.n)]))


def locus_cells(case):
    """Cells of the L-sampler's tables at each locus."""
    legal = np.array([bin(x).count("1") for x in range(16)])[case.legal & 15]
    return sum(np.prod(legal[case.ops.cutset(o)], axis=0, dtype=int) for o in range(case.ops.n))
