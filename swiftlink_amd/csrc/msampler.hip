// M-sampler kernels for gfx950.
//
// MeiosisSampler (meiosis_sampler.cc:17-203) resamples one meiosis at a time,
// in a shuffled order, at every locus jointly given all other indicators.
// Step k (meiosis m_k) needs, at every locus, the founder-allele-graph
// likelihood of the column with m_k flipped, then a forward-backward pass
// along the loci.
//  * Likelihoods (fag_job): one wavefront per (locus, chain) evaluates
//    FounderAlleleGraph4::likelihood (founder_allele_graph4.cc:34-442).  The
//    reference adds typed persons one by one to components that carry two
//    complementary allele assignments; its result is the sum, over the allele
//    assignments of the founder alleles that satisfy every genotype, of the
//    product of allele frequencies, or 0 when none does.  Here the wave's
//    lanes work on all persons at once: founder-allele labels are propagated
//    generation by generation; every homozygous person fixes its two founder
//    alleles, every heterozygous one is an edge between two alleles that
//    differ; fixed alleles pass along the edges until nothing changes (two or
//    three rounds).  The fixed nodes are counted by ballot: their share of the
//    likelihood is maj^nA min^nB.  Components that no homozygous person reaches
//    (a locus in twenty at ped150) get a union-find with a parity bit per node,
//    built by rounds of hooking roots onto smaller roots and path compression;
//    with n0/n1 the numbers of a root's nodes of parity 0/1 such a component
//    contributes maj^n0 min^n1 + maj^n1 min^n0, taken in log space.  Legality is
//    exactly the reference's; the likelihood agrees with its products to
//    rounding.  With a union-find over every edge of every locus a launch for
//    64 chains at ped150 (half of them on an M-sweep) took 41 us and one for 32
//    at 600 people and 2000 loci 169 us; now 14.5 us and 51.5 us, a third of the
//    loci being evaluated (next point).
//  * Of the flips of a step only those whose outcome depends on the descent
//    graph are evaluated: where the meiosis's parent cannot be heterozygous the
//    flip changes nothing, and where its phase and the transmitted allele are
//    known the flip is illegal (mclass_kernel, once per context).
//  * Forward-backward (forward_backward): one workgroup per chain; a block
//    scan of the 2x2 matrices T(theta_{l-1}) diag(e_l) gives the forward
//    probabilities; a locus draws a uniform only when both its states are
//    possible, so its draw index is the number of drawing loci above it
//    (reverse scan); each locus becomes a 2-bit map from the next locus's
//    indicator to its own, and a reverse scan of map compositions gives every
//    new indicator; changed indicators are written back and the current
//    column's likelihood carried over (raw_matrix, :116-134).  The likelihood
//    rounding and the reassociated products move thresholds only by rounding:
//    draws within 1e-12 of their threshold are counted per chain.
// Step k+1's likelihoods depend on step k's outcome at a locus only through
// the one bit of m_k there.  With few chains (mspec_kernel) one launch runs
// step k's forward-backward pass in one workgroup per chain and, in the other
// workgroups, step k+1's likelihoods for both values of that bit, so a step
// costs one launch.  With more chains the jobs of a step are planned at the
// sweep's start over all of them (mplan_kernel) and shared by as many wavefronts
// as an average step has jobs; while those are few, they run beside the
// forward-backward passes (mbeside_kernel), otherwise each step is a
// forward-backward launch (mfb_kernel) then a likelihood launch
// (mplanned_kernel).  The start of a sweep (mstep_kernel) also computes the
// current columns' likelihoods (MeiosisSampler::reset, :17-40).
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstdint>

#include "msampler_kernels.h"
#include "philox.h"

namespace sl {

namespace {

constexpr int G_HETERO = 1, G_HOMOZ_B = 3;  // genotype codes (genotype.h)
constexpr int kIllegalGraph = -5;
// |ln L(flipped) - ln L(current)| below which both states stay non-zero in
// the FP64 pass (exp(-708) is still a normal double)
constexpr double kFp64DrawLimit = 708.0;
constexpr int kGenoPrefetch = 4;  // genotype chunks of 64 persons loaded ahead

// the sweep index: an argument, or a device counter advanced between
// replays of a captured sweep
__device__ __forceinline__ uint32_t sweep_of(const MsampArgs& A) { return A.sweep_dev ? *A.sweep_dev : A.sweep; }

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63u); }

// x, and s, as values the compiler knows nothing about: what is formed from
// them in a loop stays there.  A planned kernel's job loop otherwise kept every
// address and comparison of a job in registers across jobs (208 registers and
// 243 spilled scalars at 12 chunks).
__device__ __forceinline__ int opaque_v(int x) {
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ int opaque_s(int x) {
    asm volatile("" : "+s"(x));
    return x;
}

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// value of the lane CTRL selects (DPP, within row mask ROWS), 0 where there
// is no source
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_or_zero(double x) {
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, ROWS, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, ROWS, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// sum over the wavefront's lanes, for every lane: an inclusive DPP scan
// (shifts within rows of 16, then each row's total added into the rows
// above it), read from lane 63
__device__ __forceinline__ double wave_sum(double x) {
    x += dpp_or_zero<0x111, 0xf>(x);  // row_shr:1
    x += dpp_or_zero<0x112, 0xf>(x);  // row_shr:2
    x += dpp_or_zero<0x114, 0xf>(x);  // row_shr:4
    x += dpp_or_zero<0x118, 0xf>(x);  // row_shr:8
    x += dpp_or_zero<0x142, 0xa>(x);  // row_bcast:15 into rows 1 and 3
    x += dpp_or_zero<0x143, 0xc>(x);  // row_bcast:31 into rows 2 and 3
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, 63);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), 63);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// A wave's LDS: column words, union-find words, per-node words, edges and
// founder-allele labels.
struct WaveArea {
    uint32_t* colw;   // [W]
    uint32_t* uf;     // [2F] parent (bits 0-15) | parity to parent (bit 16)
    uint32_t* acc;    // [2F] fixed to allele A (bit 0), to B (bit 1), touched (bit 2);
                      //      a free component's root: n0 (bits 3-13), n1 (bits 14-24)
    uint32_t* edges;  // [N] x (bits 0-9) | y (bits 10-19) | kEdge, 0 once settled
    uint16_t* lab;    // [2(N-F)] founder allele of (person, parent); founders first, [2N],
                      //      for the register-resident likelihood
};

// an edge word in use (its nodes may both be node 0 only when it is illegal)
constexpr uint32_t kEdge = 1u << 20;
// a node's word once its component's root has counted it (above the counts)
constexpr uint32_t kCounted = 1u << 25;

__device__ __forceinline__ WaveArea wave_area(const MsampArgs& A, unsigned char* base) {
    WaveArea w;
    w.colw = reinterpret_cast<uint32_t*>(base);
    w.uf = w.colw + A.W;
    w.acc = w.uf + 2 * A.F;
    w.edges = w.acc + 2 * A.F;
    w.lab = reinterpret_cast<uint16_t*>(w.edges + A.N);
    return w;
}

// root of x and the parity of x relative to it; parents only ever point at
// smaller nodes, so the walk ends
__device__ __forceinline__ uint32_t uf_find(const uint32_t* uf, uint32_t x, uint32_t* par) {
    uint32_t p = 0, w = uf[x];
    while ((w & 0xFFFFu) != x) {
        p ^= (w >> 16) & 1u;
        x = w & 0xFFFFu;
        w = uf[x];
    }
    *par = p;
    return x;
}

// genotype of person i at locus l from the 2-bit packed table (0: untyped)
__device__ __forceinline__ int genotype_at(const MsampArgs& A, int l, int i) {
    return (int)((A.geno2[(size_t)l * A.GW + (i >> 4)] >> (2 * (i & 15))) & 3u);
}

// One typed person with genotype g and founder alleles x, y: both are touched,
// and a homozygous person fixes them to its genotype's allele
__device__ __forceinline__ void mark_person(const WaveArea& w, int g, uint32_t x, uint32_t y) {
    const uint32_t mark = g == G_HETERO ? 4u : g == G_HOMOZ_B ? 6u : 5u;
    atomicOr(&w.acc[x], mark);
    atomicOr(&w.acc[y], mark);
}

// An edge whose nodes hold fixed alleles a, b (bits 0-1 of their words, 0:
// none): passes the opposite allele on where one side is fixed.  Returns
// whether the edge is settled (one side fixed), setting *conflict when both
// sides hold the same allele.
__device__ __forceinline__ bool pass_fixed(const WaveArea& w, uint32_t e, uint32_t a, uint32_t b, bool* changed,
                                           bool* conflict) {
    if ((a | b) == 0u) return false;
    if (a == 0u || b == 0u) {
        atomicOr(&w.acc[(a ? e >> 10 : e) & 0x3FFu], (a | b) ^ 3u);
        *changed = true;
    } else {
        *conflict |= (a & b) != 0u;
    }
    return true;
}

// ln(1 + e^-x), out of line: its FP64 constants, kept in registers over a job
// loop, took half of a planned kernel's; a count difference of kLsumK or more is
// the only caller
__device__ __attribute__((noinline)) double log1p_exp_minus(double x) { return log1p(exp(-x)); }

// the share of nA and nB founder alleles fixed to A and to B; a count of 0 has
// none, also where its allele's frequency is 0 and the log infinite
__device__ __forceinline__ double fixed_term(int nA, int nB, double lmaj, double lmin) {
    return (nA ? (double)nA * lmaj : 0.0) + (nB ? (double)nB * lmin : 0.0);
}

// ln(e^l0 + e^l1) of a component free to take either assignment, from its
// root's counts
__device__ __forceinline__ double free_term(const MsampArgs& A, int l, uint32_t a, double lmaj, double lmin) {
    const uint32_t c0 = (a >> 3) & 0x7FFu, c1 = (a >> 14) & 0x7FFu, kd = c0 > c1 ? c0 - c1 : c1 - c0;
    const double n0 = (double)c0, n1 = (double)c1;
    const double l0 = n0 * lmaj + n1 * lmin;  // root allele A
    const double l1 = n1 * lmaj + n0 * lmin;  // root allele B
    return fmax(l0, l1) + (kd < (uint32_t)kLsumK ? A.lsum[(size_t)l * kLsumK + kd] : log1p_exp_minus(fabs(l0 - l1)));
}

// log of the founder-allele-graph likelihood of the column in w.colw at locus
// l (-inf when illegal), computed by one wavefront
__device__ double fag_log_likelihood(const MsampArgs& A, const uint2* ptab, const WaveArea& w, int l) {
    const int lane = lane_id();
    const int F = A.F, nodes = 2 * A.F;
    // the first genotype chunks are loaded before the label pass so that the
    // global-load latency overlaps it
    int gpre[kGenoPrefetch];
#pragma unroll
    for (int c = 0; c < kGenoPrefetch; ++c) {
        const int i = 64 * c + lane;
        gpre[c] = i < A.N ? genotype_at(A, l, i) : 0;
    }
    // founder-allele labels of non-founders, parents first (reset, :543-569)
    for (int gen = 0; gen < A.n_gen; ++gen) {
        const int k1 = A.gen_off[gen + 1];
        for (int k = A.gen_off[gen] + lane; k < k1; k += 64) {
            const uint2 e = ptab[k];
            const int i = (int)(e.x & 0xFFFFu), mo = (int)(e.y & 0xFFFFu), fa = (int)(e.y >> 16);
            const int b = 2 * (i - F);
            const uint32_t bm = (w.colw[b >> 5] >> (b & 31)) & 1u;
            const uint32_t bp = (w.colw[(b + 1) >> 5] >> ((b + 1) & 31)) & 1u;
            w.lab[b] = mo < F ? (uint16_t)(2 * mo + (int)bm) : w.lab[2 * (mo - F) + (int)bm];
            w.lab[b + 1] = fa < F ? (uint16_t)(2 * fa + (int)bp) : w.lab[2 * (fa - F) + (int)bp];
        }
        wave_sync();
    }
    for (int x = lane; x < nodes; x += 64) w.acc[x] = 0u;
    wave_sync();
    // the typed persons with a genotype: a homozygous one fixes both its
    // founder alleles, a heterozygous one is an edge between them
    const uint64_t below = (1ull << lane) - 1ull;
    int E = 0;
    bool bad = false;
    for (int i0 = 0, c = 0; i0 < A.N; i0 += 64, ++c) {
        const int i = i0 + lane;
        int g = 0;
#pragma unroll
        for (int k = 0; k < kGenoPrefetch; ++k)
            if (c == k) g = gpre[k];
        if (c >= kGenoPrefetch) g = i < A.N ? genotype_at(A, l, i) : 0;
        uint32_t x = 0, y = 0;
        if (g) {
            x = i < F ? (uint32_t)(2 * i) : w.lab[2 * (i - F)];
            y = i < F ? (uint32_t)(2 * i + 1) : w.lab[2 * (i - F) + 1];
            bad |= g == G_HETERO && x == y;  // an autozygous heterozygote (:77-81)
            mark_person(w, g, x, y);
        }
        const uint64_t mask = __ballot(g == G_HETERO);
        if (g == G_HETERO) w.edges[E + __popcll(mask & below)] = x | (y << 10) | kEdge;
        E += __popcll(mask);
    }
    if (__ballot(bad)) return -INFINITY;
    // fixed alleles pass along the edges until nothing changes
    bool conflict = false, pending = false;
    for (;;) {
        wave_sync();
        bool changed = false;
        pending = false;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + lane;
            uint32_t ed = e < E ? w.edges[e] : 0u;
            if (ed) {
                const uint32_t a = w.acc[ed & 0x3FFu] & 3u, b = w.acc[(ed >> 10) & 0x3FFu] & 3u;
                if (pass_fixed(w, ed, a, b, &changed, &conflict)) w.edges[e] = 0u;
                else pending = true;
            }
        }
        if (!__ballot(changed)) break;
    }
    int nA = 0, nB = 0;
    for (int x0 = 0; x0 < nodes; x0 += 64) {
        const uint32_t a = x0 + lane < nodes ? w.acc[x0 + lane] & 3u : 0u;
        conflict |= a == 3u;
        nA += __popcll(__ballot(a == 1u));
        nB += __popcll(__ballot(a == 2u));
    }
    if (__ballot(conflict)) return -INFINITY;
    const double lmaj = A.lfreq[2 * (size_t)l], lmin = A.lfreq[2 * (size_t)l + 1];
    const double ll = fixed_term(nA, nB, lmaj, lmin);
    if (!__ballot(pending)) return ll;
    // components no homozygous person reaches: hook the larger root under the
    // smaller one with the parity the edge implies (the alleles of an edge
    // differ), compress paths, until no edge joins two components (every
    // productive round removes a component, so at most 2F rounds)
    for (int x = lane; x < nodes; x += 64) w.uf[x] = (uint32_t)x;
    wave_sync();
    bool converged = false;
    for (int round = 0; round <= nodes && !converged; ++round) {
        bool changed = false;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + lane;
            if (e < E && w.edges[e]) {
                const uint32_t ed = w.edges[e];
                uint32_t px, py;
                const uint32_t rx = uf_find(w.uf, ed & 0x3FFu, &px);
                const uint32_t ry = uf_find(w.uf, (ed >> 10) & 0x3FFu, &py);
                if (rx != ry) {
                    w.uf[rx > ry ? rx : ry] = (rx < ry ? rx : ry) | ((px ^ py ^ 1u) << 16);
                    changed = true;
                }
            }
            wave_sync();
        }
        for (int x0 = 0; x0 < nodes; x0 += 64) {
            const int x = x0 + lane;
            uint32_t r = 0, p = 0;
            if (x < nodes) r = uf_find(w.uf, (uint32_t)x, &p);
            wave_sync();
            if (x < nodes) w.uf[x] = r | (p << 16);
            wave_sync();
        }
        converged = !__ballot(changed);
    }
    // converged and compressed: every node's word holds its root and parity
    bool illegal = !converged;
    for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane;
        if (e < E && w.edges[e]) {
            const uint32_t ed = w.edges[e];
            const uint32_t ux = w.uf[ed & 0x3FFu], uy = w.uf[(ed >> 10) & 0x3FFu];
            illegal |= (ux & 0xFFFFu) != (uy & 0xFFFFu) || (((ux ^ uy) >> 16) & 1u) != 1u;
        }
    }
    if (__ballot(illegal)) return -INFINITY;
    // touched nodes without a fixed allele, counted at their root by parity
    for (int x = lane; x < nodes; x += 64)
        if ((w.acc[x] & 7u) == 4u) {
            const uint32_t u = w.uf[x];
            atomicAdd(&w.acc[u & 0xFFFFu], ((u >> 16) & 1u) ? (1u << 14) : (1u << 3));
        }
    wave_sync();
    double free_ll = 0.0;
    for (int x = lane; x < nodes; x += 64) {
        const uint32_t a = w.acc[x];
        if ((a & 7u) == 4u && (w.uf[x] & 0xFFFFu) == (uint32_t)x) free_ll += free_term(A, l, a, lmaj, lmin);
    }
    return ll + wave_sum(free_ll);
}

// The same likelihood for pedigrees of at most 64*KC people and 32*KC
// founders: lane j holds people j, j+64, ... (genotype, edge) and slots j,
// j+64, ... of the generation-ordered person table.  One pass over the edges
// settles nearly all of them (at 600 people 187 heterozygous people leave 0 to
// 31 edges, at 150 people 0 or 1), so the rest are packed into a list, which
// the later rounds and the union-find go through 64 at a time (32 chains of 600
// people and 2000 loci: 66.5 -> 53 us a launch; before, every round went over
// every person's edge and the union-find over every founder allele).  Their
// launches are bound by instruction issue; one chain waits for its slowest job.
// The per-root terms and their order of summation are those of
// fag_log_likelihood, so the result is the same.
// A job's global inputs for the register-resident likelihood, loaded at once
// at its start: lane j's genotypes and person-table slots j, j+64, ..., and
// the locus's log allele-frequency terms.
template <int KC>
struct JobInputs {
    int g[KC];
    uint2 pt[KC];
    double lmaj, lmin;
    __device__ __forceinline__ void load(const MsampArgs& A, int l) {
        const int lane = opaque_v(lane_id()), N = opaque_s(A.N), NF = N - opaque_s(A.F);
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            const int i = 64 * c + lane;
            g[c] = i < N ? genotype_at(A, l, i) : 0;
            pt[c] = i < NF ? A.ptab[i] : make_uint2(0u, 0u);
        }
        lmaj = A.lfreq[2 * (size_t)l];
        lmin = A.lfreq[2 * (size_t)l + 1];
    }
};

// Chunks up to which every round goes over all edges, in registers (a launch of
// one chain of 150 people waits for its slowest job: 7.47 us a step against 7.61
// through the list).
constexpr int kRegisterRounds = 3;

// lanes of m below this one
__device__ __forceinline__ uint32_t count_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

template <int KC>
__device__ double fag_log_likelihood_r(const MsampArgs& A, const JobInputs<KC>& in, const WaveArea& w, int l) {
    const int lane = opaque_v(lane_id());
    const int N = opaque_s(A.N), F = opaque_s(A.F), NF = N - F, nodes = 2 * F;
    const double lmaj = in.lmaj, lmin = in.lmin;
    // (the nodes' words and the founders' labels were written by fag_job while
    // the job's loads were in flight)
    // label slots (reset, founder_allele_graph4.cc:543-569): where each of a
    // person's two labels comes from.  The slots are in generation order and a
    // parent's generation is below its child's, so a chunk's slots only read
    // slots of earlier chunks or of earlier generations of their own chunk:
    // each chunk runs just the generations it spans (its first and last slot's)
#pragma unroll
    for (int c = 0; c < KC; ++c) {
        if (64 * c < NF) {
            const bool in_use = 64 * c + lane < NF;
            const uint2 e = in.pt[c];
            const uint32_t i = in_use ? e.x & 0xFFFFu : (uint32_t)F, b = 2u * (i - (uint32_t)F);
            const uint32_t bits = w.colw[b >> 5] >> (b & 31u);
            const uint32_t s0 = 2u * (e.y & 0xFFFFu) + (bits & 1u), s1 = 2u * (e.y >> 16) + ((bits >> 1) & 1u);
            const int gen = in_use ? (int)(e.x >> 16) : -1;
            const int last = NF - 64 * c > 64 ? 63 : NF - 1 - 64 * c;
            const int g1 = __builtin_amdgcn_readlane(gen, last);
            for (int g = __builtin_amdgcn_readlane(gen, 0); g <= g1; ++g) {
                if (gen == g) {
                    const uint32_t l0 = w.lab[s0], l1 = w.lab[s1];
                    *reinterpret_cast<uint32_t*>(w.lab + 2 * i) = l0 | (l1 << 16);
                }
                wave_sync();
            }
        }
    }
    // the typed people: homozygous ones fix both their founder alleles,
    // heterozygous ones are edges between them
    uint32_t e[KC];
    bool bad = false;
#pragma unroll
    for (int c = 0; c < KC; ++c) {
        e[c] = 0u;
        if (64 * c < N) {
            if (in.g[c]) {
                const uint32_t xy = *reinterpret_cast<const uint32_t*>(w.lab + 2 * (64 * c + lane));
                const uint32_t x = xy & 0xFFFFu, y = xy >> 16;
                if (in.g[c] == G_HETERO) {
                    bad |= x == y;  // an autozygous heterozygote (:77-81)
                    e[c] = x | (y << 10) | kEdge;
                }
                mark_person(w, in.g[c], x, y);
            }
        }
    }
    if (__ballot(bad)) return -INFINITY;
    // fixed alleles pass along the edges; those with neither side fixed are
    // packed into w.edges
    bool conflict = false, changed = false;
    int listed = 0;
    const auto list_edges = [&](bool pend, uint32_t word) {
        const uint64_t m = __ballot(pend);
        if (m) {
            if (pend) w.edges[listed + (int)count_below(m)] = word;
            listed += __popcll(m);
        }
    };
    if constexpr (KC <= kRegisterRounds) {
        do {
            wave_sync();
            changed = false;
            uint32_t fa[KC], fb[KC];
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                fa[c] = w.acc[e[c] & 0x3FFu] & 3u;
                fb[c] = w.acc[(e[c] >> 10) & 0x3FFu] & 3u;
            }
#pragma unroll
            for (int c = 0; c < KC; ++c)
                if (e[c] && pass_fixed(w, e[c], fa[c], fb[c], &changed, &conflict)) e[c] = 0u;
        } while (__ballot(changed));
#pragma unroll
        for (int c = 0; c < KC; ++c) list_edges(e[c] != 0u, e[c]);
    } else {
        wave_sync();
#pragma unroll
        for (int c0 = 0; c0 < KC; c0 += 4) {
            if (64 * c0 < N) {
                uint32_t fa[4] = {0, 0, 0, 0}, fb[4] = {0, 0, 0, 0};
#pragma unroll
                for (int c = c0; c < KC && c < c0 + 4; ++c) {
                    fa[c - c0] = w.acc[e[c] & 0x3FFu] & 3u;
                    fb[c - c0] = w.acc[(e[c] >> 10) & 0x3FFu] & 3u;
                }
#pragma unroll
                for (int c = c0; c < KC && c < c0 + 4; ++c)
                    list_edges(e[c] != 0u && !pass_fixed(w, e[c], fa[c - c0], fb[c - c0], &changed, &conflict), e[c]);
            }
        }
    }
    // round after round over the list until nothing changes
    bool pending = listed > 0;
    while (pending && __ballot(changed)) {
        wave_sync();
        changed = pending = false;
        for (int k0 = 0; k0 < listed; k0 += 64) {
            const uint32_t x = k0 + lane < listed ? w.edges[k0 + lane] : 0u;
            bool pend = false;
            if (x) {
                const uint32_t a = w.acc[x & 0x3FFu] & 3u, b = w.acc[(x >> 10) & 0x3FFu] & 3u;
                if (pass_fixed(w, x, a, b, &changed, &conflict)) w.edges[k0 + lane] = 0u;
                else pend = true;
            }
            pending |= __ballot(pend) != 0;
        }
    }
    wave_sync();
    int nA = 0, nB = 0;
#pragma unroll
    for (int n = 0; n < KC; ++n) {
        if (64 * n < nodes) {
            const int x = 64 * n + lane;
            const uint32_t t = x < nodes ? w.acc[x] & 3u : 0u;
            conflict |= t == 3u;
            nA += __popcll(__ballot(t == 1u));
            nB += __popcll(__ballot(t == 2u));
        }
    }
    if (__ballot(conflict)) return -INFINITY;
    const double ll = fixed_term(nA, nB, lmaj, lmin);
    if (!pending) return ll;
    if (listed <= 64) {
        // one edge left (half of the rest, nearly all of it at 150 people): its
        // two alleles are a component of their own
        const uint64_t m = __ballot(lane < listed && w.edges[lane] != 0u);
        if (__popcll(m) == 1) return ll + free_term(A, l, (1u << 3) | (1u << 14), lmaj, lmin);
    }
    // components no homozygous person reaches.  Their nodes are the ends of the
    // edges left; rounds of hooking larger roots onto smaller ones until a round
    // hooks nothing (each hooking round removes a component, so at most 2F
    // rounds hook); the alleles of an edge differ
    for (int k0 = 0; k0 < listed; k0 += 64) {
        const uint32_t e0 = k0 + lane < listed ? w.edges[k0 + lane] : 0u;
        if (e0) {
            const uint32_t x = e0 & 0x3FFu, y = (e0 >> 10) & 0x3FFu;
            w.uf[x] = x;
            w.uf[y] = y;
        }
    }
    bool converged = false, illegal = false;
    for (int round = 0; round <= nodes; ++round) {
        bool hooked = false;
        illegal = false;
        for (int k0 = 0; k0 < listed; k0 += 64) {
            wave_sync();
            const uint32_t e0 = k0 + lane < listed ? w.edges[k0 + lane] : 0u;
            uint32_t rx = 0, ry = 0, px = 0, py = 0;
            if (e0) {
                rx = uf_find(w.uf, e0 & 0x3FFu, &px);
                ry = uf_find(w.uf, (e0 >> 10) & 0x3FFu, &py);
            }
            wave_sync();
            if (e0) {
                if (rx != ry) {
                    w.uf[rx > ry ? rx : ry] = (rx < ry ? rx : ry) | ((px ^ py ^ 1u) << 16);
                    hooked = true;
                } else {
                    illegal |= (px ^ py) != 1u;
                }
            }
        }
        if (!__ballot(hooked)) {
            converged = true;
            break;
        }
    }
    // the last round found every edge's ends in one component: their parities
    if (!converged || __ballot(illegal)) return -INFINITY;
    // each end once, counted at its root by parity
    for (int k0 = 0; k0 < listed; k0 += 64) {
        const uint32_t e0 = k0 + lane < listed ? w.edges[k0 + lane] : 0u;
        if (e0) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const uint32_t x = (e0 >> (10 * s)) & 0x3FFu;
                if (!(atomicOr(&w.acc[x], kCounted) & kCounted)) {
                    uint32_t p;
                    const uint32_t r = uf_find(w.uf, x, &p);
                    atomicAdd(&w.acc[r], p ? (1u << 14) : (1u << 3));
                }
            }
        }
    }
    wave_sync();
    double free_ll = 0.0;
#pragma unroll
    for (int n = 0; n < KC; ++n) {
        if (64 * n < nodes) {
            const int x = 64 * n + lane;
            const uint32_t a = x < nodes ? w.acc[x] : 0u;
            if ((a & (kCounted - 8u)) != 0u) free_ll += free_term(A, l, a, lmaj, lmin);
        }
    }
    return ll + wave_sum(free_ll);
}

// The forward-backward pass runs in FP64 (SL_FP64 contexts: the reference's
// arithmetic, draws decided as it decides them) or in FP32 (FP32-rescaled
// contexts): 2x2 products keep their largest entry in [0.5, 1) by an exact
// power of two in both.  The founder-allele log-likelihoods it reads are FP64
// in both.
template <typename T>
struct MatT {
    T a, b, c, d;  // [[a, b], [c, d]]
};
using Mat = MatT<double>;
static_assert(fb_static_lds(64) == sizeof(Mat) + 2 * sizeof(uint32_t), "LDS of the scans: wtot, wcnt, wmap");

// product with an exact power-of-two rescale keeping the largest entry in
// [0.5, 1): for a normal largest entry m with biased exponent E the factor is
// 2^(1022-E) (FP64) or 2^(126-E) (FP32), built from its bits; a subnormal m
// takes frexp/ldexp, behind a wavefront-wide test that is seldom taken, so
// that the usual product has no divergent branch (a pass is one wavefront's
// instruction chain: with a branch per product it was a third longer)
__device__ __forceinline__ Mat mmul(const Mat& x, const Mat& y) {
    Mat r{x.a * y.a + x.b * y.c, x.a * y.b + x.b * y.d, x.c * y.a + x.d * y.c, x.c * y.b + x.d * y.d};
    const double m = fmax(fmax(r.a, r.b), fmax(r.c, r.d));
    const uint32_t E = (uint32_t)(__builtin_bit_cast(uint64_t, m) >> 52) & 0x7FFu;
    const double f = __builtin_bit_cast(double, (uint64_t)(E - 1u < 2044u ? 2045u - E : 1023u) << 52);
    r.a *= f;
    r.b *= f;
    r.c *= f;
    r.d *= f;
    const bool sub = m > 0.0 && E == 0u;
    if (__builtin_expect(__ballot(sub) != 0ull, 0)) {
        if (sub) {
            int e;
            (void)frexp(m, &e);
            r.a = ldexp(r.a, -e);
            r.b = ldexp(r.b, -e);
            r.c = ldexp(r.c, -e);
            r.d = ldexp(r.d, -e);
        }
    }
    return r;
}

__device__ __forceinline__ MatT<float> mmul(const MatT<float>& x, const MatT<float>& y) {
#pragma clang fp contract(fast)
    MatT<float> r{x.a * y.a + x.b * y.c, x.a * y.b + x.b * y.d, x.c * y.a + x.d * y.c, x.c * y.b + x.d * y.d};
    const float m = fmaxf(fmaxf(r.a, r.b), fmaxf(r.c, r.d));
    const uint32_t E = (__float_as_uint(m) >> 23) & 0xFFu;
    const float f = __uint_as_float((E - 1u < 252u ? 253u - E : 127u) << 23);
    r.a *= f;
    r.b *= f;
    r.c *= f;
    r.d *= f;
    const bool sub = m > 0.0f && E == 0u;
    if (__builtin_expect(__ballot(sub) != 0ull, 0)) {
        if (sub) {
            const int e = __builtin_amdgcn_frexp_expf(m);
            r.a = __builtin_amdgcn_ldexpf(r.a, -e);
            r.b = __builtin_amdgcn_ldexpf(r.b, -e);
            r.c = __builtin_amdgcn_ldexpf(r.c, -e);
            r.d = __builtin_amdgcn_ldexpf(r.d, -e);
        }
    }
    return r;
}

__device__ __forceinline__ uint32_t compose(uint32_t f, uint32_t h) {
    // 2-bit maps: bit x = image of x; (f o h)(x) = f(h(x))
    return ((f >> (h & 1u)) & 1u) | (((f >> ((h >> 1) & 1u)) & 1u) << 1);
}

// DPP lane moves of GFX9: row_shr:n / row_shl:n within rows of 16 lanes,
// wave_shr:1 / wave_shl:1 across the wavefront, row_bcast:15 / row_bcast:31
// from the last lane of a row to the rows above it.  Lanes without a source,
// and rows outside the row mask, keep `old`.
constexpr int kDppWaveShr1 = 0x138, kDppRowBcast15 = 0x142, kDppRowBcast31 = 0x143;
constexpr int dpp_row_shl(int n) { return 0x100 + n; }
constexpr int dpp_row_shr(int n) { return 0x110 + n; }

template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ uint32_t u32_dpp(uint32_t old, uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)x, CTRL, ROWS, 0xf, false);
}

template <int CTRL, int ROWS>
__device__ __forceinline__ double t_dpp(double old, double x) {
    const uint64_t o = __builtin_bit_cast(uint64_t, old), u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = u32_dpp<CTRL, ROWS>((uint32_t)o, (uint32_t)u);
    const uint32_t hi = u32_dpp<CTRL, ROWS>((uint32_t)(o >> 32), (uint32_t)(u >> 32));
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

template <int CTRL, int ROWS>
__device__ __forceinline__ float t_dpp(float old, float x) {
    return __uint_as_float(u32_dpp<CTRL, ROWS>(__float_as_uint(old), __float_as_uint(x)));
}

template <int CTRL, int ROWS = 0xf, typename T>
__device__ __forceinline__ MatT<T> mat_dpp(const MatT<T>& x) {  // the identity where there is no source
    return MatT<T>{t_dpp<CTRL, ROWS>((T)1, x.a), t_dpp<CTRL, ROWS>((T)0, x.b), t_dpp<CTRL, ROWS>((T)0, x.c),
                   t_dpp<CTRL, ROWS>((T)1, x.d)};
}

__device__ __forceinline__ uint32_t readlane_u32(uint32_t x, int lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)x, lane);
}

__device__ __forceinline__ double readlane_t(double x, int lane) {
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = readlane_u32((uint32_t)u, lane), hi = readlane_u32((uint32_t)(u >> 32), lane);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

__device__ __forceinline__ float readlane_t(float x, int lane) {
    return __uint_as_float(readlane_u32(__float_as_uint(x), lane));
}

// inclusive left-to-right products across the wavefront
template <typename T>
__device__ __forceinline__ MatT<T> wave_products(MatT<T> P) {
    P = mmul(mat_dpp<dpp_row_shr(1)>(P), P);
    P = mmul(mat_dpp<dpp_row_shr(2)>(P), P);
    P = mmul(mat_dpp<dpp_row_shr(4)>(P), P);
    P = mmul(mat_dpp<dpp_row_shr(8)>(P), P);
    P = mmul(mat_dpp<kDppRowBcast15, 0xa>(P), P);
    return mmul(mat_dpp<kDppRowBcast31, 0xc>(P), P);
}

__device__ __forceinline__ bool is_msweep(const MsampArgs& A, int chain) {
    return !A.check_kind || !(philox_uniform(A.seed, (uint32_t)chain, sweep_of(A), kStepSched, 0) < A.lprob);
}

// flipped-column log-likelihoods: [step parity][variant][chain][locus]
__device__ __forceinline__ size_t lflip_index(const MsampArgs& A, int k, int v, int chain, int l) {
    return (((size_t)(k & 1) * 2 + (size_t)v) * (size_t)A.n_chains + (size_t)chain) * (size_t)A.M + (size_t)l;
}

// the uniforms of step k: [step parity][chain][draw index]
__device__ __forceinline__ size_t udev_index(const MsampArgs& A, int k, int chain) {
    return ((size_t)(k & 1) * (size_t)A.n_chains + (size_t)chain) * (size_t)A.M;
}

__device__ __forceinline__ int order_at(const MsampArgs& A, int chain, int k) {
    return A.order[(size_t)chain * A.n_meioses + k];
}

// One founder-allele likelihood job of a wavefront, job q of this launch:
//  * with A.with_lcur, jobs [0, M) are the current columns (into lcur; a zero
//    marks the chain's graph illegal, meiosis_sampler.cc:33-36);
//  * the other jobs are step A.step's columns with meiosis m_k flipped (into
//    lflip, MeiosisSampler::step, :116-134), at the loci where that has to be
//    computed (class kFlipCompute).  With A.spec and k > 0, variant v first
//    forces meiosis m_{k-1}'s bit to v: the forward-backward pass of step k-1
//    may be deciding that bit in the same launch, and it is the only bit it
//    changes.  Where m_{k-1}'s own flip changes nothing or is illegal one job
//    serves both variants: the bit's value does not matter (it is taken as 0),
//    or it cannot change.
template <int KC>
__device__ void fag_job(const MsampArgs& A, int chain, int q, const uint2* ptab, unsigned char* wbase) {
    const int lane = lane_id(), M = A.M;
    // the chain's status, read with the job's other loads: a chain whose
    // graph is illegal keeps its buffers as they are
    const int status = A.status[chain];
    int l, v = 0, flip = -1, force = -1;
    int fc = kFlipCompute, pc = kFlipCompute;
    bool current = false, two = false;
    if (A.with_lcur && q < M) {
        l = q;
        current = true;
    } else {
        // with two variants (A.spec, k > 0), jobs 2e and 2e+1 share a
        // workgroup, and so an XCD's L2, for their locus's column
        const int r = A.with_lcur ? q - M : q;
        two = A.spec && A.step > 0;
        v = two ? (r & 1) : 0;
        const int e = two ? (r >> 1) : r;
        flip = order_at(A, chain, A.step);
        if (two) force = order_at(A, chain, A.step - 1);
        if (A.compact) {
            // an illegal chain's order may be stale
            if (status != 0 || e >= A.jobcnt[flip]) return;
            l = A.joblist[(size_t)flip * M + e];
        } else {
            // the class is read beside the job's data, whatever the status;
            // a stale order may hold anything
            l = e;
            const int top = 2 * (A.N - A.F) - 1;
            fc = A.cls[(size_t)min((uint32_t)flip, (uint32_t)top) * M + l];
            if (two) force = (int)min((uint32_t)force, (uint32_t)top);
        }
        if (two) pc = A.cls[(size_t)force * M + l];
    }
    WaveArea w = wave_area(A, wbase);
    const uint32_t* src = A.graphs + ((size_t)chain * M + l) * A.W;
    // where the likelihood goes, formed before the work that produces it
    double* const dst = current ? A.lcur + (size_t)chain * M + l : A.lflip + lflip_index(A, A.step, v, chain, l);
    if (pc == kFlipIllegal) force = -1;
    const bool serves_both = two && pc != kFlipCompute;
    double* const dst1 = serves_both ? A.lflip + lflip_index(A, A.step, 1, chain, l) : nullptr;
    JobInputs<KC> in;
    if constexpr (KC > 0) {
        in.load(A, l);
        // no node fixed or touched, and the founders' labels, written while
        // the loads above are in flight
        for (int x = lane; x < 2 * A.F; x += 64) w.acc[x] = 0u;
        for (int f = lane; f < A.F; f += 64)
            *reinterpret_cast<uint32_t*>(w.lab + 2 * f) = (uint32_t)(2 * f) | ((uint32_t)(2 * f + 1) << 16);
    }
    for (int k = lane; k < A.W; k += 64) {
        uint32_t x = src[k];
        if (force >= 0 && (force >> 5) == k) x = (x & ~(1u << (force & 31))) | ((uint32_t)v << (force & 31));
        if (flip >= 0 && (flip >> 5) == k) x ^= 1u << (flip & 31);
        w.colw[k] = x;
    }
    if (fc != kFlipCompute || (serves_both && v)) return;
    wave_sync();
    double L;
    if constexpr (KC > 0) L = fag_log_likelihood_r<KC>(A, in, w, l);
    else L = fag_log_likelihood(A, ptab, w, l);
    if (status != 0) return;
    if (lane == 0) {
        *dst = L;
        if (serves_both) *dst1 = L;
        if (current && L == -INFINITY) A.status[chain] = kIllegalGraph;
    }
}

// likelihood buffers of step k at locus l: the flipped column's variant is the
// bit of meiosis m_{k-1} there (already decided when step k's pass runs)
struct StepView {
    const MsampArgs* A;
    int chain, k, word, pword;
    uint32_t bm, pbm;
    bool spec;
    const uint8_t* cls;  // the classes of m_k's flip by locus
    __device__ __forceinline__ double lf(const uint32_t* g, int l, double lcur) const {
        const int c = cls[l];
        if (c != kFlipCompute) return c == kFlipSame ? lcur : -INFINITY;
        const int v = spec ? ((g[(size_t)l * A->W + pword] & pbm) ? 1 : 0) : 0;
        return A->lflip[lflip_index(*A, k, v, chain, l)];
    }
};

// Pieces of the forward-backward pass (meiosis_sampler.cc:136-203).

// locus matrix from the two states' likelihoods scaled by the larger one:
// T(theta_{l-1}) diag(e_l), A_0 = diag(e_0)
template <typename T>
__device__ __forceinline__ MatT<T> emission_matrix_th(T e0, T e1, bool first, double theta) {
    if (first) return MatT<T>{e0, (T)0, (T)0, e1};
    const T th = (T)theta, an = (T)(1.0 - theta);
    return MatT<T>{an * e0, th * e1, th * e0, an * e1};
}

template <typename T>
__device__ __forceinline__ MatT<T> emission_matrix(const MsampArgs& A, T e0, T e1, int l) {
    return emission_matrix_th(e0, e1, l == 0, l == 0 ? 0.0 : A.theta[l - 1]);
}

__device__ __forceinline__ double exp_t(double x) { return exp(x); }
__device__ __forceinline__ float exp_t(float x) { return expf(x); }

// e0, e1 of locus l from the current and flipped columns' log-likelihoods,
// exp(x - max): exactly 1 for the larger state and exp(-|x0 - x1|) for the
// other (x1 - x0 is exactly -(x0 - x1)), so one exp per locus.  The current
// column's is finite; exp(-inf) = 0 for an illegal flip.  The difference is
// formed in FP64 in both precisions.  Returns whether both states are
// possible in FP64 terms (the FP32 pass draws where the FP64 one would).
template <typename T>
__device__ __forceinline__ bool emissions(bool cur, double lcur, double lflip, T* e0, T* e1) {
    const double x0 = cur ? lflip : lcur, x1 = cur ? lcur : lflip;
    const double d = x0 - x1;
    const bool first = d >= 0.0;
    const T t = exp_t((T)(first ? -d : d));
    *e0 = first ? (T)1 : t;
    *e1 = first ? t : (T)1;
    return fabs(d) < kFp64DrawLimit;
}

// 1 when locus l draws a uniform: both weighted states non-zero (:193-203).
// FP64 decides it from the forward values as the reference does; FP32 takes
// the FP64 emission test (`both`), so that it consumes the same draws.
template <typename T>
__device__ __forceinline__ uint32_t locus_draws(const MsampArgs& A, T f0, T f1, int l, bool both) {
    if constexpr (sizeof(T) == 4) {
        return both ? 1u : 0u;
    } else {
        const double t = l < A.M - 1 ? A.theta[l] : 1.0, a = l < A.M - 1 ? 1.0 - A.theta[l] : 1.0;
        return (f0 * a != 0.0 && f1 * t != 0.0) ? 1u : 0u;
    }
}

// uniforms within this distance of a threshold are counted as near an edge:
// the reassociated FP64 sums move thresholds by rounding; FP32 by its epsilon
// times the depth of the product scan
template <typename T>
__device__ __forceinline__ double edge_tol() { return sizeof(T) == 4 ? 1e-5 : 1e-12; }

// 4-bit decision map of a locus (`last`: locus M-1; theta: of the interval to
// the next locus): bit bn = new indicator when the next locus's is bn; bit
// 2+bn = that decision's uniform u lay within edge_tol of its threshold.  A
// drawing locus (draws, from locus_draws) takes u; locus_map draws it as draw
// index ctr of step k.
template <typename T>
__device__ __forceinline__ uint32_t locus_map_u(bool last, double theta, T f0, T f1, double u, bool draws,
                                                uint32_t* near) {
    T w0[2], w1[2];
    if (!last) {
        const T th = (T)theta, an = (T)(1.0 - theta);
        w0[0] = f0 * an;
        w1[0] = f1 * th;
        w0[1] = f0 * th;
        w1[1] = f1 * an;
    } else {
        w0[0] = w0[1] = f0;
        w1[0] = w1[1] = f1;
    }
    if constexpr (sizeof(T) == 8) {
        // with theta in (0, 1) whether a locus draws does not depend on the next
        // indicator; a difference (underflow in one branch only) is counted
        if (draws != (w0[1] != 0.0 && w1[1] != 0.0)) ++*near;
    } else {
        // an FP32 underflow of a state the FP64 pass keeps is counted
        if (draws && !(w0[0] != 0.0f && w1[0] != 0.0f && w0[1] != 0.0f && w1[1] != 0.0f)) ++*near;
    }
    // w0 = 0 gives a threshold of 0 (0/0: NaN) and so bit 1, w1 = 0 one of 1 and
    // so bit 0, for any u in [0, 1)
    uint32_t map = 0;
#pragma unroll
    for (int bn = 0; bn < 2; ++bn) {
        const double thr = (double)(w0[bn] / (w0[bn] + w1[bn]));
        const uint32_t b = u < thr ? 0u : 1u;
        const uint32_t edge = w0[bn] != (T)0 && w1[bn] != (T)0 && fabs(u - thr) < edge_tol<T>() ? 1u : 0u;
        map |= (b << bn) | (edge << (2 + bn));
    }
    return map;
}

template <typename T>
__device__ __forceinline__ uint32_t locus_map(const MsampArgs& A, int chain, int k, T f0, T f1, int l,
                                              uint32_t ctr, bool draws, uint32_t* near) {
    const double u = draws ? philox_uniform(A.seed, (uint32_t)chain, sweep_of(A), (uint32_t)k, ctr) : 0.0;
    return locus_map_u(l == A.M - 1, l < A.M - 1 ? A.theta[l] : 0.0, f0, f1, u, draws, near);
}

// exclusive left-to-right product of the threads' segment products: within
// wavefronts by DPP, across them through LDS (by one row of lanes when there
// are more than four).  The one barrier also publishes what the caller wrote
// to LDS before.
template <typename T>
__device__ __forceinline__ MatT<T> scan_products(MatT<T> P, MatT<T>* wtot) {
    const int lane = lane_id(), nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    P = wave_products(P);
    if (lane == 63) wtot[wave] = P;
    __syncthreads();
    MatT<T> R{(T)1, (T)0, (T)0, (T)1};
    if (nw <= 4) {
        for (int q = 0; q < wave; ++q) R = mmul(R, wtot[q]);
    } else {
        MatT<T> Q = lane < nw ? wtot[lane] : MatT<T>{(T)1, (T)0, (T)0, (T)1};
        Q = mmul(mat_dpp<dpp_row_shr(1)>(Q), Q);
        Q = mmul(mat_dpp<dpp_row_shr(2)>(Q), Q);
        Q = mmul(mat_dpp<dpp_row_shr(4)>(Q), Q);
        if (nw > 8) Q = mmul(mat_dpp<dpp_row_shr(8)>(Q), Q);  // lanes below 8 have no source
        if (wave > 0)
            R = MatT<T>{readlane_t(Q.a, wave - 1), readlane_t(Q.b, wave - 1), readlane_t(Q.c, wave - 1),
                        readlane_t(Q.d, wave - 1)};
    }
    return mmul(R, mat_dpp<kDppWaveShr1>(P));
}

// Draws and decision maps are single bits per (thread, locus of its segment),
// so their scans across a wavefront are ballots: a suffix count is the number
// of set bits above the lane, and a composition of 2-bit maps is the nearest
// constant map above, inverted by each inverting map on the way.

// bits of m above this lane
__device__ __forceinline__ uint32_t count_above(uint64_t m) {
    const uint32_t upto = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    return (uint32_t)__popcll(m) - upto - (uint32_t)((m >> lane_id()) & 1ull);
}

// the total over the wavefronts after this one of per-wavefront counts
__device__ __forceinline__ uint32_t counts_after(const uint32_t* wcnt) {
    const int lane = lane_id(), wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    uint32_t v = lane < nw && lane > wave ? wcnt[lane] : 0u;
    v += u32_dpp<dpp_row_shr(1)>(0u, v);
    v += u32_dpp<dpp_row_shr(2)>(0u, v);
    v += u32_dpp<dpp_row_shr(4)>(0u, v);
    v += u32_dpp<dpp_row_shr(8)>(0u, v);
    return readlane_u32(v, 15);  // at most 16 wavefronts
}

// per-thread bit counts v (a ballot per locus of the segments, formed by the
// caller's masks): the sum over the threads after this one; wave_total is the
// wavefront's sum
template <int SM>
__device__ __forceinline__ uint32_t sum_above_bits(uint32_t bits, uint32_t* wave_total) {
    uint32_t r = 0, tot = 0;
#pragma unroll
    for (int s = 0; s < SM; ++s) {
        const uint64_t m = __ballot((bits >> s) & 1u);
        r += count_above(m);
        tot += (uint32_t)__popcll(m);
    }
    *wave_total = tot;
    return r;
}

// within a wavefront: inclusive suffix sums of v (this lane and the lanes
// after it)
__device__ __forceinline__ uint32_t wave_suffix_sums(uint32_t v) {
    const int lane = lane_id();
    uint32_t sc = v;  // within rows, then across them
    sc += u32_dpp<dpp_row_shl(1)>(0u, sc);
    sc += u32_dpp<dpp_row_shl(2)>(0u, sc);
    sc += u32_dpp<dpp_row_shl(4)>(0u, sc);
    sc += u32_dpp<dpp_row_shl(8)>(0u, sc);
    const uint32_t t1 = readlane_u32(sc, 16), t2 = readlane_u32(sc, 32), t3 = readlane_u32(sc, 48);
    const int row = lane >> 4;
    return sc + (row < 1 ? t1 : 0u) + (row < 2 ? t2 : 0u) + (row < 3 ? t3 : 0u);
}

// sum of v over the threads after this one
__device__ __forceinline__ uint32_t sum_above(uint32_t v, uint32_t* wcnt) {
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    const uint32_t sc = wave_suffix_sums(v);
    if (lane == 0) wcnt[wave] = sc;
    __syncthreads();
    return sc - v + counts_after(wcnt);
}

// image of anything under the composition of the maps of the lanes in `sel`
// (lowest applied last): cst: constant maps, one: those giving 1, neg:
// inverting maps; `in` enters above the topmost lane
__device__ __forceinline__ uint32_t through_maps(uint64_t cst, uint64_t one, uint64_t neg, uint32_t in) {
    const int j = cst ? __ffsll((unsigned long long)cst) - 1 : 64;
    const uint64_t below = j < 64 ? (1ull << j) - 1ull : ~0ull;
    const uint32_t v = cst ? (uint32_t)((one >> j) & 1ull) : in;
    return v ^ ((uint32_t)__popcll(neg & below) & 1u);
}

// indicator entering this thread's segment from above: the composition of the
// segment maps of every later thread applied to anything (the map of locus M-1
// is constant, so the composite is too)
__device__ __forceinline__ uint32_t bit_from_above(uint32_t comp, uint32_t* wmap) {
    const int lane = lane_id(), nw = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint64_t cst = __ballot(comp == 0u || comp == 3u), one = __ballot(comp == 3u), neg = __ballot(comp == 1u);
    if (lane == 0) wmap[wave] = through_maps(cst, one, neg, 0u) | (through_maps(cst, one, neg, 1u) << 1);
    __syncthreads();
    const uint32_t wm = lane < nw && lane > wave ? wmap[lane] : 2u;
    const uint32_t up = through_maps(__ballot(wm == 0u || wm == 3u), __ballot(wm == 3u), __ballot(wm == 1u), 0u);
    const uint64_t above = lane < 63 ? ~0ull << (lane + 1) : 0ull;
    return through_maps(cst & above, one, neg & above, up);
}

// Forward-backward pass of step k on one chain by the whole workgroup; thread
// t owns a contiguous segment of loci.  Scans run within wavefronts by lane
// shuffles and across them through LDS.  SM > 0: segments of at most SM loci
// whose likelihoods, forward probabilities and maps stay in registers; SM = 0:
// any length, through the chain's global scratch.  T: the arithmetic of the
// forward values and thresholds.  A chain whose status is set or whose sweep
// is an L-sweep is left as it is.  ubuf (SM > 0, may be null): LDS for the M
// uniforms that draw indices 0..M-1 of the step take.
template <int SM, typename T>
__device__ void forward_backward(const MsampArgs& A, int chain, int k, MatT<T>* wtot, uint32_t* wcnt,
                                 uint32_t* wmap, double* ubuf) {
    const int B = blockDim.x, tid = threadIdx.x, M = A.M;
    if (!is_msweep(A, chain)) return;
    // the status is read beside the meiosis order (an illegal chain's order
    // may be stale) and checked before any load the order addresses
    const int status = A.status[chain];
    const int m = order_at(A, chain, k);
    StepView sv;
    sv.A = &A;
    sv.chain = chain;
    sv.k = k;
    sv.word = m >> 5;
    sv.bm = 1u << (m & 31);
    sv.spec = A.spec && k > 0;
    sv.cls = A.cls + (size_t)m * M;
    const int pm = sv.spec ? order_at(A, chain, k - 1) : 0;
    if (status != 0) return;
    sv.pword = pm >> 5;
    sv.pbm = 1u << (pm & 31);
    const int word = sv.word;
    const uint32_t bm = sv.bm;
    uint32_t* g = A.graphs + (size_t)chain * M * A.W;
    double* lc = A.lcur + (size_t)chain * M;
    const int S = (M + B - 1) / B;
    const int a0 = min(M, tid * S), a1 = min(M, a0 + S);
    uint32_t near = 0;
    if constexpr (SM > 0) {
        // every load of the pass at once: the column words holding m_k and
        // m_{k-1}, the current column's likelihood, both flipped variants and
        // the thetas of the segment's intervals
        uint32_t gw[SM], pw[SM];
        int cl[SM];
        double lcv[SM], lf0[SM], lf1[SM], thv[SM + 1];
#pragma unroll
        for (int s = 0; s <= SM; ++s) {
            const int i = a0 + s - 1;  // interval i joins loci i and i+1
            thv[s] = (i >= 0 && i < M - 1 && a0 + s - 1 < a1) ? A.theta[i] : 0.0;
        }
#pragma unroll
        for (int s = 0; s < SM; ++s) {
            const int l = a0 + s;
            gw[s] = pw[s] = 0u;
            lcv[s] = lf0[s] = lf1[s] = 0.0;
            cl[s] = kFlipCompute;
            if (l < a1) {
                cl[s] = sv.cls[l];
                gw[s] = g[(size_t)l * A.W + word];
                lcv[s] = lc[l];
                lf0[s] = A.lflip[lflip_index(A, k, 0, chain, l)];
                if (sv.spec) {
                    pw[s] = g[(size_t)l * A.W + sv.pword];
                    lf1[s] = A.lflip[lflip_index(A, k, 1, chain, l)];
                }
            }
        }
        // the step's uniforms by draw index, drawn beside the step's
        // likelihoods (the first barrier of the scans below publishes them)
        if (ubuf) {
            const double* ud = A.udev + udev_index(A, k, chain);
            double uv[SM];
#pragma unroll
            for (int s = 0; s < SM; ++s) uv[s] = tid + s * B < M ? ud[tid + s * B] : 0.0;
#pragma unroll
            for (int s = 0; s < SM; ++s)
                if (tid + s * B < M) ubuf[tid + s * B] = uv[s];
        }
        T e0[SM], e1[SM], f0[SM], f1[SM];
        double lfv[SM];
        uint32_t curm = 0, drm = 0, both = 0;
#pragma unroll
        for (int s = 0; s < SM; ++s) {
            const bool cur = (gw[s] & bm) != 0;
            lfv[s] = (pw[s] & sv.pbm) ? lf1[s] : lf0[s];
            if (cl[s] != kFlipCompute) lfv[s] = cl[s] == kFlipSame ? lcv[s] : -INFINITY;
            e0[s] = e1[s] = (T)0;
            if (a0 + s < a1) both |= (emissions(cur, lcv[s], lfv[s], &e0[s], &e1[s]) ? 1u : 0u) << s;
            curm |= (cur ? 1u : 0u) << s;
        }
        MatT<T> P{(T)1, (T)0, (T)0, (T)1};
#pragma unroll
        for (int s = 0; s < SM; ++s)
            if (a0 + s < a1) P = mmul(P, emission_matrix_th(e0[s], e1[s], a0 + s == 0, thv[s]));
        // the backward pass runs from the last locus down, so a drawing
        // locus's draw index counts the draws of later threads and of the
        // later loci of this segment.  FP32 draws where FP64 emissions allow
        // both states, known before the forward pass: the products' barrier
        // then publishes the counts too
        uint32_t cnt, wtotal;
        if constexpr (sizeof(T) == 4) {
            drm = both;
            cnt = sum_above_bits<SM>(drm, &wtotal);
            if (lane_id() == 0) wcnt[tid >> 6] = wtotal;
        }
        MatT<T> R = scan_products(P, wtot);
#pragma unroll
        for (int s = 0; s < SM; ++s) {
            f0[s] = f1[s] = (T)0;
            if (a0 + s < a1) {
                R = mmul(R, emission_matrix_th(e0[s], e1[s], a0 + s == 0, thv[s]));
                f0[s] = R.a + R.c;
                f1[s] = R.b + R.d;
                if constexpr (sizeof(T) == 8) {
                    const bool last = a0 + s == M - 1;
                    const double t = last ? 1.0 : thv[s + 1], a = last ? 1.0 : 1.0 - thv[s + 1];
                    drm |= ((f0[s] * a != 0.0 && f1[s] * t != 0.0) ? 1u : 0u) << s;
                }
            }
        }
        if constexpr (sizeof(T) == 8) {
            cnt = sum_above_bits<SM>(drm, &wtotal);
            if (lane_id() == 0) wcnt[tid >> 6] = wtotal;
            __syncthreads();
        }
        cnt += counts_after(wcnt);
        uint32_t mp[SM];
#pragma unroll
        for (int s = 0; s < SM; ++s) {
            mp[s] = 0u;
            if (a0 + s < a1) {
                const bool dr = ((drm >> s) & 1u) != 0u;
                const uint32_t ctr = cnt + (uint32_t)__popc(drm >> (s + 1));
                const double u = !dr ? 0.0
                                 : ubuf ? ubuf[ctr]
                                        : philox_uniform(A.seed, (uint32_t)chain, sweep_of(A), (uint32_t)k, ctr);
                mp[s] = locus_map_u(a0 + s == M - 1, thv[s + 1], f0[s], f1[s], u, dr, &near);
            }
        }
        uint32_t comp = 2u;  // identity
#pragma unroll
        for (int s = SM - 1; s >= 0; --s)
            if (a0 + s < a1) comp = compose(mp[s] & 3u, comp);
        uint32_t next = bit_from_above(comp, wmap);
#pragma unroll
        for (int s = SM - 1; s >= 0; --s) {
            const int l = a0 + s;
            if (l < a1) {
                const uint32_t nb = (mp[s] >> next) & 1u;
                near += (mp[s] >> (2 + next)) & 1u;
                if (nb != ((curm >> s) & 1u)) {
                    g[(size_t)l * A.W + word] ^= bm;
                    lc[l] = lfv[s];
                }
                next = nb;
            }
        }
    } else {
        double* fb = A.fbuf + (size_t)chain * M * 2;
        uint8_t* mp = A.maps + (size_t)chain * M;
        auto locus = [&](int l, bool* both) {
            T e0, e1;
            const bool b = emissions((g[(size_t)l * A.W + word] & bm) != 0, lc[l], sv.lf(g, l, lc[l]), &e0, &e1);
            if (both) *both = b;
            return emission_matrix(A, e0, e1, l);
        };
        MatT<T> P{(T)1, (T)0, (T)0, (T)1};
        for (int l = a0; l < a1; ++l) P = mmul(P, locus(l, nullptr));
        MatT<T> R = scan_products(P, wtot);
        uint32_t draws = 0;
        for (int l = a0; l < a1; ++l) {
            bool both;
            R = mmul(R, locus(l, &both));
            fb[2 * l] = (double)(R.a + R.c);
            fb[2 * l + 1] = (double)(R.b + R.d);
            draws += locus_draws(A, R.a + R.c, R.b + R.d, l, both);
        }
        uint32_t cnt = sum_above(draws, wcnt);
        uint32_t comp = 2u;
        for (int l = a1 - 1; l >= a0; --l) {
            bool both;
            (void)locus(l, &both);
            const T f0 = (T)fb[2 * l], f1 = (T)fb[2 * l + 1];
            const bool dr = locus_draws(A, f0, f1, l, both) != 0u;
            const uint32_t map = locus_map(A, chain, k, f0, f1, l, cnt, dr, &near);
            cnt += dr ? 1u : 0u;
            mp[l] = (uint8_t)map;
            comp = compose(map & 3u, comp);
        }
        uint32_t next = bit_from_above(comp, wmap);
        for (int l = a1 - 1; l >= a0; --l) {
            const uint32_t map = mp[l];
            const uint32_t nb = (map >> next) & 1u;
            near += (map >> (2 + next)) & 1u;
            uint32_t* wp = g + (size_t)l * A.W + word;
            if (nb != ((*wp & bm) ? 1u : 0u)) {
                lc[l] = sv.lf(g, l, lc[l]);
                *wp ^= bm;
            }
            next = nb;
        }
    }
    if (near) atomicAdd(&A.near_edge[chain], near);
}

// The workgroup's jobs of a chain in an M-sweep.  The register-resident
// likelihood reads its slots of the person table with its other loads; the
// LDS one reads a copy staged once per workgroup.
template <int KC>
__device__ __forceinline__ void run_jobs(const MsampArgs& A, int chain, int block, unsigned char* smem) {
    if (!is_msweep(A, chain)) return;
    const int nw = blockDim.x >> 6, wave = threadIdx.x >> 6;
    const int job_blocks = (A.n_jobs + nw - 1) / nw;
    if (block >= job_blocks) {
        // the workgroups past the jobs draw the step's uniforms: a Philox
        // call is 20 quarter-rate multiplies, which the forward-backward
        // pass's one workgroup would wait for
        const int i = (block - job_blocks) * (int)blockDim.x + (int)threadIdx.x;
        if (i < A.M)
            A.udev[udev_index(A, A.step, chain) + i] =
                philox_uniform(A.seed, (uint32_t)chain, sweep_of(A), (uint32_t)A.step, (uint32_t)i);
        return;
    }
    uint2* ptab = reinterpret_cast<uint2*>(smem);
    if constexpr (KC == 0) {
        for (int k = threadIdx.x; k < A.N - A.F; k += blockDim.x) ptab[k] = A.ptab[k];
        __syncthreads();
    }
    const int q = block * nw + wave;
    if (q < A.n_jobs) fag_job<KC>(A, chain, q, ptab, smem + A.ptab_bytes + (size_t)wave * A.wave_bytes);
}

// The planned jobs of step A.step: the flips to compute over all chains, in the
// plan's order, shared by n_waves wavefronts.  A grid of one job slot per chain
// and locus of the longest list sized every step for its worst meiosis, and most
// wavefronts only found out that they had nothing to do: 64 chains of 150 people
// 19.1 us a launch, planned 14.5; 32 chains of 600 people, whose jobs fill the
// device, 53 and 51.5.  With A.spec and k > 0 a job
// gives both variants (fag_job), the second from the same inputs.
template <int KC>
__device__ __forceinline__ void planned_jobs(const MsampArgs& A, uint32_t wave, uint32_t n_waves, const uint2* ptab,
                                             unsigned char* smem, int area) {
    const int M = A.M;
    const uint2* row = A.plan + (size_t)A.step * A.n_chains;
    const uint32_t total = A.plan_total[A.step];
    const bool two = A.spec && A.step > 0;
    for (uint32_t q = wave; q < total; q += n_waves) {
        const int lane = opaque_v(lane_id()), F = opaque_s(A.F);
        const WaveArea w = wave_area(A, smem + opaque_s(area));
        // its chain: the last whose first job is at or below q, 64 candidates a round
        int chain = 0, n = A.n_chains, flip, stride;
        uint32_t first;
        do {
            stride = (n + 63) >> 6;
            const int i = lane * stride;
            const uint2 r = i < n ? row[chain + i] : make_uint2(~0u, 0u);
            const int at = __popcll(__ballot(r.x <= q)) - 1;
            first = readlane_u32(r.x, at);
            flip = (int)readlane_u32(r.y, at);
            chain += at * stride;
            n = n - at * stride < stride ? n - at * stride : stride;
        } while (stride > 1);
        const int l = A.joblist[(size_t)flip * M + (q - first)];
        const int status = A.status[chain];
        int force = two ? (int)A.plan[(size_t)(A.step - 1) * A.n_chains + chain].y : -1;
        const int pc = two ? A.cls[(size_t)force * M + l] : kFlipSame;
        if (pc == kFlipIllegal) force = -1;
        const uint32_t* src = A.graphs + ((size_t)chain * M + l) * A.W;
        double* const dst = A.lflip + lflip_index(A, A.step, 0, chain, l);
        double* const dst1 = A.lflip + lflip_index(A, A.step, 1, chain, l);
        JobInputs<KC> in;
        if constexpr (KC > 0) {
            in.load(A, l);
            for (int f = lane; f < F; f += 64)
                *reinterpret_cast<uint32_t*>(w.lab + 2 * f) = (uint32_t)(2 * f) | ((uint32_t)(2 * f + 1) << 16);
        }
        for (int k = lane; k < A.W; k += 64) {
            uint32_t x = src[k];
            if (force >= 0 && (force >> 5) == k) x &= ~(1u << (force & 31));
            if ((flip >> 5) == k) x ^= 1u << (flip & 31);
            w.colw[k] = x;
        }
        if (status != 0) continue;  // illegal since the plan was made
        const int variants = two && pc == kFlipCompute ? 2 : 1;
        for (int v = 0; v < variants; ++v) {
            if (v && lane == 0) w.colw[force >> 5] ^= 1u << (force & 31);
            if constexpr (KC > 0)
                for (int x = lane; x < 2 * F; x += 64) w.acc[x] = 0u;
            wave_sync();
            double L;
            if constexpr (KC > 0) L = fag_log_likelihood_r<KC>(A, in, w, l);
            else L = fag_log_likelihood(A, ptab, w, l);
            if (lane == 0) {
                *(v ? dst1 : dst) = L;
                if (two && variants == 1) *dst1 = L;
            }
            wave_sync();
        }
    }
}

// A workgroup of a planned launch: the first n_job_blocks take the jobs, the
// others draw step A.step's uniforms.
template <int KC>
__device__ __forceinline__ void planned_block(const MsampArgs& A, int block, int n_job_blocks, unsigned char* smem) {
    const int nw = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (block >= n_job_blocks) {
        const int per_chain = (A.M + (int)blockDim.x - 1) / (int)blockDim.x;
        const int chain = (block - n_job_blocks) / per_chain;
        const int i = (block - n_job_blocks) % per_chain * (int)blockDim.x + (int)threadIdx.x;
        if (i < A.M && is_msweep(A, chain))
            A.udev[udev_index(A, A.step, chain) + i] =
                philox_uniform(A.seed, (uint32_t)chain, sweep_of(A), (uint32_t)A.step, (uint32_t)i);
        return;
    }
    uint2* ptab = reinterpret_cast<uint2*>(smem);
    if constexpr (KC == 0) {
        for (int k = threadIdx.x; k < A.N - A.F; k += blockDim.x) ptab[k] = A.ptab[k];
        __syncthreads();
    }
    planned_jobs<KC>(A, (uint32_t)(block * nw + wave), (uint32_t)(n_job_blocks * nw), ptab, smem,
                     A.ptab_bytes + wave * A.wave_bytes);
}

// The plan of a sweep: for every step the chains' jobs, summed over the chains
// before.  One workgroup per step.
constexpr int kPlanBlock = 256;
__global__ void __launch_bounds__(kPlanBlock) mplan_kernel(MsampArgs A) {
    __shared__ uint32_t wsum[kPlanBlock / 64];
    const int k = blockIdx.x, tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
    uint32_t before = 0;
    for (int c0 = 0; c0 < A.n_chains; c0 += kPlanBlock) {
        const int c = c0 + tid;
        int flip = 0;
        uint32_t cnt = 0;
        if (c < A.n_chains && A.status[c] == 0 && is_msweep(A, c)) {
            flip = order_at(A, c, k);
            cnt = (uint32_t)A.jobcnt[flip];
        }
        uint32_t up = cnt;  // inclusive over the wavefront
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t x = (uint32_t)__shfl_up((int)up, d);
            if (lane >= d) up += x;
        }
        if (lane == 63) wsum[wave] = up;
        __syncthreads();
        uint32_t mine = before + up - cnt;
        for (int x = 0; x < kPlanBlock / 64; ++x) {
            if (x < wave) mine += wsum[x];
            before += wsum[x];
        }
        if (c < A.n_chains) A.plan[(size_t)k * A.n_chains + c] = make_uint2(mine, (uint32_t)flip);
        __syncthreads();
    }
    if (tid == 0) A.plan_total[k] = before;
}

// What flipping a meiosis does to a legal column, for every meiosis and locus,
// by genotype elimination (a descent graph only adds constraints, so what no
// assignment of phased genotypes to the family allows, no column allows).  A
// thread per locus keeps each person's possible (maternal, paternal) alleles
// as a 4-bit mask, bit 2 maternal + paternal, and narrows every trio down and
// up the generations until nothing changes.  Any narrowing is sound, so the
// rounds are bounded; two or three settle.  For a meiosis of person p from
// parent q:
//  * q cannot be heterozygous: in every assignment consistent with a column q's
//    two founder alleles are equal, so exchanging them in the edges below p
//    keeps every constraint: flipping the bit leaves the likelihood as it is;
//  * q is heterozygous with known phase and the allele p took from q is known:
//    the bit is fixed, and the flipped column has no consistent assignment.
// At ped150 (10% missing) 55% of the (meiosis, locus) pairs are the first,
// and together about two thirds need no founder-allele graph.
constexpr int kClassBlock = 64;
constexpr int kClassRounds = 8;

__device__ __forceinline__ uint32_t transmits(uint32_t m) { return ((m & 0x7u) ? 1u : 0u) | ((m & 0xEu) ? 2u : 0u); }
__device__ __forceinline__ uint32_t maternal_alleles(uint32_t m) {
    return ((m & 0x3u) ? 1u : 0u) | ((m & 0xCu) ? 2u : 0u);
}
__device__ __forceinline__ uint32_t paternal_alleles(uint32_t m) {
    return ((m & 0x5u) ? 1u : 0u) | ((m & 0xAu) ? 2u : 0u);
}
__device__ __forceinline__ uint32_t carries(uint32_t s) { return ((s & 1u) ? 0x7u : 0u) | ((s & 2u) ? 0xEu : 0u); }

__global__ void __launch_bounds__(kClassBlock) mclass_kernel(MsampArgs A, uint8_t* masks, uint8_t* cls) {
    const int l = blockIdx.x * kClassBlock + threadIdx.x;
    if (l >= A.M) return;
    const int M = A.M, F = A.F, NF = A.N - F;
    uint8_t* mk = masks + l;
    for (int i = 0; i < A.N; ++i) {
        const int g = genotype_at(A, l, i);
        mk[(size_t)i * M] = g == 0 ? 0xFu : g == G_HETERO ? 0x6u : g == G_HOMOZ_B ? 0x8u : 0x1u;
    }
    for (int round = 0; round < kClassRounds; ++round) {
        bool changed = false;
        for (int j = 0; j < 2 * NF; ++j) {
            const uint2 e = A.ptab[j < NF ? j : 2 * NF - 1 - j];  // down the generations, then up
            uint8_t* pc = mk + (size_t)(e.x & 0xFFFFu) * M;
            uint8_t* pm = mk + (size_t)(e.y & 0xFFFFu) * M;
            uint8_t* pf = mk + (size_t)(e.y >> 16) * M;
            const uint32_t c = *pc, mo = *pm, fa = *pf;
            const uint32_t tm = transmits(mo), tf = transmits(fa);
            const uint32_t c2 = c & (((tm & 1u) ? 0x3u : 0u) | ((tm & 2u) ? 0xCu : 0u)) &
                                (((tf & 1u) ? 0x5u : 0u) | ((tf & 2u) ? 0xAu : 0u));
            const uint32_t m2 = mo & carries(maternal_alleles(c2)), f2 = fa & carries(paternal_alleles(c2));
            if (c2 != c) *pc = (uint8_t)c2;
            if (m2 != mo) *pm = (uint8_t)m2;
            if (f2 != fa) *pf = (uint8_t)f2;
            changed |= c2 != c || m2 != mo || f2 != fa;
        }
        if (!changed) break;
    }
    for (int j = 0; j < NF; ++j) {
        const uint2 e = A.ptab[j];
        const int p = (int)(e.x & 0xFFFFu);
        const uint32_t c = mk[(size_t)p * M];
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            const uint32_t q = mk[(size_t)(side ? e.y >> 16 : e.y & 0xFFFFu) * M];
            const uint32_t got = side ? paternal_alleles(c) : maternal_alleles(c);
            int k = kFlipCompute;
            if (q != 0u && (q & 0x6u) == 0u) k = kFlipSame;
            else if ((q == 0x2u || q == 0x4u) && (got == 1u || got == 2u)) k = kFlipIllegal;
            cls[(size_t)(2 * (p - F) + side) * M + l] = (uint8_t)k;
        }
    }
}

// the kFlipCompute loci of meiosis blockIdx.x, ascending; one wavefront
__global__ void __launch_bounds__(64) mjobs_kernel(int M, const uint8_t* cls, int32_t* joblist, int32_t* jobcnt) {
    const int b = blockIdx.x, lane = threadIdx.x;
    const uint64_t below = (1ull << lane) - 1ull;
    int n = 0;
    for (int l0 = 0; l0 < M; l0 += 64) {
        const int l = l0 + lane;
        const bool take = l < M && cls[(size_t)b * M + l] == kFlipCompute;
        const uint64_t mask = __ballot(take);
        if (take) joblist[(size_t)b * M + n + __popcll(mask & below)] = l;
        n += __popcll(mask);
    }
    if (lane == 0) jobcnt[b] = n;
}

// founder-allele likelihood jobs only; grid (jobs / waves, chains).  KC > 0:
// the register-resident likelihood for at most 64*KC people
template <int KC>
__global__ void __launch_bounds__(kMsampBlock) mstep_kernel(MsampArgs A) {
    extern __shared__ __align__(16) unsigned char smem[];
    run_jobs<KC>(A, blockIdx.y, blockIdx.x, smem);
}

// forward-backward pass of step fb_step only; one workgroup per chain.  The
// dynamic LDS, when A.fb_ubuf, holds the step's uniforms.
template <int SM, typename T>
__global__ void __launch_bounds__(kFbBlock) mfb_kernel(MsampArgs A) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ MatT<T> wtot[kFbBlock / 64];
    __shared__ uint32_t wcnt[kFbBlock / 64], wmap[kFbBlock / 64];
    forward_backward<SM, T>(A, blockIdx.x, A.fb_step, wtot, wcnt, wmap,
                            A.fb_ubuf ? reinterpret_cast<double*>(smem) : nullptr);
}

// one speculative launch: workgroup 0 of each chain runs step fb_step's
// forward-backward pass while the others run the jobs of step fb_step + 1
template <int SM, int KC, typename T>
__global__ void __launch_bounds__(kSpecBlock) mspec_kernel(MsampArgs A) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ MatT<T> wtot[kSpecBlock / 64];
    __shared__ uint32_t wcnt[kSpecBlock / 64], wmap[kSpecBlock / 64];
    if (blockIdx.x == 0)
        forward_backward<SM, T>(A, blockIdx.y, A.fb_step, wtot, wcnt, wmap,
                                A.fb_ubuf ? reinterpret_cast<double*>(smem) : nullptr);
    else
        run_jobs<KC>(A, blockIdx.y, blockIdx.x - 1, smem);
}

// planned jobs only
template <int KC>
__global__ void __launch_bounds__(kMsampBlock) mplanned_kernel(MsampArgs A) {
    extern __shared__ __align__(16) unsigned char smem[];
    planned_block<KC>(A, blockIdx.x, (A.plan_waves * 64 + kMsampBlock - 1) / kMsampBlock, smem);
}

// the first workgroups run step fb_step's forward-backward pass, one chain each,
// in mfb_kernel's shape (the same scans, the same rounding), the others the
// planned jobs of step fb_step + 1
template <int SM, int KC, typename T>
__global__ void __launch_bounds__(kFbBlock) mbeside_kernel(MsampArgs A) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ MatT<T> wtot[kFbBlock / 64];
    __shared__ uint32_t wcnt[kFbBlock / 64], wmap[kFbBlock / 64];
    const int b = blockIdx.x;
    if (b < A.n_chains)
        forward_backward<SM, T>(A, b, A.fb_step, wtot, wcnt, wmap, A.fb_ubuf ? reinterpret_cast<double*>(smem) : nullptr);
    else
        planned_block<KC>(A, b - A.n_chains, (A.plan_waves * 64 + kFbBlock - 1) / kFbBlock, smem);
}

// this sweep's meiosis order: the given order, or a Fisher-Yates shuffle of the
// non-ignorable meioses (random_shuffle, markov_chain.cc:346) driven by the
// chain's draws at step kStepShuffle.  Position i (from the top, i = n-1 .. 1)
// swaps with floor(u_d (i+1)), d = n-1-i.  The swap partners are drawn in
// parallel into LDS.  Up to kOrderChunk meioses, every output position follows
// its element back through the swaps (last swap first), all positions at once:
// n^2 compares instead of a chain of n dependent memory round trips.  Larger
// orders swap in global memory one after another, kOrderChunk partners per pass.
// One workgroup per chain.
constexpr int kOrderBlock = 1024;
constexpr int kOrderChunk = 1024;

__device__ __forceinline__ int shuffle_partner(const MsampArgs& A, int chain, int n, int i) {
    const double u = philox_uniform(A.seed, (uint32_t)chain, sweep_of(A), kStepShuffle, (uint32_t)(n - 1 - i));
    const int j = (int)(u * (double)(i + 1));
    return j > i ? i : j;
}

__global__ void __launch_bounds__(kOrderBlock) morder_kernel(MsampArgs A, const int32_t* fixed_order) {
    __shared__ int32_t jdx[kOrderChunk];
    __shared__ int s_skip;
    const int chain = blockIdx.x;
    if (threadIdx.x == 0) s_skip = A.status[chain] != 0 || !is_msweep(A, chain);
    __syncthreads();
    if (s_skip) return;
    const int n = A.n_meioses;
    int32_t* o = A.order + (size_t)chain * n;
    if (fixed_order) {
        for (int i = threadIdx.x; i < n; i += blockDim.x) o[i] = fixed_order[i];
        return;
    }
    if (n <= kOrderChunk) {
        for (int i = threadIdx.x + 1; i < n; i += blockDim.x) jdx[i] = shuffle_partner(A, chain, n, i);
        __syncthreads();
        const int q = threadIdx.x;
        if (q >= n) return;
        // swaps apply for i = n-1 down to 1; undo them from i = 1 up
        int p = q;
#pragma unroll 8
        for (int i = 1; i < n; ++i) {
            const int j = jdx[i];
            p = p == i ? j : p == j ? i : p;
        }
        o[q] = A.meioses[p];
        return;
    }
    for (int i = threadIdx.x; i < n; i += blockDim.x) o[i] = A.meioses[i];
    for (int hi = n - 1; hi > 0; hi -= kOrderChunk) {
        const int lo = hi - kOrderChunk + 1 > 1 ? hi - kOrderChunk + 1 : 1;
        __syncthreads();  // o written; the previous pass's partners consumed
        for (int i = lo + (int)threadIdx.x; i <= hi; i += blockDim.x) jdx[i - lo] = shuffle_partner(A, chain, n, i);
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int i = hi; i >= lo; --i) {
                const int j = jdx[i - lo];
                const int32_t t = o[i];
                o[i] = o[j];
                o[j] = t;
            }
        }
    }
}

// The CODA trace line of each chain (markov_chain.cc:362-370):
// DescentGraph::get_likelihood (descent_graph.cc:184-189), the transmission
// 2(N-F) ln 1/2 plus the recombination log-probability of every interval
// (:195-242), plus ln of the founder-allele likelihood of every locus
// (:244-267) from the current columns' log-likelihoods in lcur; -inf when a
// locus is illegal.  One workgroup per chain.
constexpr int kTraceBlock = 256;
__global__ void __launch_bounds__(kTraceBlock) trace_kernel(MsampArgs A, const double* log_theta,
                                                            const double* log_anti, double trans, double* out) {
    __shared__ double red[2][kTraceBlock / 64];
    __shared__ int s_bad;
    const int chain = blockIdx.x, tid = threadIdx.x, M = A.M, W = A.W;
    const uint32_t* g = A.graphs + (size_t)chain * M * W;
    const double* lc = A.lcur + (size_t)chain * M;
    const int nm = 2 * (A.N - A.F);
    if (tid == 0) s_bad = 0;
    __syncthreads();
    double rec = 0.0, prior = 0.0;
    bool bad = false;
    for (int l = tid; l < M; l += kTraceBlock) {
        const double x = lc[l];
        if (x == -INFINITY) bad = true;
        else prior += x;
        if (l + 1 < M) {
            int nc = 0;
            for (int w = 0; w < W; ++w) nc += __popc(g[(size_t)l * W + w] ^ g[(size_t)(l + 1) * W + w]);
            rec += (double)nc * log_theta[l] + (double)(nm - nc) * log_anti[l];
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        rec += __shfl_xor(rec, off);
        prior += __shfl_xor(prior, off);
    }
    if (bad) s_bad = 1;
    if (lane_id() == 0) {
        red[0][tid >> 6] = rec;
        red[1][tid >> 6] = prior;
    }
    __syncthreads();
    if (tid == 0) {
        double r = 0.0, p = 0.0;
        for (int w = 0; w < kTraceBlock / 64; ++w) {
            r += red[0][w];
            p += red[1][w];
        }
        out[chain] = s_bad ? -INFINITY : (trans + r) + p;  // log_product(transmission, prior)
    }
}

}  // namespace

hipError_t launch_trace(const MsampArgs& A, const double* log_theta, const double* log_anti, double trans, double* out,
                        hipStream_t s) {
    hipLaunchKernelGGL(trace_kernel, dim3(A.n_chains), dim3(kTraceBlock), 0, s, A, log_theta, log_anti, trans, out);
    return hipGetLastError();
}

bool msampler_supported(int N, int F) { return F >= 1 && 2 * F <= kMaxFagNodes && N <= 65535; }

int msampler_people_chunks(int N, int F) {
    const int n = N > 2 * F ? N : 2 * F;  // people and founder alleles, 64 per chunk
    return n <= 128 ? 2 : n <= 192 ? 3 : n <= 256 ? 4 : n <= 384 ? 6 : n <= 512 ? 8 : n <= 768 ? 12 : n <= 1024 ? 16 : 0;
}

size_t msampler_wave_bytes(int N, int F, int W) {
    const size_t labelled = msampler_people_chunks(N, F) ? (size_t)N : (size_t)(N - F);
    const size_t b = 4 * (size_t)W + 2 * 4 * (size_t)(2 * F) + 4 * (size_t)N + 2 * 2 * labelled;
    return (b + 15) / 16 * 16;
}

size_t msampler_ptab_bytes(int N, int F) { return ((size_t)(N - F) * 8 + 15) / 16 * 16; }

size_t msampler_lds_bytes(const MsampArgs& A, int block) {
    return (size_t)A.ptab_bytes + (size_t)(block / 64) * (size_t)A.wave_bytes;
}

namespace {

// workgroups of `block` threads for a launch's jobs and, where the passes read
// them, its step's uniforms
int job_blocks(const MsampArgs& A, int block) {
    const int nw = block / 64;
    return (A.n_jobs + nw - 1) / nw + (A.fb_ubuf && A.draw_uniforms ? (A.M + block - 1) / block : 0);
}

hipError_t set_lds(const void* kernel, size_t b) {
    if (b <= 64 * 1024) return hipSuccess;
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)b);
}

template <int KC, typename T>
hipError_t set_lds_spec(size_t spec) {
    hipError_t e = set_lds((const void*)mspec_kernel<0, KC, T>, spec);
    if (e == hipSuccess) e = set_lds((const void*)mspec_kernel<1, KC, T>, spec);
    if (e == hipSuccess) e = set_lds((const void*)mspec_kernel<2, KC, T>, spec);
    if (e == hipSuccess) e = set_lds((const void*)mspec_kernel<4, KC, T>, spec);
    if (e == hipSuccess) e = set_lds((const void*)mspec_kernel<8, KC, T>, spec);
    return e;
}

template <int KC, typename T>
hipError_t set_lds_beside(size_t beside) {
    hipError_t e = set_lds((const void*)mbeside_kernel<1, KC, T>, beside);
    if (e == hipSuccess) e = set_lds((const void*)mbeside_kernel<2, KC, T>, beside);
    if (e == hipSuccess) e = set_lds((const void*)mbeside_kernel<4, KC, T>, beside);
    return e;
}

template <int KC>
hipError_t set_lds_kc(size_t job, size_t spec, size_t beside) {
    hipError_t e = set_lds((const void*)mstep_kernel<KC>, job);
    if (e == hipSuccess) e = set_lds((const void*)mplanned_kernel<KC>, job);
    if (e == hipSuccess && beside) e = set_lds_beside<KC, double>(beside);
    if (e == hipSuccess && beside) e = set_lds_beside<KC, float>(beside);
    if (spec == 0) return e;
    if (e == hipSuccess) e = set_lds_spec<KC, double>(spec);
    if (e == hipSuccess) e = set_lds_spec<KC, float>(spec);
    return e;
}

// workgroups of a planned launch: jobs, then the uniforms
int planned_blocks(const MsampArgs& A, int block) {
    return (A.plan_waves * 64 + block - 1) / block +
           (A.fb_ubuf && A.draw_uniforms ? A.n_chains * ((A.M + block - 1) / block) : 0);
}

template <int KC, typename T>
void launch_mbeside_kc(const MsampArgs& A, size_t lds, hipStream_t s) {
    const int seg = (A.M + kFbBlock - 1) / kFbBlock;
    const dim3 grid(A.n_chains + planned_blocks(A, kFbBlock)), block(kFbBlock);
    if (seg <= 1) hipLaunchKernelGGL((mbeside_kernel<1, KC, T>), grid, block, lds, s, A);
    else if (seg <= 2) hipLaunchKernelGGL((mbeside_kernel<2, KC, T>), grid, block, lds, s, A);
    else hipLaunchKernelGGL((mbeside_kernel<4, KC, T>), grid, block, lds, s, A);
}

template <int KC>
void launch_mbeside_kc(const MsampArgs& A, size_t lds, hipStream_t s) {
    if (A.fp32) launch_mbeside_kc<KC, float>(A, lds, s);
    else launch_mbeside_kc<KC, double>(A, lds, s);
}

template <int KC, typename T>
void launch_mspec_kc(const MsampArgs& A, size_t lds, hipStream_t s) {
    const int seg = (A.M + kSpecBlock - 1) / kSpecBlock;
    const dim3 grid(1 + job_blocks(A, kSpecBlock), A.n_chains), block(kSpecBlock);
    if (seg <= 1) hipLaunchKernelGGL((mspec_kernel<1, KC, T>), grid, block, lds, s, A);
    else if (seg <= 2) hipLaunchKernelGGL((mspec_kernel<2, KC, T>), grid, block, lds, s, A);
    else if (seg <= 4) hipLaunchKernelGGL((mspec_kernel<4, KC, T>), grid, block, lds, s, A);
    else if (seg <= 8) hipLaunchKernelGGL((mspec_kernel<8, KC, T>), grid, block, lds, s, A);
    else hipLaunchKernelGGL((mspec_kernel<0, KC, T>), grid, block, lds, s, A);
}

template <int KC>
void launch_mspec_kc(const MsampArgs& A, size_t lds, hipStream_t s) {
    if (A.fp32) launch_mspec_kc<KC, float>(A, lds, s);
    else launch_mspec_kc<KC, double>(A, lds, s);
}

template <typename T>
void launch_mfb_t(const MsampArgs& A, hipStream_t s) {
    const int seg = (A.M + kFbBlock - 1) / kFbBlock;
    const dim3 grid(A.n_chains), block(kFbBlock);
    const size_t lds = A.fb_ubuf ? sizeof(double) * (size_t)A.M : 0;
    if (seg <= 1) hipLaunchKernelGGL((mfb_kernel<1, T>), grid, block, lds, s, A);
    else if (seg <= 2) hipLaunchKernelGGL((mfb_kernel<2, T>), grid, block, lds, s, A);
    else if (seg <= 4) hipLaunchKernelGGL((mfb_kernel<4, T>), grid, block, lds, s, A);
    else if (seg <= 8) hipLaunchKernelGGL((mfb_kernel<8, T>), grid, block, lds, s, A);
    else hipLaunchKernelGGL((mfb_kernel<0, T>), grid, block, lds, s, A);
}

}  // namespace

hipError_t configure_msampler_lds(size_t job_lds, size_t spec_lds, size_t beside_lds) {
    hipError_t e = set_lds_kc<0>(job_lds, spec_lds, beside_lds);
    if (e == hipSuccess) e = set_lds_kc<2>(job_lds, spec_lds, beside_lds);
    if (e == hipSuccess) e = set_lds_kc<3>(job_lds, spec_lds, beside_lds);
    if (e == hipSuccess) e = set_lds_kc<4>(job_lds, spec_lds, beside_lds);
    if (e == hipSuccess) e = set_lds_kc<6>(job_lds, spec_lds, beside_lds);
    if (e == hipSuccess) e = set_lds_kc<8>(job_lds, spec_lds, beside_lds);
    if (e == hipSuccess) e = set_lds_kc<12>(job_lds, spec_lds, beside_lds);
    if (e == hipSuccess) e = set_lds_kc<16>(job_lds, spec_lds, beside_lds);
    return e;
}

hipError_t launch_mclass(const MsampArgs& A, uint8_t* masks, uint8_t* cls, int32_t* joblist, int32_t* jobcnt,
                         hipStream_t s) {
    hipLaunchKernelGGL(mclass_kernel, dim3((A.M + kClassBlock - 1) / kClassBlock), dim3(kClassBlock), 0, s, A, masks,
                       cls);
    hipLaunchKernelGGL(mjobs_kernel, dim3(2 * (A.N - A.F)), dim3(64), 0, s, A.M, cls, joblist, jobcnt);
    return hipGetLastError();
}

hipError_t launch_morder(const MsampArgs& A, const int32_t* fixed_order, hipStream_t s) {
    hipLaunchKernelGGL(morder_kernel, dim3(A.n_chains), dim3(kOrderBlock), 0, s, A, fixed_order);
    return hipGetLastError();
}

hipError_t launch_mstep(const MsampArgs& A, size_t lds, hipStream_t s) {
    const dim3 grid(job_blocks(A, kMsampBlock), A.n_chains);
    if (grid.x == 0) return hipSuccess;  // no flip needs a graph
    switch (A.people_chunks) {
        case 2: hipLaunchKernelGGL(mstep_kernel<2>, grid, dim3(kMsampBlock), lds, s, A); break;
        case 3: hipLaunchKernelGGL(mstep_kernel<3>, grid, dim3(kMsampBlock), lds, s, A); break;
        case 4: hipLaunchKernelGGL(mstep_kernel<4>, grid, dim3(kMsampBlock), lds, s, A); break;
        case 6: hipLaunchKernelGGL(mstep_kernel<6>, grid, dim3(kMsampBlock), lds, s, A); break;
        case 8: hipLaunchKernelGGL(mstep_kernel<8>, grid, dim3(kMsampBlock), lds, s, A); break;
        case 12: hipLaunchKernelGGL(mstep_kernel<12>, grid, dim3(kMsampBlock), lds, s, A); break;
        case 16: hipLaunchKernelGGL(mstep_kernel<16>, grid, dim3(kMsampBlock), lds, s, A); break;
        default: hipLaunchKernelGGL(mstep_kernel<0>, grid, dim3(kMsampBlock), lds, s, A); break;
    }
    return hipGetLastError();
}

hipError_t launch_mplan(const MsampArgs& A, hipStream_t s) {
    hipLaunchKernelGGL(mplan_kernel, dim3(A.n_meioses), dim3(kPlanBlock), 0, s, A);
    return hipGetLastError();
}

hipError_t launch_mplanned(const MsampArgs& A, size_t lds, hipStream_t s) {
    const dim3 grid(planned_blocks(A, kMsampBlock)), block(kMsampBlock);
    if (grid.x == 0) return hipSuccess;
    switch (A.people_chunks) {
        case 2: hipLaunchKernelGGL(mplanned_kernel<2>, grid, block, lds, s, A); break;
        case 3: hipLaunchKernelGGL(mplanned_kernel<3>, grid, block, lds, s, A); break;
        case 4: hipLaunchKernelGGL(mplanned_kernel<4>, grid, block, lds, s, A); break;
        case 6: hipLaunchKernelGGL(mplanned_kernel<6>, grid, block, lds, s, A); break;
        case 8: hipLaunchKernelGGL(mplanned_kernel<8>, grid, block, lds, s, A); break;
        case 12: hipLaunchKernelGGL(mplanned_kernel<12>, grid, block, lds, s, A); break;
        case 16: hipLaunchKernelGGL(mplanned_kernel<16>, grid, block, lds, s, A); break;
        default: hipLaunchKernelGGL(mplanned_kernel<0>, grid, block, lds, s, A); break;
    }
    return hipGetLastError();
}

hipError_t launch_mbeside(const MsampArgs& A, size_t lds, hipStream_t s) {
    switch (A.people_chunks) {
        case 2: launch_mbeside_kc<2>(A, lds, s); break;
        case 3: launch_mbeside_kc<3>(A, lds, s); break;
        case 4: launch_mbeside_kc<4>(A, lds, s); break;
        case 6: launch_mbeside_kc<6>(A, lds, s); break;
        case 8: launch_mbeside_kc<8>(A, lds, s); break;
        case 12: launch_mbeside_kc<12>(A, lds, s); break;
        case 16: launch_mbeside_kc<16>(A, lds, s); break;
        default: launch_mbeside_kc<0>(A, lds, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_mfb(const MsampArgs& A, hipStream_t s) {
    if (A.fp32) launch_mfb_t<float>(A, s);
    else launch_mfb_t<double>(A, s);
    return hipGetLastError();
}

hipError_t launch_mspec(const MsampArgs& A, size_t lds, hipStream_t s) {
    switch (A.people_chunks) {
        case 2: launch_mspec_kc<2>(A, lds, s); break;
        case 3: launch_mspec_kc<3>(A, lds, s); break;
        case 4: launch_mspec_kc<4>(A, lds, s); break;
        case 6: launch_mspec_kc<6>(A, lds, s); break;
        case 8: launch_mspec_kc<8>(A, lds, s); break;
        case 12: launch_mspec_kc<12>(A, lds, s); break;
        case 16: launch_mspec_kc<16>(A, lds, s); break;
        default: launch_mspec_kc<0>(A, lds, s); break;
    }
    return hipGetLastError();
}

}  // namespace sl
