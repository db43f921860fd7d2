// Trait peel (FP64, FP32) and its FP64 adjoint for gfx950, one (graph, interval,
// position) evaluation per lane.
//
// A wavefront takes 64 evaluations and walks the peel program's ops in
// sequential order; the program is the same for every evaluation, so op and
// cell descriptors are wave-uniform (scalar loads), no lane idles on a small
// table and there is no barrier.  What differs per lane is the two graph
// columns (LDS) and the position's thetas.
//
// Most ops of a pedigree peel a child from its two parents' table, or a
// married-in founder from that (kLpChild, kLpFounder).  Their 16-cell tables
// are formed in registers and handed to the next op in registers when it
// consumes them, as it does along a sibship; three quarters of all cells at
// 150 to 600 people never reach memory.  The others live in a slot of global
// memory, cell c of the wave at 64 c + lane, reused as tables die.
//
// Forward arithmetic is that of the kernel a launch would otherwise run on
// (lod.hip), operation for operation.  Workgroup kernel: per term the trait
// probability, the consumed tables in order, then the transmission factor; terms
// summed in order; a term it skips is an exact zero here; FP32 takes the same
// power of two out of the likelihood (max_over_positions).  FP32 lane kernel: the
// transmission factor before the tables and the last product fused.  FP64 and
// workgroup-order FP32 terms are equal to that kernel's bit for bit; lane-order
// ones up to the rounding of ln L + E ln 2 where that kernel's unread padding
// cells delayed a rescale.
//
// Adjoint: the forward pass keeps every table (a tape), then the ops run in
// reverse.  A register op recomputes its transmission core, a generic one
// gathers every consumed cell's adjoint from the list of its contributions, so
// nothing is accumulated through memory.
//
// Bound: instruction issue (about 200 instructions per register op) and memory
// latency at two to four wavefronts per SIMD; the adjoint waits on memory for
// half its time (tape and generic cells).  Measured, us:
//   FP64, 50 graphs x 9995 positions, 200 people: 1936 (workgroup kernel 11500:
//   idle lanes, a barrier per level)
//   FP32, 64 x 4995, 150 people: 793 (lane kernel 1334: tables in LDS, four
//   wavefronts per CU; descriptors read as vectors)
//   FP32, 31 x 2495, 600 people: 2295 (workgroup kernel 12494)
//   adjoint, 32 x 9995, 200 people: 22000 (165000: a workgroup per evaluation,
//   LDS atomics)
#include <hip/hip_runtime.h>
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>

#include "kernels.h"
#include "lanepeel.h"

namespace sl {

namespace {

typedef const __attribute__((address_space(4))) uint32_t* cu32_p;
typedef const __attribute__((address_space(4))) double* cf64_p;

constexpr int kWave = 64;

// kid trait from the parents' phased traits (UU, AA, AU, UA) and the
// transmitted alleles (rfunction.cc:94-113, rfunction.h:81-107)
__host__ __device__ constexpr int kid_value(int mat, int pat, int t) {
    const unsigned aff = 0x9Cu, kt = 0x6Cu;
    const unsigned ma = (aff >> (2 * mat + (t >> 1))) & 1u, pa = (aff >> (2 * pat + (t & 1))) & 1u;
    return (int)((kt >> (2 * ((ma << 1) | pa))) & 3u);
}

template <typename T>
struct Lane {
    const uint32_t* col;  // this lane's column words in LDS: [2W][64] + lane
    int W, lane;
    T t1, a1, t2, a2;  // flanking thetas (set_thetas, trait_rfunction.h:50-56)
    int E;             // FP32: log2 of the scale taken out of the tables so far
    float mx;          // FP32: the largest cell of the last op's table
};

// The phased-trait code of non-founder r at (l, l+1): maternal bits 0-1, paternal 2-3
template <typename T>
__device__ __forceinline__ uint32_t code_of(const Lane<T>& L, int r) {
    const int w = r >> 4, sh = 2 * (r & 15);
    const uint32_t x0 = L.col[(size_t)w * kWave] >> sh, x1 = L.col[(size_t)(L.W + w) * kWave] >> sh;
    return (x0 & 1u) | ((x1 & 1u) << 1) | ((x0 & 2u) << 1) | ((x1 & 2u) << 2);
}

// q[t] = 0.25 rho(code, i = t >> 1, j = t & 1) in the order of the kernel this
// form follows: the workgroup kernel's rho as one product, the FP32 lane
// kernel's as the product of its parents' halves (zentry)
template <typename T, bool HALVES>
__device__ __forceinline__ void transmission(const Lane<T>& L, int r, T q[4]) {
    const uint32_t c = code_of(L, r);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const uint32_t i = (uint32_t)(t >> 1), j = (uint32_t)(t & 1);
        const T f1 = (c & 1u) == i ? L.a1 : L.t1, f2 = ((c >> 1) & 1u) == i ? L.a2 : L.t2;
        const T g1 = ((c >> 2) & 1u) == j ? L.a1 : L.t1, g2 = ((c >> 3) & 1u) == j ? L.a2 : L.t2;
        if (HALVES) q[t] = ((T)0.25 * (f1 * f2)) * (g1 * g2);
        else q[t] = (T)0.25 * (((f1 * f2) * g1) * g2);
    }
}

// A child's transmission factors for the PARENT sums over its allowed (i, j):
// the four q in order (workgroup kernel), or the parents' halves, whose sums
// over the allowed alleles are multiplied (FP32 lane kernel)
template <typename T, bool HALVES>
struct KidFactors {
    T q[4], f[3], g[3];  // f, g: allele 0, allele 1, both
    __device__ __forceinline__ void load(const Lane<T>& L, int r) {
        if (!HALVES) {
            transmission<T, false>(L, r, q);
        } else {
            const uint32_t c = code_of(L, r);
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) {
                f[i] = (T)0.25 * (((c & 1u) == i ? L.a1 : L.t1) * (((c >> 1) & 1u) == i ? L.a2 : L.t2));
                g[i] = (((c >> 2) & 1u) == i ? L.a1 : L.t1) * (((c >> 3) & 1u) == i ? L.a2 : L.t2);
            }
            f[2] = f[0] + f[1];
            g[2] = g[0] + g[1];
        }
    }
    // m: bit 2i+j set when (i, j) gives the child its trait; the allowed pairs form a product set
    __device__ __forceinline__ T sum(uint32_t m) const {
        if (!HALVES) {
            T s = (T)0;
#pragma unroll
            for (int ij = 0; ij < 4; ++ij)
                if ((m >> ij) & 1u) s += q[ij];
            return s;
        }
        const bool i0 = (m & 3u) != 0u, i1 = (m & 12u) != 0u, j0 = (m & 5u) != 0u, j1 = (m & 10u) != 0u;
        const T a = i0 ? (i1 ? f[2] : f[0]) : i1 ? f[1] : (T)0;
        const T b = j0 ? (j1 ? g[2] : g[0]) : j1 ? g[1] : (T)0;
        return a * b;
    }
};

// The sum of a cell's four terms, each a product whose last factors are a[t],
// b[t].  Workgroup order: products rounded, summed in order.  FP32 lane kernel:
// its compiled contraction, in which term 1 is rounded and terms 0, 2, 3 are
// fused into the running sum.
template <typename T, bool FUSED>
__device__ __forceinline__ T cell_sum(const T a[4], const T b[4]) {
    if (FUSED) {
        T s = __builtin_fmaf(a[0], b[0], a[1] * b[1]);
        s = __builtin_fmaf(a[2], b[2], s);
        return __builtin_fmaf(a[3], b[3], s);
    }
    T s = a[0] * b[0];
#pragma unroll
    for (int t = 1; t < 4; ++t) s += a[t] * b[t];
    return s;
}

// the derivatives of q with respect to theta_L and theta_R
__device__ __forceinline__ void transmission_grad(const Lane<double>& L, int r, double ql[4], double qr[4]) {
    const uint32_t c = code_of(L, r);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const uint32_t i = (uint32_t)(t >> 1), j = (uint32_t)(t & 1);
        const bool e1 = (c & 1u) == i, e2 = ((c >> 1) & 1u) == i, e3 = ((c >> 2) & 1u) == j, e4 = ((c >> 3) & 1u) == j;
        const double f1 = e1 ? L.a1 : L.t1, f2 = e2 ? L.a2 : L.t2, f3 = e3 ? L.a1 : L.t1, f4 = e4 ? L.a2 : L.t2;
        const double s1 = e1 ? -0.25 : 0.25, s2 = e2 ? -0.25 : 0.25, s3 = e3 ? -0.25 : 0.25, s4 = e4 ? -0.25 : 0.25;
        ql[t] = (f2 * f4) * (s1 * f3 + f1 * s3);
        qr[t] = (f1 * f3) * (s2 * f4 + f2 * s4);
    }
}

// byte v of a 16-byte map of header words
__device__ __forceinline__ uint32_t map_byte(cu32_p m, int v) { return (m[v >> 2] >> (8 * (v & 3))) & 0xFFu; }

// cells of a stored table by a byte map; 0 where illegal (its terms' trait
// probability is zero)
template <int N, typename T>
__device__ __forceinline__ void load_map(const T* ar, cu32_p off, cu32_p map, int lane, T* x) {
    const T* base = ar + (size_t)off[0] * kWave;
#pragma unroll
    for (int v = 0; v < N; ++v) {
        const uint32_t c = map_byte(map, v);
        x[v] = (T)0;
        if (c != 0xFFu) x[v] = base[(size_t)c * kWave + lane];
    }
}

template <int N, typename T>
__device__ __forceinline__ void store_map(T* ar, uint32_t off, cu32_p map, int lane, const T* x) {
    T* base = ar + (size_t)off * kWave;
#pragma unroll
    for (int v = 0; v < N; ++v) {
        const uint32_t c = map_byte(map, v);
        if (c != 0xFFu) base[(size_t)c * kWave + lane] = x[v];
    }
}

template <typename T>
struct Trait {
    T v[4];
    __device__ __forceinline__ explicit Trait(cu32_p h) {
        cf64_p t = (cf64_p)(h + kHTrait);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = (T)t[k];
    }
};

// FP32: a table whose largest cell leaves [2^-6, 2^6) is multiplied by a power
// of two (exact) per lane, the exponent kept for the likelihood
constexpr int kRenormLo = -6, kRenormHi = 6;
__device__ __forceinline__ int renorm_exponent(float mx) {
    const int e = mx > 0.0f ? __builtin_amdgcn_frexp_expf(mx) - 1 : 0;
    return e >= kRenormLo && e < kRenormHi ? 0 : e;
}
template <int N>
__device__ __forceinline__ void renorm(Lane<float>& L, float x[16]) {
    float mx = x[0];
#pragma unroll
    for (int v = 1; v < N; ++v) mx = fmaxf(mx, x[v]);
    const int e = renorm_exponent(mx);
    L.mx = mx;
    if (__ballot(e != 0)) {
#pragma unroll
        for (int v = 0; v < N; ++v) x[v] = __builtin_amdgcn_ldexpf(x[v], -e);
        L.E += e;
        L.mx = __builtin_amdgcn_ldexpf(mx, -e);
    }
}
template <int N>
__device__ __forceinline__ void renorm(Lane<double>&, double*) {}

// ---- forward ----
//
// T, LANE: double or float in the workgroup kernel's order (LANE false), or
// float in the FP32 lane kernel's (LANE true).

// A consumed table of a Child op: its values (class K: by the kid's trait,
// class M: by the parents'), from registers (cur) or the arena.
template <int C, typename T>
__device__ __forceinline__ void child_prev(const T* ar, cu32_p hp, int lane, const T cur[16], T* x) {
    constexpr int N = C == kLpK ? 4 : 16;
    if (C == kLpNone) return;
    if (hp[kPClass] & 16u) {
#pragma unroll
        for (int v = 0; v < N; ++v) x[v] = cur[v];
    } else {
        load_map<N>(ar, hp + kPOff, hp + kPMap, lane, x);
    }
}

template <typename T, bool LANE, int C0, int C1>
__device__ __forceinline__ void child_forward(Lane<T>& L, const T* ar, cu32_p h, T cur[16]) {
    const Trait<T> tr(h);
    T q[4];
    transmission<T, LANE>(L, (int)h[kHPeel], q);
    T p0[C0 == kLpM ? 16 : 4], p1[C1 == kLpM ? 16 : 4];
    child_prev<C0>(ar, h + kHPrev, L.lane, cur, p0);
    child_prev<C1>(ar, h + kHPrev + 8, L.lane, cur, p1);
    const uint32_t legal = h[kHMask];
    T X[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        X[v] = tr.v[v];
        if (!LANE && C0 == kLpK) X[v] *= p0[v];
        if (!LANE && C0 == kLpK && C1 == kLpK) X[v] *= p1[v];
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        // rows of an illegal maternal trait are skipped (uniform), cells of an
        // illegal paternal one zeroed
        T row[4] = {(T)0, (T)0, (T)0, (T)0};
        if ((legal >> m) & 1u) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const int mp = 4 * m + p;
                T a[4], b[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int v = kid_value(m, p, t);
                    if (LANE) {
                        a[t] = tr.v[v];
                        b[t] = q[t];
                        if (C0 != kLpNone) {
                            a[t] *= b[t];
                            b[t] = C0 == kLpK ? p0[v] : p0[mp];
                        }
                        if (C1 != kLpNone) {
                            a[t] *= b[t];
                            b[t] = C1 == kLpK ? p1[v] : p1[mp];
                        }
                    } else {
                        a[t] = X[v];
                        if (C0 == kLpM) a[t] *= p0[mp];
                        if (C0 == kLpM && C1 == kLpK) a[t] *= p1[v];
                        if (C1 == kLpM) a[t] *= p1[mp];
                        b[t] = q[t];
                    }
                }
                const T total = cell_sum<T, LANE>(a, b);
                row[p] = (legal >> (4 + p)) & 1u ? total : (T)0;
            }
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) cur[4 * m + p] = row[p];
    }
    renorm<16>(L, cur);
}

__device__ __forceinline__ int child_pattern(cu32_p h) {
    const int np = (int)h[kHPrevs];
    const int c0 = np > 0 ? (int)(h[kHPrev + kPClass] & 15u) : 0;
    const int c1 = np > 1 ? (int)(h[kHPrev + 8 + kPClass] & 15u) : 0;
    return 3 * c0 + c1;
}

template <typename T, bool LANE>
__device__ __forceinline__ void founder_forward(Lane<T>& L, const T* ar, cu32_p h, T cur[16]) {
    const Trait<T> tr(h);
    cu32_p hp = h + kHPrev;
    if (!(hp[kPClass] & 16u)) load_map<16>(ar, hp + kPOff, hp + kPMap, L.lane, cur);
    const uint32_t legal = h[kHMask];
    T out[4], b[4];
    const bool pat = h[kHPeelIsPat] != 0u;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (pat) {
#pragma unroll
            for (int v = 0; v < 4; ++v) b[v] = cur[4 * s + v];
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) b[v] = cur[4 * v + s];
        }
        const T total = cell_sum<T, LANE>(tr.v, b);
        out[s] = (legal >> s) & 1u ? total : (T)0;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) cur[s] = out[s];
    renorm<4>(L, cur);
}

// Four stream records of 4 words (a forward cell's terms, or four reverse
// contributions), in scalar registers.
struct CellRec {
    uint32_t w[16];
    __device__ __forceinline__ void load(cu32_p r) {
#pragma unroll
        for (int k = 0; k < 16; ++k) w[k] = r[k];
    }
    // the consumed cells of each term
    template <int NP, typename T>
    __device__ __forceinline__ void values(const T* ar, int lane, T v[4][NP > 0 ? NP : 1]) const {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int k = 0; k < NP; ++k) v[t][k] = ar[(size_t)w[4 * t + 1 + k] * kWave + lane];
    }
};

template <typename T, bool LANE, int TYPE, int NP, int NC>
__device__ __forceinline__ void generic_forward(Lane<T>& L, T* ar, cu32_p h, cu32_p fwd) {
    const Trait<T> tr(h);
    const int size = (int)h[kHSize];
    cu32_p rec = fwd + h[kHStream];
    T* out = ar + (size_t)h[kHOut] * kWave;
    T q[4];
    KidFactors<T, LANE> kid[NC > 0 ? NC : 1];
    if (TYPE == kChild) transmission<T, LANE>(L, (int)h[kHPeel], q);
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) kid[ch].load(L, (int)h[kHKid + ch]);
    // the next cell's values are loaded while this one is summed, and the
    // records one cell further (a dependent scalar and vector load per cell
    // would each wait out the memory latency)
    CellRec nr;
    nr.load(rec);
    T nv[4][NP > 0 ? NP : 1];
    nr.values<NP>(ar, L.lane, nv);
    CellRec fr;
    fr.load(rec + (size > 1 ? 16 : 0));
    float mx = 0.0f;
    for (int c = 0; c < size; ++c) {
        const CellRec cr = nr;
        T pv[4][NP > 0 ? NP : 1];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int k = 0; k < NP; ++k) pv[t][k] = nv[t][k];
        nr = fr;
        nr.values<NP>(ar, L.lane, nv);
        fr.load(rec + 16 * (size_t)min(c + 2, size - 1));
        T a[4], b[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            // a pruned term (uniform) is an exact zero; its values are a
            // consumed table's first cell
            const uint32_t info = cr.w[4 * t];
            const bool valid = (info & 4u) != 0u;
            const uint32_t v = TYPE == kChild ? info & 3u : (uint32_t)t;
            a[t] = v == 0u ? tr.v[0] : v == 1u ? tr.v[1] : v == 2u ? tr.v[2] : tr.v[3];
            b[t] = (T)1;
            if (LANE && TYPE == kChild) b[t] = q[t];
#pragma unroll
            for (int k = 0; k < NP; ++k) {
                a[t] *= b[t];
                b[t] = pv[t][k];
            }
            if (!LANE && TYPE == kChild) {
                a[t] *= b[t];
                b[t] = q[t];
            }
            if (TYPE == kParent) {
                if (LANE) {
#pragma unroll
                    for (int ch = 0; ch < NC; ++ch) {
                        a[t] *= b[t];
                        b[t] = kid[ch].sum((info >> (4 + 4 * ch)) & 15u);
                    }
                } else {
                    T s = (T)1;
#pragma unroll
                    for (int ch = 0; ch < NC; ++ch) s *= kid[ch].sum((info >> (4 + 4 * ch)) & 15u);
                    a[t] *= b[t];
                    b[t] = s;
                }
            }
            a[t] = valid ? a[t] : (T)0;
        }
        const T total = cell_sum<T, LANE>(a, b);
        out[(size_t)c * kWave + L.lane] = total;
        if (sizeof(T) == 4) mx = fmaxf(mx, (float)total);
    }
    if constexpr (sizeof(T) == 4) {
        const int e = renorm_exponent(mx);
        L.mx = __builtin_amdgcn_ldexpf(mx, -e);
        if (__ballot(e != 0)) {
            for (int c = 0; c < size; ++c) {
                T* x = out + (size_t)c * kWave + L.lane;
                *x = __builtin_amdgcn_ldexpf(*x, -e);
            }
            L.E += e;
        }
    }
}

template <typename T, bool LANE, int NP>
__device__ __forceinline__ void generic_forward_np(Lane<T>& L, T* ar, cu32_p h, cu32_p fwd) {
    const int type = (int)h[kHType];
    if (type == kChild) generic_forward<T, LANE, kChild, NP, 0>(L, ar, h, fwd);
    else if (type == kParent) {
        switch (h[kHKids]) {
            case 0: generic_forward<T, LANE, kParent, NP, 0>(L, ar, h, fwd); break;
            case 1: generic_forward<T, LANE, kParent, NP, 1>(L, ar, h, fwd); break;
            case 2: generic_forward<T, LANE, kParent, NP, 2>(L, ar, h, fwd); break;
            default: generic_forward<T, LANE, kParent, NP, 3>(L, ar, h, fwd); break;
        }
    } else generic_forward<T, LANE, kPartner, NP, 0>(L, ar, h, fwd);
}

// The workgroup kernel's FP32 tables share one exponent over an interval's
// positions, which makes a subtree's accumulated exponent that of its top
// table's largest true cell over those positions.  What it divides out of the
// likelihood is the sum of these over the tables the last op consumes; taking
// the same (exact) power of two keeps ln L + E ln 2 the same bit for bit.  x:
// this lane's exponent of such a table (its positions are the npos lanes from
// its group's first).
__device__ __forceinline__ int max_over_positions(int x, int npos, int lane) {
    const int first = lane - lane % npos;
    int m = x;
    for (int j = 0; j < npos; ++j) m = max(m, __shfl(x, first + j));
    return m;
}

// the whole program; returns the likelihood.  shared (FP32, workgroup order):
// the exponent the workgroup kernel divides out
template <typename T, bool LANE>
__device__ __forceinline__ T peel_forward(const LanePeelArgs& A, Lane<T>& L, T* ar, int* shared) {
    int before = 0;  // L.E where the current subtree of the last op began (its subtrees are contiguous)
    T cur[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) cur[v] = (T)0;
    for (int s = 0; s < A.n_ops; ++s) {
        cu32_p h = (cu32_p)(A.hdr + (size_t)s * kLpHeader);
        const int kind = (int)h[kHKind];
        if (kind == kLpChild) {
            switch (child_pattern(h)) {
                case 0: child_forward<T, LANE, kLpNone, kLpNone>(L, ar, h, cur); break;
                case 3 * kLpK: child_forward<T, LANE, kLpK, kLpNone>(L, ar, h, cur); break;
                case 3 * kLpM: child_forward<T, LANE, kLpM, kLpNone>(L, ar, h, cur); break;
                case 3 * kLpK + kLpK: child_forward<T, LANE, kLpK, kLpK>(L, ar, h, cur); break;
                case 3 * kLpK + kLpM: child_forward<T, LANE, kLpK, kLpM>(L, ar, h, cur); break;
                case 3 * kLpM + kLpK: child_forward<T, LANE, kLpM, kLpK>(L, ar, h, cur); break;
                default: child_forward<T, LANE, kLpM, kLpM>(L, ar, h, cur); break;
            }
            if ((int)h[kHOut] >= 0) store_map<16>(ar, h[kHOut], h + kHMap, L.lane, cur);
        } else if (kind == kLpFounder) {
            founder_forward<T, LANE>(L, ar, h, cur);
            if ((int)h[kHOut] >= 0) store_map<4>(ar, h[kHOut], h + kHMap, L.lane, cur);
        } else {
            cu32_p fwd = (cu32_p)A.fwd;
            switch (h[kHPrevs]) {
                case 0: generic_forward_np<T, LANE, 0>(L, ar, h, fwd); break;
                case 1: generic_forward_np<T, LANE, 1>(L, ar, h, fwd); break;
                case 2: generic_forward_np<T, LANE, 2>(L, ar, h, fwd); break;
                default: generic_forward_np<T, LANE, 3>(L, ar, h, fwd); break;
            }
        }
        if (sizeof(T) == 4 && !LANE && h[kHIntoLast]) {
            const int x = L.mx > 0.0f ? __builtin_amdgcn_frexp_expf(L.mx) + L.E - before : INT_MIN / 2;
            const int m = max_over_positions(x, A.npos, L.lane);
            *shared += m > INT_MIN / 2 ? m : 0;
            before = L.E;
        }
    }
    // the last op is a generic one of a single cell
    const int out = (int)((cu32_p)(A.hdr + (size_t)(A.n_ops - 1) * kLpHeader))[kHOut];
    return ar[(size_t)out * kWave + L.lane];
}

// ---- reverse ----

// adds the derivatives of one op's trait probabilities (dv[v] = d ln L / d
// disease_prob[person][v]), through the model's Jacobian
__device__ __forceinline__ void add_model(const LanePeelArgs& A, cu32_p h, const double dv[4], double acc[6]) {
    cf64_p J = (cf64_p)(A.jac + (size_t)16 * h[kHPerson]);
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[k] = fma(dv[v], J[4 * v + k], acc[k]);
}

// The adjoint of a table that goes on in registers (the next reverse op's
// table) or to the adjoint arena.
template <int C>
__device__ __forceinline__ void pass_adjoint(double* adj, cu32_p hp, int lane, const double* x, double cur[16]) {
    constexpr int N = C == kLpK ? 4 : 16;
    if ((int)hp[kPAdj] < 0) {
#pragma unroll
        for (int v = 0; v < N; ++v) cur[v] = x[v];
    } else {
        store_map<N>(adj, hp[kPAdj], hp + kPMap, lane, x);
    }
}

// cur: on entry the adjoint of the op's table when it came in registers; on
// exit that of the consumed table that goes on in registers
template <int C0, int C1>
__device__ __forceinline__ void child_reverse(const LanePeelArgs& A, const Lane<double>& L, const double* ar, double* adj, cu32_p h,
                                              double cur[16], double acc[6]) {
    const Trait<double> tr(h);
    const int r = (int)h[kHPeel];
    double D[16];  // adjoint of the table, then times the M tables
    if ((int)h[kHAdj] < 0) {
#pragma unroll
        for (int v = 0; v < 16; ++v) D[v] = cur[v];
    } else {
        load_map<16>(adj, h + kHAdj, h + kHMap, L.lane, D);
    }
    double p0[C0 == kLpM ? 16 : 4], p1[C1 == kLpM ? 16 : 4];
    if (C0 != kLpNone) load_map<(C0 == kLpK ? 4 : 16)>(ar, h + kHPrev + kPOff, h + kHPrev + kPMap, L.lane, p0);
    if (C1 != kLpNone) load_map<(C1 == kLpK ? 4 : 16)>(ar, h + kHPrev + 8 + kPOff, h + kHPrev + 8 + kPMap, L.lane, p1);
    double X[4], q[4];
    transmission<double, false>(L, r, q);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        X[v] = tr.v[v];
        if (C0 == kLpK) X[v] *= p0[v];
        if (C1 == kLpK) X[v] *= p1[v];
    }
    if (C0 == kLpM || C1 == kLpM) {
        // the table is core x M tables: their adjoints
        double g0[16], g1[C0 == kLpM && C1 == kLpM ? 16 : 1];
#pragma unroll
        for (int mp = 0; mp < 16; ++mp) {
            double core = X[kid_value(mp >> 2, mp & 3, 0)] * q[0];
#pragma unroll
            for (int t = 1; t < 4; ++t) core = fma(X[kid_value(mp >> 2, mp & 3, t)], q[t], core);
            const double a = D[mp] * core;
            if (C0 == kLpM && C1 == kLpM) {
                g0[mp] = a * p1[mp];
                g1[mp] = a * p0[mp];
                D[mp] *= p0[mp] * p1[mp];
            } else {
                g0[mp] = a;
                D[mp] *= C0 == kLpM ? p0[mp] : p1[mp];
            }
        }
        if (C0 == kLpM) pass_adjoint<kLpM>(adj, h + kHPrev, L.lane, g0, cur);
        if (C1 == kLpM) pass_adjoint<kLpM>(adj, h + kHPrev + 8, L.lane, C0 == kLpM ? g1 : g0, cur);
    }
    // d / d X[v] and, per transmitted pair, d / d q[t]
    double H[4] = {0.0, 0.0, 0.0, 0.0}, G[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int mp = 0; mp < 16; ++mp)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int v = kid_value(mp >> 2, mp & 3, t);
            H[v] = fma(D[mp], q[t], H[v]);
            G[t] = fma(D[mp], X[v], G[t]);
        }
    double ql[4], qr[4];
    transmission_grad(L, r, ql, qr);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        acc[4] = fma(G[t], ql[t], acc[4]);
        acc[5] = fma(G[t], qr[t], acc[5]);
    }
    double dv[4], k0[4], k1[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const double a = C0 == kLpK ? p0[v] : 1.0, b = C1 == kLpK ? p1[v] : 1.0;
        dv[v] = H[v] * (a * b);
        k0[v] = H[v] * (tr.v[v] * b);
        k1[v] = H[v] * (tr.v[v] * a);
    }
    add_model(A, h, dv, acc);
    if (C0 == kLpK) pass_adjoint<kLpK>(adj, h + kHPrev, L.lane, k0, cur);
    if (C1 == kLpK) pass_adjoint<kLpK>(adj, h + kHPrev + 8, L.lane, k1, cur);
}

__device__ __forceinline__ void founder_reverse(const LanePeelArgs& A, const Lane<double>& L, const double* ar, double* adj, cu32_p h,
                                                double cur[16], double acc[6]) {
    const Trait<double> tr(h);
    cu32_p hp = h + kHPrev;
    double a[4], P[16], g[16], dv[4];
    if ((int)h[kHAdj] < 0) {
#pragma unroll
        for (int v = 0; v < 4; ++v) a[v] = cur[v];
    } else {
        load_map<4>(adj, h + kHAdj, h + kHMap, L.lane, a);
    }
    load_map<16>(ar, hp + kPOff, hp + kPMap, L.lane, P);
    const bool pat = h[kHPeelIsPat] != 0u;
#pragma unroll
    for (int v = 0; v < 4; ++v) dv[v] = 0.0;
    if (pat) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                g[4 * s + v] = a[s] * tr.v[v];
                dv[v] = fma(a[s], P[4 * s + v], dv[v]);
            }
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                g[4 * v + s] = a[s] * tr.v[v];
                dv[v] = fma(a[s], P[4 * v + s], dv[v]);
            }
    }
    add_model(A, h, dv, acc);
    pass_adjoint<kLpM>(adj, hp, L.lane, g, cur);
}

// sum of a child's transmission factors over its allowed (i, j)
__device__ __forceinline__ double allowed_sum(const double q[4], uint32_t m) {
    double s = 0.0;
#pragma unroll
    for (int ij = 0; ij < 4; ++ij)
        if ((m >> ij) & 1u) s += q[ij];
    return s;
}

// a term's factor besides its consumed tables
template <int TYPE, int NC>
__device__ __forceinline__ double term_factor(const Trait<double>& tr, const double q[4], const double (*qk)[4], uint32_t info,
                                              uint32_t t) {
    const uint32_t v = TYPE == kChild ? info & 3u : t;
    double f = v == 0u ? tr.v[0] : v == 1u ? tr.v[1] : v == 2u ? tr.v[2] : tr.v[3];
    if (TYPE == kChild) f *= t == 0u ? q[0] : t == 1u ? q[1] : t == 2u ? q[2] : q[3];
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) f *= allowed_sum(qk[ch], (info >> (4 + 4 * ch)) & 15u);
    return f;
}

// adds a term's derivatives, x being its adjoint times (some of) its consumed
// cells: dv[v] by the trait probability of value v, G[t] by the CHILD factor of
// pair t, acc[4..5] by the thetas (PARENT)
template <int TYPE, int NC>
__device__ __forceinline__ void term_share(const Trait<double>& tr, const double q[4], const double (*qk)[4],
                                           const double (*lk)[4], const double (*rk)[4], uint32_t info, uint32_t t,
                                           double x, double dv[4], double G[4], double acc[6]) {
    const uint32_t v = TYPE == kChild ? info & 3u : t;
    double y = x;
    if (TYPE == kChild) {
        const double z = x * (v == 0u ? tr.v[0] : v == 1u ? tr.v[1] : v == 2u ? tr.v[2] : tr.v[3]);
        if (t == 0u) G[0] += z;
        else if (t == 1u) G[1] += z;
        else if (t == 2u) G[2] += z;
        else G[3] += z;
        y *= t == 0u ? q[0] : t == 1u ? q[1] : t == 2u ? q[2] : q[3];
    }
    if (TYPE == kParent) {
        double S = 1.0, SL = 0.0, SR = 0.0;
#pragma unroll
        for (int ch = 0; ch < NC; ++ch) {
            const uint32_t m = (info >> (4 + 4 * ch)) & 15u;
            const double s = allowed_sum(qk[ch], m);
            SL = fma(SL, s, S * allowed_sum(lk[ch], m));
            SR = fma(SR, s, S * allowed_sum(rk[ch], m));
            S *= s;
        }
        const double z = x * (v == 0u ? tr.v[0] : v == 1u ? tr.v[1] : v == 2u ? tr.v[2] : tr.v[3]);
        acc[4] = fma(z, SL, acc[4]);
        acc[5] = fma(z, SR, acc[5]);
        y *= S;
    }
    if (v == 0u) dv[0] += y;
    else if (v == 1u) dv[1] += y;
    else if (v == 2u) dv[2] += y;
    else dv[3] += y;
}

// four contributions' adjoint cells times their other consumed cells
template <int NP>
__device__ __forceinline__ void rev_values(const CellRec& r, const double* adj, const double* ar, int lane, double x[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        x[e] = adj[(size_t)(r.w[4 * e] & ~kRevLast) * kWave + lane];
        if (NP > 1) x[e] *= ar[(size_t)r.w[4 * e + 2] * kWave + lane];
        if (NP > 2) x[e] *= ar[(size_t)r.w[4 * e + 3] * kWave + lane];
    }
}

template <int TYPE, int NP, int NC>
__device__ __forceinline__ void generic_reverse(const LanePeelArgs& A, const Lane<double>& L, const double* ar, double* adj, cu32_p h,
                                                double acc[6]) {
    const Trait<double> tr(h);
    double q[4], ql[4], qr[4], qk[NC > 0 ? NC : 1][4], lk[NC > 0 ? NC : 1][4], rk[NC > 0 ? NC : 1][4];
    if (TYPE == kChild) {
        transmission<double, false>(L, (int)h[kHPeel], q);
        transmission_grad(L, (int)h[kHPeel], ql, qr);
    }
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) {
        transmission<double, false>(L, (int)h[kHKid + ch], qk[ch]);
        transmission_grad(L, (int)h[kHKid + ch], lk[ch], rk[ch]);
    }
    const int size = (int)h[kHSize];
    double dv[4] = {0.0, 0.0, 0.0, 0.0}, G[4] = {0.0, 0.0, 0.0, 0.0};
    if (NP == 0) {
        // no consumed table: only the parameters' share of every term
        const double* own = adj + (size_t)h[kHAdj] * kWave;
        cu32_p rec = (cu32_p)A.fwd + h[kHStream];
        for (int c = 0; c < size; ++c, rec += 16) {
            const double a = own[(size_t)c * kWave + L.lane];
            CellRec cr;
            cr.load(rec);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                term_share<TYPE, NC>(tr, q, qk, lk, rk, cr.w[4 * t], (uint32_t)t, a, dv, G, acc);
        }
    }
    // each consumed cell's adjoint, gathered from the contributions that read
    // it, four at a time: the next four's values and the records after them
    // are loaded meanwhile.  The first table's pass also sums the parameters'
    // share of its terms, which that table's cell multiplies.
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        cu32_p hp = h + kHPrev + 8 * k;
        double* out = adj + (size_t)hp[kPAdj] * kWave + L.lane;
        const double* val = ar + (size_t)hp[kPOff] * kWave + L.lane;
        cu32_p rv = (cu32_p)A.rev + h[kHRev + k];
        const int groups = (int)h[kHGroups + k];
        CellRec nr, fr;
        nr.load(rv);
        fr.load(rv + (groups > 1 ? 16 : 0));
        double nx[4];
        rev_values<NP>(nr, adj, ar, L.lane, nx);
        double sum = 0.0, pd[4] = {0.0, 0.0, 0.0, 0.0}, pg[4] = {0.0, 0.0, 0.0, 0.0}, pa[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (int b = 0; b < groups; ++b) {
            const CellRec cr = nr;
            double x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = nx[e];
            nr = fr;
            rev_values<NP>(nr, adj, ar, L.lane, nx);
            fr.load(rv + 16 * (size_t)min(b + 2, groups - 1));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t info = cr.w[4 * e + 1], t = info >> 30;
                if (info & 4u) {
                    sum = fma(x[e], term_factor<TYPE, NC>(tr, q, qk, info, t), sum);
                    if (k == 0) term_share<TYPE, NC>(tr, q, qk, lk, rk, info, t, x[e], pd, pg, pa);
                }
                if (cr.w[4 * e] & kRevLast) {
                    *out = sum;
                    out += kWave;
                    sum = 0.0;
                    if (k == 0) {
                        const double p = *val;
                        val += kWave;
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            dv[v] = fma(pd[v], p, dv[v]);
                            G[v] = fma(pg[v], p, G[v]);
                            pd[v] = pg[v] = 0.0;
                        }
                        acc[4] = fma(pa[4], p, acc[4]);
                        acc[5] = fma(pa[5], p, acc[5]);
                        pa[4] = pa[5] = 0.0;
                    }
                }
            }
        }
    }
    if (TYPE == kChild) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            acc[4] = fma(G[t], ql[t], acc[4]);
            acc[5] = fma(G[t], qr[t], acc[5]);
        }
    }
    add_model(A, h, dv, acc);
}

template <int NP>
__device__ __forceinline__ void generic_reverse_np(const LanePeelArgs& A, const Lane<double>& L, const double* ar, double* adj, cu32_p h,
                                   double acc[6]) {
    const int type = (int)h[kHType];
    if (type == kChild) generic_reverse<kChild, NP, 0>(A, L, ar, adj, h, acc);
    else if (type == kParent) {
        switch (h[kHKids]) {
            case 0: generic_reverse<kParent, NP, 0>(A, L, ar, adj, h, acc); break;
            case 1: generic_reverse<kParent, NP, 1>(A, L, ar, adj, h, acc); break;
            case 2: generic_reverse<kParent, NP, 2>(A, L, ar, adj, h, acc); break;
            default: generic_reverse<kParent, NP, 3>(A, L, ar, adj, h, acc); break;
        }
    } else generic_reverse<kPartner, NP, 0>(A, L, ar, adj, h, acc);
}

__device__ __forceinline__ void peel_reverse(const LanePeelArgs& A, const Lane<double>& L, const double* ar, double* adj, double like,
                             double acc[6]) {
    double cur[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) cur[v] = 0.0;
    {
        cu32_p h = (cu32_p)(A.hdr + (size_t)(A.n_ops - 1) * kLpHeader);
        adj[(size_t)h[kHAdj] * kWave + L.lane] = like > 0.0 ? 1.0 / like : 0.0;
    }
    for (int s = A.n_ops - 1; s >= 0; --s) {
        cu32_p h = (cu32_p)(A.hdr + (size_t)s * kLpHeader);
        const int kind = (int)h[kHKind];
        if (kind == kLpChild) {
            switch (child_pattern(h)) {
                case 0: child_reverse<kLpNone, kLpNone>(A, L, ar, adj, h, cur, acc); break;
                case 3 * kLpK: child_reverse<kLpK, kLpNone>(A, L, ar, adj, h, cur, acc); break;
                case 3 * kLpM: child_reverse<kLpM, kLpNone>(A, L, ar, adj, h, cur, acc); break;
                case 3 * kLpK + kLpK: child_reverse<kLpK, kLpK>(A, L, ar, adj, h, cur, acc); break;
                case 3 * kLpK + kLpM: child_reverse<kLpK, kLpM>(A, L, ar, adj, h, cur, acc); break;
                case 3 * kLpM + kLpK: child_reverse<kLpM, kLpK>(A, L, ar, adj, h, cur, acc); break;
                default: child_reverse<kLpM, kLpM>(A, L, ar, adj, h, cur, acc); break;
            }
        } else if (kind == kLpFounder) {
            founder_reverse(A, L, ar, adj, h, cur, acc);
        } else {
            switch (h[kHPrevs]) {
                case 0: generic_reverse_np<0>(A, L, ar, adj, h, acc); break;
                case 1: generic_reverse_np<1>(A, L, ar, adj, h, acc); break;
                case 2: generic_reverse_np<2>(A, L, ar, adj, h, acc); break;
                default: generic_reverse_np<3>(A, L, ar, adj, h, acc); break;
            }
        }
    }
}

// ln sum over the wavefront's lanes of e^v, in the FP32 lane kernel's order
__device__ __forceinline__ double wave_log_sum(double v) {
    double m = v;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
    double sum = (m == -INFINITY || v == -INFINITY) ? 0.0 : exp(v - m);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    return m == -INFINITY ? -INFINITY : m + log(sum);
}

// a wavefront per (accumulator, 64 graphs)
constexpr int kSumBlock = 256;
__global__ void __launch_bounds__(kSumBlock) chunk_sums_kernel(const double* terms, double* partial, int G, int n,
                                                               const uint32_t* gate_sweep, int gate_burnin,
                                                               int gate_period) {
    if (gate_sweep && !gate_open(*gate_sweep, gate_burnin, gate_period)) return;
    const int i = (int)blockIdx.x * (kSumBlock / kWave) + (int)(threadIdx.x / kWave), lane = (int)(threadIdx.x % kWave);
    if (i >= n) return;
    const int g = (int)blockIdx.y * kWave + lane;
    const double r = wave_log_sum(g < G ? terms[(size_t)g * n + i] : -INFINITY);
    if (lane == 0) partial[(size_t)blockIdx.y * n + i] = r;
}

// Workgroups of one wavefront; each takes chunks of evaluations in turn.  With
// A.chunked (LANE): 64 graphs of one interval and position, their terms
// log-summed over the wavefront into one partial, as the FP32 lane kernel's
// launches do.  FP32 in the workgroup kernel's order: the positions of as many
// (graph, interval) pairs as fit.  Otherwise 64 consecutive evaluations, evaluation e being graph e mod G, then
// position, then interval, each term a partial of its own.
template <typename T, bool LANE, bool GRAD>
__global__ void __launch_bounds__(kWave, 2) lanepeel_kernel(LanePeelArgs A) {
    extern __shared__ __align__(16) uint32_t cols[];
    if (!GRAD && A.gate_sweep && !gate_open(*A.gate_sweep, A.gate_burnin, A.gate_period)) return;
    const int lane = (int)threadIdx.x;
    T* ar = reinterpret_cast<T*>(A.scratch) + (size_t)blockIdx.x * (size_t)(A.arena_cells + A.adj_cells) * kWave;
    const int64_t nlp = (int64_t)(A.M - 1) * A.npos;
    const bool chunked = LANE && A.chunked;
    constexpr bool kGrouped = sizeof(T) == 4 && !LANE;
    const int pairs = kWave / A.npos;  // (graph, interval) pairs of a wavefront
    const int64_t E = chunked    ? nlp * ((A.G + kWave - 1) / kWave) * kWave
                      : kGrouped ? ((int64_t)A.G * (A.M - 1) + pairs - 1) / pairs * kWave
                                 : (int64_t)A.G * nlp;
    for (int64_t c0 = (int64_t)blockIdx.x * kWave; c0 < E; c0 += (int64_t)gridDim.x * kWave) {
        int g, l, pos, chunk = 0;
        bool live;
        if (chunked) {
            // chunks of graphs innermost
            const int nch = (A.G + kWave - 1) / kWave;
            const int64_t w = c0 / kWave;
            chunk = (int)(w % nch);
            const int lp = (int)(w / nch);
            pos = lp % A.npos;
            l = lp / A.npos;
            g = chunk * kWave + lane;
            live = g < A.G;
            g = live ? g : A.G - 1;
        } else if (kGrouped) {
            const int64_t gl = c0 / kWave * pairs + lane / A.npos;
            live = lane < pairs * A.npos && gl < (int64_t)A.G * (A.M - 1);
            const int64_t e = live ? gl : 0;
            g = (int)(e % A.G);
            l = (int)(e / A.G);
            pos = lane % A.npos;
        } else {
            live = c0 + lane < E;
            const int64_t e = live ? c0 + lane : E - 1;
            g = (int)(e % A.G);
            const int lp = (int)(e / A.G);
            pos = lp % A.npos;
            l = lp / A.npos;
        }
        const uint32_t* w0 = A.graphs + ((size_t)g * A.M + l) * A.W;
        int ncross = 0;
        for (int w = 0; w < A.W; ++w) {
            const uint32_t x0 = w0[w], x1 = w0[A.W + w];
            ncross += __popc(x0 ^ x1);
            cols[(size_t)w * kWave + lane] = x0;
            cols[(size_t)(A.W + w) * kWave + lane] = x1;
        }
        Lane<T> L;
        L.col = cols + lane;
        L.W = A.W;
        L.lane = lane;
        L.E = 0;
        const double ptheta = A.partial_theta[l];
        const double tl = ptheta * (double)(pos + 1), tr = ptheta * (double)(A.npos - pos);
        L.t1 = (T)tl;
        L.a1 = (T)(1.0 - tl);
        L.t2 = (T)tr;
        L.a2 = (T)(1.0 - tr);
        int shared = 0;
        double like = (double)peel_forward<T, LANE>(A, L, ar, &shared);
        if (kGrouped) {
            like = __builtin_ldexp(like, L.E - shared);
            L.E = shared;
        }
        const int nm = 2 * (A.N - A.F);
        const double R = (double)ncross * A.log_theta[l] + (double)(nm - ncross) * A.log_anti[l];
        const double lnl = like > 0.0 ? log(like) + (sizeof(T) == 4 ? (double)L.E * 0.69314718055994530942 : 0.0) : -INFINITY;
        const size_t at = ((size_t)g * (A.M - 1) + l) * A.npos + pos;
        if constexpr (GRAD) {
            double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            peel_reverse(A, L, ar, ar + (size_t)A.arena_cells * kWave, like, acc);
            if (live) {
                double* o = A.out + at * 7;
                o[0] = lnl - (R + A.trans);
#pragma unroll
                for (int k = 0; k < 6; ++k) o[1 + k] = like > 0.0 ? acc[k] : 0.0;
            }
        } else {
            const double term = lnl - R - A.trans;
            if (live && A.terms) A.terms[at] = term;
            if (!chunked) {
                if (live && A.partial) A.partial[at] = term;
                continue;
            }
            const double r = wave_log_sum(live ? term : -INFINITY);
            if (lane == 0 && A.partial) A.partial[((size_t)chunk * (A.M - 1) + l) * A.npos + pos] = r;
        }
    }
}

}  // namespace

int64_t lanepeel_lanes(LanePeelForm form, int G, int n_intervals, int npos) {
    const int64_t nlp = (int64_t)n_intervals * npos;
    if (form == kLpFloatLanes) return nlp * ((G + kWave - 1) / kWave) * kWave;
    if (form == kLpFloat) {
        const int pairs = kWave / npos;
        return ((int64_t)G * n_intervals + pairs - 1) / pairs * kWave;
    }
    return nlp * G;
}

hipError_t launch_chunk_sums(const double* terms, double* partial, int G, int n, const uint32_t* gate_sweep,
                             int gate_burnin, int gate_period, hipStream_t s) {
    constexpr int per = kSumBlock / kWave;
    hipLaunchKernelGGL(chunk_sums_kernel, dim3((n + per - 1) / per, (G + kWave - 1) / kWave), dim3(kSumBlock), 0, s, terms,
                       partial, G, n, gate_sweep, gate_burnin, gate_period);
    return hipGetLastError();
}

int lanepeel_waves(LanePeelForm form, int64_t E, size_t slot_bytes, size_t budget) {
    const int64_t chunks = (E + kWave - 1) / kWave;
    const int64_t cap = std::max<int64_t>(1, std::min<int64_t>(lanepeel_max_waves(form), (int64_t)(budget / slot_bytes)));
    const int64_t rounds = (chunks + cap - 1) / cap;
    return (int)((chunks + rounds - 1) / rounds);
}

hipError_t launch_lanepeel(const LanePeelArgs& A, LanePeelForm form, int waves, size_t lds, hipStream_t s) {
    const dim3 grid(waves), block(kWave);
    switch (form) {
        case kLpAdjoint: hipLaunchKernelGGL((lanepeel_kernel<double, false, true>), grid, block, lds, s, A); break;
        case kLpDouble: hipLaunchKernelGGL((lanepeel_kernel<double, false, false>), grid, block, lds, s, A); break;
        case kLpFloat: hipLaunchKernelGGL((lanepeel_kernel<float, false, false>), grid, block, lds, s, A); break;
        default: hipLaunchKernelGGL((lanepeel_kernel<float, true, false>), grid, block, lds, s, A); break;
    }
    return hipGetLastError();
}

}  // namespace sl
