// FP64 trait peel and its adjoint for gfx950, one (graph, interval, position)
// evaluation per lane.
//
// A wavefront takes 64 evaluations and walks the peel program's ops in
// sequential order; the program is the same for every evaluation, so op and
// cell descriptors are wave-uniform (scalar loads), no lane idles on a small
// table and there is no barrier.  What differs per lane is the two graph
// columns (LDS) and the position's thetas.
//
// Most ops of a pedigree peel a child from its two parents' table, or a
// married-in founder from that (kL64Child, kL64Founder).  Their 16-cell tables
// are formed in registers and handed to the next op in registers when it
// consumes them, as it does along a sibship; three quarters of all cells at
// 150 to 600 people never reach memory.  The others live in a slot of global
// memory, cell c of the wave at 64 c + lane, reused as tables die.
//
// Forward arithmetic is the workgroup kernel's (lod.hip), operation for
// operation: per term the trait probability, the consumed tables in order,
// then the transmission factor; terms summed in order.  A skipped (zero) term
// there is an exact zero here.  So the two kernels' terms are equal bit for bit.
//
// Adjoint: the forward pass keeps every table (a tape), then the ops run in
// reverse.  A register op recomputes its transmission core, a generic one
// gathers every consumed cell's adjoint from the list of its contributions, so
// nothing is accumulated through memory.
//
// Bound: instruction issue (about 200 FP64 instructions per register op) and
// memory latency at two to three wavefronts per SIMD; the adjoint waits on memory
// for half its time (tape and generic cells).  Measured: 50 graphs x 9995
// positions at 200 people 1.9 ms (workgroup kernel 11.4 ms: idle lanes and a
// barrier per level); the adjoint over 32 of them 21.9 ms (165 ms: one workgroup
// per evaluation, LDS atomics).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstdint>

#include "kernels.h"
#include "lane64.h"

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

struct Lane {
    const uint32_t* col;  // this lane's column words in LDS: [2W][64] + lane
    int W, lane;
    double t1, a1, t2, a2;  // flanking thetas (set_thetas, trait_rfunction.h:50-56)
};

// The phased-trait code of non-founder r at (l, l+1): maternal bits 0-1, paternal 2-3
__device__ __forceinline__ uint32_t code_of(const Lane& L, int r) {
    const int w = r >> 4, sh = 2 * (r & 15);
    const uint32_t x0 = L.col[(size_t)w * kWave] >> sh, x1 = L.col[(size_t)(L.W + w) * kWave] >> sh;
    return (x0 & 1u) | ((x1 & 1u) << 1) | ((x0 & 2u) << 1) | ((x1 & 2u) << 2);
}

// q[t] = 0.25 rho(code, i = t >> 1, j = t & 1) in the workgroup kernel's order
__device__ __forceinline__ void transmission(const Lane& L, int r, double q[4]) {
    const uint32_t c = code_of(L, r);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const uint32_t i = (uint32_t)(t >> 1), j = (uint32_t)(t & 1);
        double x = (c & 1u) == i ? L.a1 : L.t1;
        x *= ((c >> 1) & 1u) == i ? L.a2 : L.t2;
        x *= ((c >> 2) & 1u) == j ? L.a1 : L.t1;
        x *= ((c >> 3) & 1u) == j ? L.a2 : L.t2;
        q[t] = 0.25 * x;
    }
}

// the derivatives of q with respect to theta_L and theta_R
__device__ __forceinline__ void transmission_grad(const Lane& L, int r, double ql[4], double qr[4]) {
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
template <int N>
__device__ __forceinline__ void load_map(const double* ar, cu32_p off, cu32_p map, int lane, double* x) {
    const double* base = ar + (size_t)off[0] * kWave;
#pragma unroll
    for (int v = 0; v < N; ++v) {
        const uint32_t c = map_byte(map, v);
        x[v] = 0.0;
        if (c != 0xFFu) x[v] = base[(size_t)c * kWave + lane];
    }
}

template <int N>
__device__ __forceinline__ void store_map(double* ar, uint32_t off, cu32_p map, int lane, const double* x) {
    double* base = ar + (size_t)off * kWave;
#pragma unroll
    for (int v = 0; v < N; ++v) {
        const uint32_t c = map_byte(map, v);
        if (c != 0xFFu) base[(size_t)c * kWave + lane] = x[v];
    }
}

struct Trait {
    double v[4];
    __device__ __forceinline__ explicit Trait(cu32_p h) {
        cf64_p t = (cf64_p)(h + kHTrait);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = t[k];
    }
};

// ---- forward ----

// A consumed table of a Child op: its values (class K: by the kid's trait,
// class M: by the parents'), from registers (cur) or the arena.
template <int C>
__device__ __forceinline__ void child_prev(const double* ar, cu32_p hp, int lane, const double cur[16], double* x) {
    constexpr int N = C == kL64K ? 4 : 16;
    if (C == kL64None) return;
    if (hp[kPClass] & 16u) {
#pragma unroll
        for (int v = 0; v < N; ++v) x[v] = cur[v];
    } else {
        load_map<N>(ar, hp + kPOff, hp + kPMap, lane, x);
    }
}

template <int C0, int C1>
__device__ __forceinline__ void child_forward(const Lane& L, const double* ar, cu32_p h, double cur[16]) {
    const Trait tr(h);
    double q[4];
    transmission(L, (int)h[kHPeel], q);
    double p0[C0 == kL64M ? 16 : 4], p1[C1 == kL64M ? 16 : 4];
    child_prev<C0>(ar, h + kHPrev, L.lane, cur, p0);
    child_prev<C1>(ar, h + kHPrev + 8, L.lane, cur, p1);
    double X[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        X[v] = tr.v[v];
        if (C0 == kL64K) X[v] *= p0[v];
        if (C0 == kL64K && C1 == kL64K) X[v] *= p1[v];
    }
#pragma unroll
    for (int mp = 0; mp < 16; ++mp) {
        double total = 0.0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int v = kid_value(mp >> 2, mp & 3, t);
            double x = X[v];
            if (C0 == kL64M) x *= p0[mp];
            if (C0 == kL64M && C1 == kL64K) x *= p1[v];
            if (C1 == kL64M) x *= p1[mp];
            x *= q[t];
            total = t == 0 ? x : total + x;
        }
        cur[mp] = total;
    }
}

__device__ __forceinline__ int child_pattern(cu32_p h) {
    const int np = (int)h[kHPrevs];
    const int c0 = np > 0 ? (int)(h[kHPrev + kPClass] & 15u) : 0;
    const int c1 = np > 1 ? (int)(h[kHPrev + 8 + kPClass] & 15u) : 0;
    return 3 * c0 + c1;
}

__device__ __forceinline__ void founder_forward(const Lane& L, const double* ar, cu32_p h, double cur[16]) {
    const Trait tr(h);
    cu32_p hp = h + kHPrev;
    if (!(hp[kPClass] & 16u)) load_map<16>(ar, hp + kPOff, hp + kPMap, L.lane, cur);
    double out[4];
    if (h[kHPeelIsPat]) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            out[s] = tr.v[0] * cur[4 * s];
#pragma unroll
            for (int v = 1; v < 4; ++v) out[s] += tr.v[v] * cur[4 * s + v];
        }
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            out[s] = tr.v[0] * cur[s];
#pragma unroll
            for (int v = 1; v < 4; ++v) out[s] += tr.v[v] * cur[4 * v + s];
        }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) cur[s] = out[s];
}

// sum of a child's transmission factors q over its allowed (i, j), in order
__device__ __forceinline__ double allowed_sum(const double q[4], uint32_t m) {
    double s = 0.0;
#pragma unroll
    for (int ij = 0; ij < 4; ++ij)
        if ((m >> ij) & 1u) s += q[ij];
    return s;
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
    template <int NP>
    __device__ __forceinline__ void values(const double* ar, int lane, double v[4][NP > 0 ? NP : 1]) const {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int k = 0; k < NP; ++k) v[t][k] = ar[(size_t)w[4 * t + 1 + k] * kWave + lane];
    }
};

template <int TYPE, int NP, int NC>
__device__ __forceinline__ void generic_forward(const Lane& L, double* ar, cu32_p h, cu32_p fwd) {
    const Trait tr(h);
    const int size = (int)h[kHSize];
    cu32_p rec = fwd + h[kHStream];
    double* out = ar + (size_t)h[kHOut] * kWave;
    double q[4], qk[NC > 0 ? NC : 1][4];
    if (TYPE == kChild) transmission(L, (int)h[kHPeel], q);
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) transmission(L, (int)h[kHKid + ch], qk[ch]);
    // the next cell's values are loaded while this one is summed, and the
    // records one cell further (a dependent scalar and vector load per cell
    // would each wait out the memory latency)
    CellRec nr;
    nr.load(rec);
    double nv[4][NP > 0 ? NP : 1];
    nr.values<NP>(ar, L.lane, nv);
    CellRec fr;
    fr.load(rec + (size > 1 ? 16 : 0));
    for (int c = 0; c < size; ++c) {
        const CellRec cr = nr;
        double pv[4][NP > 0 ? NP : 1];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int k = 0; k < NP; ++k) pv[t][k] = nv[t][k];
        nr = fr;
        nr.values<NP>(ar, L.lane, nv);
        fr.load(rec + 16 * (size_t)min(c + 2, size - 1));
        double total = 0.0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t info = cr.w[4 * t];
            if (!(info & 4u)) continue;  // uniform; its values are a consumed table's first cell
            const uint32_t v = TYPE == kChild ? info & 3u : (uint32_t)t;
            double x = v == 0u ? tr.v[0] : v == 1u ? tr.v[1] : v == 2u ? tr.v[2] : tr.v[3];
#pragma unroll
            for (int k = 0; k < NP; ++k) x *= pv[t][k];
            if (TYPE == kChild) x *= q[t];
            if (TYPE == kParent) {
                double s = 1.0;
#pragma unroll
                for (int ch = 0; ch < NC; ++ch) s *= allowed_sum(qk[ch], (info >> (4 + 4 * ch)) & 15u);
                x *= s;
            }
            total += x;
        }
        out[(size_t)c * kWave + L.lane] = total;
    }
}

template <int NP>
__device__ __forceinline__ void generic_forward_np(const Lane& L, double* ar, cu32_p h, cu32_p fwd) {
    const int type = (int)h[kHType];
    if (type == kChild) generic_forward<kChild, NP, 0>(L, ar, h, fwd);
    else if (type == kParent) {
        switch (h[kHKids]) {
            case 0: generic_forward<kParent, NP, 0>(L, ar, h, fwd); break;
            case 1: generic_forward<kParent, NP, 1>(L, ar, h, fwd); break;
            case 2: generic_forward<kParent, NP, 2>(L, ar, h, fwd); break;
            default: generic_forward<kParent, NP, 3>(L, ar, h, fwd); break;
        }
    } else generic_forward<kPartner, NP, 0>(L, ar, h, fwd);
}

// the whole program; returns the likelihood
__device__ __forceinline__ double peel_forward(const Lane64Args& A, const Lane& L, double* ar) {
    double cur[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) cur[v] = 0.0;
    for (int s = 0; s < A.n_ops; ++s) {
        cu32_p h = (cu32_p)(A.hdr + (size_t)s * kL64Header);
        const int kind = (int)h[kHKind];
        if (kind == kL64Child) {
            switch (child_pattern(h)) {
                case 0: child_forward<kL64None, kL64None>(L, ar, h, cur); break;
                case 3 * kL64K: child_forward<kL64K, kL64None>(L, ar, h, cur); break;
                case 3 * kL64M: child_forward<kL64M, kL64None>(L, ar, h, cur); break;
                case 3 * kL64K + kL64K: child_forward<kL64K, kL64K>(L, ar, h, cur); break;
                case 3 * kL64K + kL64M: child_forward<kL64K, kL64M>(L, ar, h, cur); break;
                case 3 * kL64M + kL64K: child_forward<kL64M, kL64K>(L, ar, h, cur); break;
                default: child_forward<kL64M, kL64M>(L, ar, h, cur); break;
            }
            if ((int)h[kHOut] >= 0) store_map<16>(ar, h[kHOut], h + kHMap, L.lane, cur);
        } else if (kind == kL64Founder) {
            founder_forward(L, ar, h, cur);
            if ((int)h[kHOut] >= 0) store_map<4>(ar, h[kHOut], h + kHMap, L.lane, cur);
        } else {
            cu32_p fwd = (cu32_p)A.fwd;
            switch (h[kHPrevs]) {
                case 0: generic_forward_np<0>(L, ar, h, fwd); break;
                case 1: generic_forward_np<1>(L, ar, h, fwd); break;
                case 2: generic_forward_np<2>(L, ar, h, fwd); break;
                default: generic_forward_np<3>(L, ar, h, fwd); break;
            }
        }
    }
    // the last op is a generic one of a single cell
    const int out = (int)((cu32_p)(A.hdr + (size_t)(A.n_ops - 1) * kL64Header))[kHOut];
    return ar[(size_t)out * kWave + L.lane];
}

// ---- reverse ----

// adds the derivatives of one op's trait probabilities (dv[v] = d ln L / d
// disease_prob[person][v]), through the model's Jacobian
__device__ __forceinline__ void add_model(const Lane64Args& A, cu32_p h, const double dv[4], double acc[6]) {
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
    constexpr int N = C == kL64K ? 4 : 16;
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
__device__ __forceinline__ void child_reverse(const Lane64Args& A, const Lane& L, const double* ar, double* adj, cu32_p h,
                                              double cur[16], double acc[6]) {
    const Trait tr(h);
    const int r = (int)h[kHPeel];
    double D[16];  // adjoint of the table, then times the M tables
    if ((int)h[kHAdj] < 0) {
#pragma unroll
        for (int v = 0; v < 16; ++v) D[v] = cur[v];
    } else {
        load_map<16>(adj, h + kHAdj, h + kHMap, L.lane, D);
    }
    double p0[C0 == kL64M ? 16 : 4], p1[C1 == kL64M ? 16 : 4];
    if (C0 != kL64None) load_map<(C0 == kL64K ? 4 : 16)>(ar, h + kHPrev + kPOff, h + kHPrev + kPMap, L.lane, p0);
    if (C1 != kL64None) load_map<(C1 == kL64K ? 4 : 16)>(ar, h + kHPrev + 8 + kPOff, h + kHPrev + 8 + kPMap, L.lane, p1);
    double X[4], q[4];
    transmission(L, r, q);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        X[v] = tr.v[v];
        if (C0 == kL64K) X[v] *= p0[v];
        if (C1 == kL64K) X[v] *= p1[v];
    }
    if (C0 == kL64M || C1 == kL64M) {
        // the table is core x M tables: their adjoints
        double g0[16], g1[C0 == kL64M && C1 == kL64M ? 16 : 1];
#pragma unroll
        for (int mp = 0; mp < 16; ++mp) {
            double core = X[kid_value(mp >> 2, mp & 3, 0)] * q[0];
#pragma unroll
            for (int t = 1; t < 4; ++t) core = fma(X[kid_value(mp >> 2, mp & 3, t)], q[t], core);
            const double a = D[mp] * core;
            if (C0 == kL64M && C1 == kL64M) {
                g0[mp] = a * p1[mp];
                g1[mp] = a * p0[mp];
                D[mp] *= p0[mp] * p1[mp];
            } else {
                g0[mp] = a;
                D[mp] *= C0 == kL64M ? p0[mp] : p1[mp];
            }
        }
        if (C0 == kL64M) pass_adjoint<kL64M>(adj, h + kHPrev, L.lane, g0, cur);
        if (C1 == kL64M) pass_adjoint<kL64M>(adj, h + kHPrev + 8, L.lane, C0 == kL64M ? g1 : g0, cur);
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
        const double a = C0 == kL64K ? p0[v] : 1.0, b = C1 == kL64K ? p1[v] : 1.0;
        dv[v] = H[v] * (a * b);
        k0[v] = H[v] * (tr.v[v] * b);
        k1[v] = H[v] * (tr.v[v] * a);
    }
    add_model(A, h, dv, acc);
    if (C0 == kL64K) pass_adjoint<kL64K>(adj, h + kHPrev, L.lane, k0, cur);
    if (C1 == kL64K) pass_adjoint<kL64K>(adj, h + kHPrev + 8, L.lane, k1, cur);
}

__device__ __forceinline__ void founder_reverse(const Lane64Args& A, const Lane& L, const double* ar, double* adj, cu32_p h,
                                                double cur[16], double acc[6]) {
    const Trait tr(h);
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
    pass_adjoint<kL64M>(adj, hp, L.lane, g, cur);
}

// A term's factor besides its consumed tables
template <int TYPE, int NC>
__device__ __forceinline__ double term_factor(const Trait& tr, const double q[4], const double (*qk)[4], uint32_t info,
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
__device__ __forceinline__ void term_share(const Trait& tr, const double q[4], const double (*qk)[4],
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
__device__ __forceinline__ void generic_reverse(const Lane64Args& A, const Lane& L, const double* ar, double* adj, cu32_p h,
                                                double acc[6]) {
    const Trait tr(h);
    double q[4], ql[4], qr[4], qk[NC > 0 ? NC : 1][4], lk[NC > 0 ? NC : 1][4], rk[NC > 0 ? NC : 1][4];
    if (TYPE == kChild) {
        transmission(L, (int)h[kHPeel], q);
        transmission_grad(L, (int)h[kHPeel], ql, qr);
    }
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) {
        transmission(L, (int)h[kHKid + ch], qk[ch]);
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
__device__ __forceinline__ void generic_reverse_np(const Lane64Args& A, const Lane& L, const double* ar, double* adj, cu32_p h,
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

__device__ __forceinline__ void peel_reverse(const Lane64Args& A, const Lane& L, const double* ar, double* adj, double like,
                             double acc[6]) {
    double cur[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) cur[v] = 0.0;
    {
        cu32_p h = (cu32_p)(A.hdr + (size_t)(A.n_ops - 1) * kL64Header);
        adj[(size_t)h[kHAdj] * kWave + L.lane] = like > 0.0 ? 1.0 / like : 0.0;
    }
    for (int s = A.n_ops - 1; s >= 0; --s) {
        cu32_p h = (cu32_p)(A.hdr + (size_t)s * kL64Header);
        const int kind = (int)h[kHKind];
        if (kind == kL64Child) {
            switch (child_pattern(h)) {
                case 0: child_reverse<kL64None, kL64None>(A, L, ar, adj, h, cur, acc); break;
                case 3 * kL64K: child_reverse<kL64K, kL64None>(A, L, ar, adj, h, cur, acc); break;
                case 3 * kL64M: child_reverse<kL64M, kL64None>(A, L, ar, adj, h, cur, acc); break;
                case 3 * kL64K + kL64K: child_reverse<kL64K, kL64K>(A, L, ar, adj, h, cur, acc); break;
                case 3 * kL64K + kL64M: child_reverse<kL64K, kL64M>(A, L, ar, adj, h, cur, acc); break;
                case 3 * kL64M + kL64K: child_reverse<kL64M, kL64K>(A, L, ar, adj, h, cur, acc); break;
                default: child_reverse<kL64M, kL64M>(A, L, ar, adj, h, cur, acc); break;
            }
        } else if (kind == kL64Founder) {
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

// Workgroups of one wavefront; each takes chunks of 64 evaluations in turn.
// Evaluation e: graph e mod G, then position, then interval, so a wavefront's
// lanes share an interval where they can.
template <bool GRAD>
__global__ void __launch_bounds__(kWave, 2) lane64_kernel(Lane64Args A) {
    extern __shared__ __align__(16) uint32_t cols[];
    if (!GRAD && A.gate_sweep && !gate_open(*A.gate_sweep, A.gate_burnin, A.gate_period)) return;
    const int lane = (int)threadIdx.x;
    double* ar = A.scratch + (size_t)blockIdx.x * (size_t)(A.arena_cells + A.adj_cells) * kWave;
    double* adj = ar + (size_t)A.arena_cells * kWave;
    const int64_t E = (int64_t)A.G * (A.M - 1) * A.npos;
    for (int64_t c0 = (int64_t)blockIdx.x * kWave; c0 < E; c0 += (int64_t)gridDim.x * kWave) {
        const int64_t e = c0 + lane < E ? c0 + lane : E - 1;
        const int g = (int)(e % A.G);
        const int lp = (int)(e / A.G);
        const int pos = lp % A.npos, l = lp / A.npos;
        const uint32_t* w0 = A.graphs + ((size_t)g * A.M + l) * A.W;
        int ncross = 0;
        for (int w = 0; w < A.W; ++w) {
            const uint32_t x0 = w0[w], x1 = w0[A.W + w];
            ncross += __popc(x0 ^ x1);
            cols[(size_t)w * kWave + lane] = x0;
            cols[(size_t)(A.W + w) * kWave + lane] = x1;
        }
        Lane L;
        L.col = cols + lane;
        L.W = A.W;
        L.lane = lane;
        const double ptheta = A.partial_theta[l];
        const double tl = ptheta * (double)(pos + 1), tr = ptheta * (double)(A.npos - pos);
        L.t1 = tl;
        L.a1 = 1.0 - tl;
        L.t2 = tr;
        L.a2 = 1.0 - tr;
        const double like = peel_forward(A, L, ar);
        const int nm = 2 * (A.N - A.F);
        const double R = (double)ncross * A.log_theta[l] + (double)(nm - ncross) * A.log_anti[l];
        const double lnl = like > 0.0 ? log(like) : -INFINITY;
        const size_t at = ((size_t)g * (A.M - 1) + l) * A.npos + pos;
        if (!GRAD) {
            const double term = lnl - R - A.trans;
            if (c0 + lane < E) {
                if (A.terms) A.terms[at] = term;
                if (A.partial) A.partial[at] = term;
            }
        } else {
            double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            peel_reverse(A, L, ar, adj, like, acc);
            if (c0 + lane < E) {
                double* o = A.out + at * 7;
                o[0] = lnl - (R + A.trans);
#pragma unroll
                for (int k = 0; k < 6; ++k) o[1 + k] = like > 0.0 ? acc[k] : 0.0;
            }
        }
    }
}

}  // namespace

int lane64_waves(int64_t E, size_t slot_bytes) {
    const int64_t chunks = (E + kWave - 1) / kWave;
    const int64_t cap = std::max<int64_t>(1, std::min<int64_t>(kL64Waves, (int64_t)(kL64ScratchBytes / slot_bytes)));
    const int64_t rounds = (chunks + cap - 1) / cap;
    return (int)((chunks + rounds - 1) / rounds);
}

hipError_t configure_lane64_lds(size_t lds) {
    if (lds <= 64 * 1024) return hipSuccess;
    hipError_t e = hipFuncSetAttribute((const void*)lane64_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void*)lane64_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    return e;
}

hipError_t launch_lane64(const Lane64Args& A, bool grad, int waves, size_t lds, hipStream_t s) {
    if (grad) hipLaunchKernelGGL(lane64_kernel<true>, dim3(waves), dim3(kWave), lds, s, A);
    else hipLaunchKernelGGL(lane64_kernel<false>, dim3(waves), dim3(kWave), lds, s, A);
    return hipGetLastError();
}

}  // namespace sl
