// The FP64 trait peel and its adjoint with one evaluation per lane: argument
// block and launcher (lane64.hip); the program is PeelProgram::l64_* (program.h).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "program.h"

namespace sl {

struct Lane64Args {
    const uint32_t* hdr;         // kL64Header words per op, in sequential order
    const uint32_t* fwd;         // generic ops: 16 words per cell
    const uint32_t* rev;         // generic ops, adjoint: 4 words per (consumed cell, contribution)
    int n_ops, arena_cells, adj_cells;
    int N, F, M, W, npos, G;
    double trans;                // 2(N-F) ln 1/2
    const double* partial_theta; // [M-1]
    const double* log_theta;     // [M-1] ln theta
    const double* log_anti;      // [M-1] ln(1 - theta)
    const uint32_t* graphs;      // packed [G][M][W]
    double* scratch;             // gridDim.x slots of (arena_cells + adj_cells) x 64 doubles
    double* partial;             // LOD: [G][M-1][npos] terms ln L - R - T (each graph a chunk of its own)
    double* terms;               // LOD, optional: the same
    const double* jac;           // adjoint: [N][4][4] d disease_prob / d(penetrance 0..2, disease freq)
    double* out;                 // adjoint: [G][M-1][npos][7] ln L - R - T and 6 derivatives of ln L
    const uint32_t* gate_sweep;  // captured sweeps (LodArgs)
    int gate_burnin, gate_period;
};

// LDS of a wavefront: both columns of its lanes' graphs
inline size_t lane64_lds_bytes(int W) { return (size_t)2 * W * 64 * 4; }
inline size_t lane64_slot_bytes(int arena_cells, int adj_cells) {
    return (size_t)(arena_cells + adj_cells) * 64 * sizeof(double);
}
// wavefronts of a launch over E evaluations when each needs a slot of
// slot_bytes: enough for two per SIMD, as many as kL64ScratchBytes holds, and
// evened out over the rounds they take
constexpr int kL64Waves = 2048;
constexpr size_t kL64ScratchBytes = (size_t)4 << 30;
int lane64_waves(int64_t E, size_t slot_bytes);
hipError_t configure_lane64_lds(size_t lds);
hipError_t launch_lane64(const Lane64Args& A, bool grad, int waves, size_t lds, hipStream_t s);

}  // namespace sl
