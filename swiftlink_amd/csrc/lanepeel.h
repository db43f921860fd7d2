// The trait peel and its adjoint with one evaluation per lane: argument block and
// launchers (lanepeel.hip); the program is PeelProgram::lp_* (program.h).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "program.h"

namespace sl {

struct LanePeelArgs {
    const uint32_t* hdr;         // kLpHeader words per op, in sequential order
    const uint32_t* fwd;         // generic ops: 16 words per cell
    const uint32_t* rev;         // generic ops, adjoint: 4 words per (consumed cell, contribution)
    int n_ops, arena_cells, adj_cells;
    int N, F, M, W, npos, G;
    double trans;                // 2(N-F) ln 1/2
    const double* partial_theta; // [M-1]
    const double* log_theta;     // [M-1] ln theta
    const double* log_anti;      // [M-1] ln(1 - theta)
    const uint32_t* graphs;      // packed [G][M][W]
    void* scratch;               // gridDim.x slots of (arena_cells + adj_cells) x 64 table cells
    double* partial;             // LOD: [chunks][M-1][npos]: a chunk is a graph, or 64 (kLpFloatLanes)
    int chunked;                 // 1: kLpFloatLanes
    double* terms;               // LOD, optional: the same
    const double* jac;           // adjoint: [N][4][4] d disease_prob / d(penetrance 0..2, disease freq)
    double* out;                 // adjoint: [G][M-1][npos][7] ln L - R - T and 6 derivatives of ln L
    const uint32_t* gate_sweep;  // captured sweeps (LodArgs)
    int gate_burnin, gate_period;
};

// LDS of a wavefront: both columns of its lanes' graphs
inline size_t lanepeel_lds_bytes(int W) { return (size_t)2 * W * 64 * 4; }
inline size_t lanepeel_slot_bytes(int arena_cells, int adj_cells, bool fp64) {
    return (size_t)(arena_cells + adj_cells) * 64 * (fp64 ? 8 : 4);
}
// FP64 scoring, FP32 scoring in the workgroup kernel's arithmetic, FP32 scoring
// in the FP32 lane kernel's (64 graphs of an interval and position to a
// wavefront, log-summed there; or 64 evaluations in a row, into A.terms alone,
// for launch_chunk_sums), the FP64 adjoint
enum LanePeelForm { kLpDouble, kLpFloat, kLpFloatLanes, kLpFloatLanesFlat, kLpAdjoint };
// wavefronts the device holds of a form, by its registers (148, 109, 125, 125
// and 256 VGPRs: three, four, four, four and two per SIMD)
constexpr int lanepeel_max_waves(LanePeelForm f) { return f == kLpAdjoint ? 2048 : f == kLpDouble ? 3072 : 4096; }
// wavefronts of a launch over E evaluations when each needs a slot of
// slot_bytes: as many as the device and `budget` bytes hold, evened out over the
// rounds they take
int lanepeel_waves(LanePeelForm form, int64_t E, size_t slot_bytes, size_t budget);
// evaluations in lanes of a launch over G graphs
int64_t lanepeel_lanes(LanePeelForm form, int G, int n_intervals, int npos);
// log-sums of each 64 graphs' terms [G][n] into partial [ceil(G/64)][n], as the
// FP32 lane kernel's wavefronts form them
hipError_t launch_chunk_sums(const double* terms, double* partial, int G, int n, const uint32_t* gate_sweep,
                             int gate_burnin, int gate_period, hipStream_t s);
hipError_t launch_lanepeel(const LanePeelArgs& A, LanePeelForm form, int waves, size_t lds, hipStream_t s);

}  // namespace sl
