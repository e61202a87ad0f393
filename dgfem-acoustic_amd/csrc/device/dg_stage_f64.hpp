// Launch of the FP64 matrix-core stage kernel (dg_kernels_f64.hpp; instances in dg_stage_f64.hip):
// tetrahedra of order 4 and 5, 4 or 5 fields, one block per 16 elements.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "dg_kernels.hpp"

namespace dgk {

constexpr int kF64Group = 16;  // elements per block

// Operator fragments per row tile: Dw [k-step][direction][64 lanes], then -LIFT [pass][k-step][64];
// lane l holds row l % 16 of the tile, column l / 16 of the k-step. False when no kernel is built.
bool buildF64Frag(int p, int nf, const double* Dw, const double* LIFT, std::vector<double>& frag);
void launchStageF64(int p, int nf, int mode, const StageArgs<double>& a, unsigned grid, hipStream_t st);

}  // namespace dgk
