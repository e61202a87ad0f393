// Launch of the matrix-core stage kernel of tetrahedra (dg_kernels_tetmm.hpp; instances in dg_stage_tetmm.hip):
// orders 4 and 5, 4 or 5 fields, one block per 16 elements.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "dg_kernels.hpp"

namespace dgk {

constexpr int kTetMMGroup = 16;  // elements per block

// Operator fragments per row tile: Dw [k-step][direction][64 lanes], then -LIFT [pass][k-step][64];
// lane l holds row l % 16 of the tile, column l / 16 of the k-step. False when no kernel is built.
template <typename T>
bool buildTetMMFrag(int p, int nf, const double* Dw, const double* LIFT, std::vector<T>& frag);
template <typename T>
void launchStageTetMM(int p, int nf, int mode, const StageArgs<T>& a, unsigned grid, hipStream_t st);

}  // namespace dgk
