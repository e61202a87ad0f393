// Launch of the lane-per-field stage kernel (dg_kernels_quad.hpp; instances in dg_stage_quad.hip):
// mixed precision, 4 fields, tetrahedra of order 3.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "dg_kernels.hpp"

namespace dgk {

constexpr int kQuadGroup = 16;     // elements per group (one wave)
constexpr int kQuadPerBlock = 64;  // elements of a block's four waves

// Operator registers of the kernel for (dim, p); false when none is built or the face-node table
// is not the one the kernel was built with.
bool buildQuadFrag(int dim, int p, const double* Dw, const double* LIFT, const int32_t* fmask, std::vector<double>& frag);
// Resident blocks per CU of the kernel of a stage mode.
int quadBlocksPerCu(int mode);
void launchStageQuad(int mode, const StageArgs<float>& a, int64_t nGroups, unsigned grid, hipStream_t st);

}  // namespace dgk
