// Instances and launch of the lane-per-field stage kernel (mixed precision, 4 fields), kept in a
// translation unit of their own.
#include <hip/hip_runtime.h>

#include "dg_stage_quad.hpp"

#include "dg_kernels_quad.hpp"

namespace dgk {
namespace {

// Tetrahedra of order 3. At the other orders the thread-per-node kernels measured as fast or faster
// (us per step, 60-step runs: tetrahedra p=2, 384,000 elements 318 against 324; p=1, 750,000: 247 /
// 262; triangles p=3, 180,000: 143 / 165; p=5, 80,000: 141 / 156): they are near the memory there.
using Kernel = void (*)(StageArgs<float>, int64_t);
Kernel kernelOf(int mode) {
    switch (mode) {
        case kModeFirst: return &stageKernelQuad<3, kModeFirst>;
        case kModeMid: return &stageKernelQuad<3, kModeMid>;
        case kModeFinal: return &stageKernelQuad<3, kModeFinal>;
        case kModeEuler: return &stageKernelQuad<3, kModeEuler>;
        default: return &stageKernelQuad<3, kModeRHS>;
    }
}

}  // namespace

bool buildQuadFrag(int dim, int p, const double* Dw, const double* LIFT, const int32_t* fmask, std::vector<double>& frag) {
    if (dim != 3 || p != 3) return false;
    constexpr int P = 3;
    using Q = QuadShape<P>;
    bool same = true;
    staticFor<Q::NFC>([&](auto fc) {
        staticFor<Q::NFP>([&](auto ac) {
            constexpr int f = decltype(fc)::value, a = decltype(ac)::value, n = faceNode<P>(f, a);
            same = same && fmask[f * Q::NFP + a] == n;
        });
    });
    if (!same) return false;
    frag.assign(Q::kFrag, 0.0);
    // slot s of a part: register s / 16, lanes 4 (s % 16) + i hold row 4 g + i
    auto put = [&](int reg0, int slot, int g, auto&& at) {
        for (int i = 0; i < 4; ++i)
            if (4 * g + i < Q::NP) frag[(reg0 + slot / 16) * 64 + 4 * (slot % 16) + i] = at(4 * g + i);
    };
    for (int g = 0; g < Q::RG; ++g)
        for (int j = 0; j < Q::NP; ++j)
            for (int r = 0; r < Q::DIM; ++r)
                put(0, (g * Q::NP + j) * Q::DIM + r, g,
                    [&](int i) { return Dw[(static_cast<size_t>(r) * Q::NP + i) * Q::NP + j]; });
    for (int fa = 0; fa < Q::NFT; ++fa)
        for (int g = 0; g < Q::RG; ++g)
            put(Q::VR, fa * Q::RG + g, g, [&](int i) { return -LIFT[static_cast<size_t>(i) * Q::NFT + fa]; });
    return true;
}

int quadBlocksPerCu(int mode) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(kernelOf(mode)), 256, 0) != hipSuccess)
        return 0;
    return n;
}

void launchStageQuad(int mode, const StageArgs<float>& a, int64_t nGroups, unsigned grid, hipStream_t st) {
    hipLaunchKernelGGL(kernelOf(mode), dim3(grid), dim3(256), 0, st, a, nGroups);
}

}  // namespace dgk
