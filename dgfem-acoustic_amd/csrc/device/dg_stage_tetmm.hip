// Instances and launch of the tetrahedra matrix-core stage kernel, kept in a translation unit of their own.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dg_kernels_tetmm.hpp"
#include "dg_stage_tetmm.hpp"

namespace dgk {
namespace {

template <typename T, int P, int NF>
void launchShape(int mode, const StageArgs<T>& a, unsigned grid, hipStream_t st) {
    const dim3 g(grid), b(TetMM<T, P, NF>::BS);
    switch (mode) {
        case kModeFirst: hipLaunchKernelGGL((stageKernelTetMM<T, P, NF, kModeFirst>), g, b, 0, st, a); break;
        case kModeMid: hipLaunchKernelGGL((stageKernelTetMM<T, P, NF, kModeMid>), g, b, 0, st, a); break;
        case kModeFinal: hipLaunchKernelGGL((stageKernelTetMM<T, P, NF, kModeFinal>), g, b, 0, st, a); break;
        case kModeEuler: hipLaunchKernelGGL((stageKernelTetMM<T, P, NF, kModeEuler>), g, b, 0, st, a); break;
        default: hipLaunchKernelGGL((stageKernelTetMM<T, P, NF, kModeRHS>), g, b, 0, st, a); break;
    }
}

// (FP32: order 4 only)
template <typename T, typename Fn>
bool dispatch(int p, int nf, Fn&& fn) {
    using std::integral_constant;
    auto byNf = [&](auto pc) {
        return nf == 4 ? fn(pc, integral_constant<int, 4>{}) : fn(pc, integral_constant<int, 5>{});
    };
    if (p == 4) return byNf(integral_constant<int, 4>{});
    if constexpr (sizeof(T) == 8)
        if (p == 5) return byNf(integral_constant<int, 5>{});
    return false;
}

}  // namespace

template <typename T>
bool buildTetMMFrag(int p, int nf, const double* Dw, const double* LIFT, std::vector<T>& frag) {
    return dispatch<T>(p, nf, [&](auto pc, auto nc) {
        using B = TetMM<T, decltype(pc)::value, decltype(nc)::value>;
        frag.assign(B::kFrag, T(0));
        T* o = frag.data();
        for (int it = 0; it < B::MT; ++it) {
            for (int ks = 0; ks < B::KS; ++ks)
                for (int r = 0; r < 3; ++r)
                    for (int lane = 0; lane < 64; ++lane, ++o) {
                        const int i = 16 * it + lane % 16, j = 4 * ks + lane / 16;
                        if (i < B::NP && j < B::NP) *o = static_cast<T>(Dw[(static_cast<size_t>(r) * B::NP + i) * B::NP + j]);
                    }
            for (int h = 0; h < B::H; ++h)
                for (int ks = 0; ks < B::KSL; ++ks)
                    for (int lane = 0; lane < 64; ++lane, ++o) {
                        const int i = 16 * it + lane % 16, k = h * B::PR + 4 * ks + lane / 16;
                        if (i < B::NP && k < B::NFT) *o = static_cast<T>(-LIFT[static_cast<size_t>(i) * B::NFT + k]);
                    }
        }
        return true;
    });
}

template <typename T>
void launchStageTetMM(int p, int nf, int mode, const StageArgs<T>& a, unsigned grid, hipStream_t st) {
    dispatch<T>(p, nf, [&](auto pc, auto nc) {
        launchShape<T, decltype(pc)::value, decltype(nc)::value>(mode, a, grid, st);
        return true;
    });
}

template bool buildTetMMFrag(int, int, const double*, const double*, std::vector<double>&);
template bool buildTetMMFrag(int, int, const double*, const double*, std::vector<float>&);
template void launchStageTetMM(int, int, int, const StageArgs<double>&, unsigned, hipStream_t);
template void launchStageTetMM(int, int, int, const StageArgs<float>&, unsigned, hipStream_t);

}  // namespace dgk
