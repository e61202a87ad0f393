// Instances and launch of the FP64 matrix-core stage kernel, kept in a translation unit of their own.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dg_kernels_f64.hpp"
#include "dg_stage_f64.hpp"

namespace dgk {
namespace {

template <int P, int NF>
void launchShape(int mode, const StageArgs<double>& a, unsigned grid, hipStream_t st) {
    const dim3 g(grid), b(F64Shape<P, NF>::BS);
    switch (mode) {
        case kModeFirst: hipLaunchKernelGGL((stageKernelF64<P, NF, kModeFirst>), g, b, 0, st, a); break;
        case kModeMid: hipLaunchKernelGGL((stageKernelF64<P, NF, kModeMid>), g, b, 0, st, a); break;
        case kModeFinal: hipLaunchKernelGGL((stageKernelF64<P, NF, kModeFinal>), g, b, 0, st, a); break;
        case kModeEuler: hipLaunchKernelGGL((stageKernelF64<P, NF, kModeEuler>), g, b, 0, st, a); break;
        default: hipLaunchKernelGGL((stageKernelF64<P, NF, kModeRHS>), g, b, 0, st, a); break;
    }
}

template <typename Fn>
bool dispatch(int p, int nf, Fn&& fn) {
    using std::integral_constant;
    auto byNf = [&](auto pc) {
        return nf == 4 ? fn(pc, integral_constant<int, 4>{}) : fn(pc, integral_constant<int, 5>{});
    };
    switch (p) {
        case 4: return byNf(integral_constant<int, 4>{});
        case 5: return byNf(integral_constant<int, 5>{});
    }
    return false;
}

}  // namespace

bool buildF64Frag(int p, int nf, const double* Dw, const double* LIFT, std::vector<double>& frag) {
    return dispatch(p, nf, [&](auto pc, auto nc) {
        using B = F64Shape<decltype(pc)::value, decltype(nc)::value>;
        frag.assign(B::kFrag, 0.0);
        double* o = frag.data();
        for (int it = 0; it < B::MT; ++it) {
            for (int ks = 0; ks < B::KS; ++ks)
                for (int r = 0; r < 3; ++r)
                    for (int lane = 0; lane < 64; ++lane, ++o) {
                        const int i = 16 * it + lane % 16, j = 4 * ks + lane / 16;
                        if (i < B::NP && j < B::NP) *o = Dw[(static_cast<size_t>(r) * B::NP + i) * B::NP + j];
                    }
            for (int h = 0; h < B::H; ++h)
                for (int ks = 0; ks < B::KSL; ++ks)
                    for (int lane = 0; lane < 64; ++lane, ++o) {
                        const int i = 16 * it + lane % 16, k = h * B::PR + 4 * ks + lane / 16;
                        if (i < B::NP && k < B::NFT) *o = -LIFT[static_cast<size_t>(i) * B::NFT + k];
                    }
        }
        return true;
    });
}

void launchStageF64(int p, int nf, int mode, const StageArgs<double>& a, unsigned grid, hipStream_t st) {
    dispatch(p, nf, [&](auto pc, auto nc) {
        launchShape<decltype(pc)::value, decltype(nc)::value>(mode, a, grid, st);
        return true;
    });
}

}  // namespace dgk
