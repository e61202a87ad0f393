// Instances and launch of the resident time loop, kept in a translation unit of their own.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dg_resident.hpp"

namespace dgk {
namespace {

// Triangles of order 1..5 and tetrahedra of order 1..3: the orders whose 256-thread blocks hold at
// least 12 elements (above, a block's elements have nearly all their neighbours in other blocks and
// the LDS holds one block per CU).
template <typename Fn>
bool dispatch(int dim, int p, int nf, Fn&& fn) {
    auto byNf = [&](auto dc, auto pc) {
        return nf == 4 ? fn(dc, pc, std::integral_constant<int, 4>{}) : fn(dc, pc, std::integral_constant<int, 5>{});
    };
    if (nf != 4 && nf != 5) return false;
    auto byP = [&](auto dc) {
        switch (p) {
            case 1: return byNf(dc, std::integral_constant<int, 1>{});
            case 2: return byNf(dc, std::integral_constant<int, 2>{});
            case 3: return byNf(dc, std::integral_constant<int, 3>{});
            case 4:
                if constexpr (decltype(dc)::value == 2) return byNf(dc, std::integral_constant<int, 4>{});
                return false;
            case 5:
                if constexpr (decltype(dc)::value == 2) return byNf(dc, std::integral_constant<int, 5>{});
                return false;
            default: return false;
        }
    };
    return dim == 2 ? byP(std::integral_constant<int, 2>{}) : byP(std::integral_constant<int, 3>{});
}

template <typename T>
const void* kernelOf(int dim, int p, int nf, int shape) {
    const void* f = nullptr;
    dispatch(dim, p, nf, [&](auto dc, auto pc, auto nc) {
        constexpr int D = decltype(dc)::value, P = decltype(pc)::value, NF = decltype(nc)::value;
        auto of = [&](auto sc) -> const void* {
            constexpr int SHAPE = decltype(sc)::value;
            if constexpr (ResidentShape<D, P, NF, T, SHAPE>::kBuilt)
                return reinterpret_cast<const void*>(&residentKernel<D, P, NF, T, sizeof(T) == 4, SHAPE>);
            else
                return nullptr;
        };
        f = shape == kResRows     ? of(std::integral_constant<int, kResRows>{})
            : shape == kResSpread ? of(std::integral_constant<int, kResSpread>{})
            : shape == kResDense  ? of(std::integral_constant<int, kResDense>{})
                                  : of(std::integral_constant<int, kResTight>{});
        return true;
    });
    return f;
}

}  // namespace

int residentElements(int dim, int p, int shape) {
    int eb = 0;
    dispatch(dim, p, 4, [&](auto dc, auto pc, auto) {
        constexpr int D = decltype(dc)::value, P = decltype(pc)::value;
        eb = shape >= kResDense ? ResidentShape<D, P, 4, float, kResDense>::EB : ResidentShape<D, P, 4, float, kResSpread>::EB;
        return true;
    });
    return eb;
}

int residentBlocksPerCu(int dim, int p, int nf, bool fp64, int shape) {
    const void* f = fp64 ? kernelOf<double>(dim, p, nf, shape) : kernelOf<float>(dim, p, nf, shape);
    int n = 0;
    hipFuncAttributes attr{};
    if (!f || hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, kBlock, 0) != hipSuccess ||
        hipFuncGetAttributes(&attr, f) != hipSuccess)
        return 0;
    // the LDS of a block is allocated in units the occupancy query does not round to: 5 blocks of
    // 32,504 bytes fit the 160 KB of a CU by division but were not resident together. A margin of 2 KB
    // per block covers the rounding without knowledge of the unit.
    const int lds = (160 * 1024) / (static_cast<int>(attr.sharedSizeBytes) + 2048);
    return n < lds ? n : lds;
}

template <typename T>
hipError_t launchResident(int dim, int p, int nf, int shape, ResidentArgs<T> a, SourceArgs s, unsigned grid, hipStream_t st) {
    const void* f = kernelOf<T>(dim, p, nf, shape);
    if (!f) return hipErrorInvalidDeviceFunction;
    void* args[] = {&a, &s};
    return hipLaunchCooperativeKernel(f, dim3(grid), dim3(kBlock), args, 0, st);
}

template hipError_t launchResident<float>(int, int, int, int, ResidentArgs<float>, SourceArgs, unsigned, hipStream_t);
template hipError_t launchResident<double>(int, int, int, int, ResidentArgs<double>, SourceArgs, unsigned, hipStream_t);

}  // namespace dgk
