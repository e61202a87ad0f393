// Stage kernel with a lane per (element, field): tetrahedra, FP32, 4 fields (mixed precision).
//
// A wave owns 16 elements; lane 4 b + f holds field f of element b, all nodes of it in registers.
// v_mfma_f32_4x4x1_16b_f32 multiplies 16 independent 4 x 1 by 1 x 4 blocks: with block = element and
// column = field, the B operand of node j is the lane's own register and the 4 result registers are
// 4 nodes of the same lane, so both contractions of a stage (nodal form of getElStiffVector and
// getElFlux, src/Mesh.cpp:734-751, :822-839) run from registers to registers. The operator column
// Op[4 g .. 4 g + 3][j] is the same for every element: 16 of them share a register and the
// instruction broadcasts one to all blocks (CBSZ = 4, ABID), so the whole operator stays in
// (DIM NP + NFT) NP / 64 registers of a persistent wave. Sums over the fields of a node (v.n, the
// divergence) and the pressure's broadcast are lane moves within 4 lanes.
//
// Why: the thread-per-node kernels are bound by VALU issue at order 3 (577 VALU instructions per 64
// nodes with the volume on the matrix cores, a third of them the lift's FMAs); here 16 elements take
// 1,230 VALU and 500 matrix instructions of 8 cycles (245 and 100 per 64 nodes). No block-wide
// barrier: a wave stages its own LDS (coalesced node vectors <-> lanes). What bounds it is still
// issue: VALU and matrix instructions of a SIMD's three waves add up (without 90% of the volume
// products a stage is 10 us shorter, without the lane moves 7, without the gathers 2, of 73), the
// rest waits for memory that three waves do not cover (First and Mid stages take the same time at 12
// and 20 bytes of state per value). Measured on the 196,608-tetrahedron workload against the
// matrix-core volume variant (vm): stages 84 -> 74 us, final stage 107 -> 101, step 367 -> 330 us;
// 413,526 tetrahedra 753 -> 676 us. Error of the state against 64 bits, 100-200 steps on six meshes:
// 1.42e-7 .. 2.48e-7 against 1.50e-7 .. 2.63e-7 (with the face coefficients h n formed in FP32 it
// was 5-10% larger than vm's).
//
// Per group of 16 elements: stage input, connectivity and geometry are loaded; stage input through
// LDS into lanes; the exterior values of all face nodes are gathered (4 lanes read a node's 16
// bytes); volume products while they are in flight; flux-Jacobian fold; per face the numerical flux
// in the form wA q + wB (v.n) + wC p + wD (q- - q+) with q = q- + q+ (boundary faces: q-, wD = 0), whose
// coefficients depend on the face and field only, straight into the lift products; results through
// LDS back to node vectors for the RK update.
#pragma once
#include <type_traits>
#include <utility>

#include "dg_kernels.hpp"

namespace dgk {

template <int P>
struct QuadShape {
    static constexpr int DIM = 3;
    using S = Sizes<DIM, P>;
    static constexpr int NP = S::NP, NFP = S::NFP, NFC = S::NFC, NFT = S::NFT;
    static constexpr int kGroup = 16;                       // elements per wave
    static constexpr int kWaves = 4;                        // per block
    static constexpr int RG = (NP + 3) / 4;                 // groups of 4 rows
    static constexpr int VR = (DIM * NP * RG + 15) / 16;    // operator registers: volume
    static constexpr int LR = (NFT * RG + 15) / 16;         //   lift
    static constexpr int kFrag = (VR + LR) * 64;
    static constexpr int ES = 4 * NP + (NP % 2 == 0 ? 4 : 0);  // LDS stride of an element: 4 x odd
    static constexpr int NCH = (kGroup * NP + 63) / 64;     // node vectors per lane
    static constexpr int TW = (NFP + 3) / 4;                // words of a row of node bytes
};

// Canonical lattice index of a barycentric tuple (loops l_3 outer .. l_1 inner).
template <int P>
constexpr int latticeIndex(int b1, int b2, int b3) {
    int n = 0;
    for (int k = 0; k <= P; ++k)
        for (int j = 0; j <= P - k; ++j)
            for (int i = 0; i <= P - j - k; ++i, ++n)
                if (i == b1 && j == b2 && k == b3) return n;
    return -1;
}

// Element node of face node a of local face f (the table dg::RefElement::fmask as a constant, so
// that it selects registers; launchStageQuad's caller checks it against the table).
template <int P>
constexpr int faceNode(int f, int a) {
    constexpr int v[4][3] = {{0, 2, 1}, {0, 1, 3}, {0, 3, 2}, {3, 1, 2}};
    int b[4] = {0, 0, 0, 0};
    int n = 0;
    for (int j = 0; j <= P; ++j)
        for (int i = 0; i <= P - j; ++i, ++n)
            if (n == a) {
                b[v[f][0]] = P - i - j;
                b[v[f][1]] = i;
                b[v[f][2]] = j;
            }
    return latticeIndex<P>(b[1], b[2], b[3]);
}

template <int N, typename Fn, int... I>
__device__ __host__ inline void staticForImpl(Fn&& fn, std::integer_sequence<int, I...>) {
    (fn(std::integral_constant<int, I>{}), ...);
}
template <int N, typename Fn>
__device__ __host__ inline void staticFor(Fn&& fn) {
    staticForImpl<N>(static_cast<Fn&&>(fn), std::make_integer_sequence<int, N>{});
}

template <int CTRL>
__device__ inline float quadMove(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
// Sum over the 4 lanes of a quad, in every lane; the value of the quad's first lane.
__device__ inline float quadSum(float v) {
    v += quadMove<0xB1>(v);
    v += quadMove<0x4E>(v);
    return v;
}
__device__ inline float quadFirst(float v) { return quadMove<0x00>(v); }

// c[0..3] += Op[.][slot ABID of a] . b for every lane's block.
template <int ABID>
__device__ inline mf4 quadMma(float a, float b, mf4 c) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 4, ABID, 0);
}

template <int P, int MODE>
__global__ __launch_bounds__(256, (MODE == kModeFinal || MODE == kModeEuler ? 2 : 3)) void stageKernelQuad(StageArgs<float> a, int64_t nGroups) {
    using Q = QuadShape<P>;
    constexpr int DIM = Q::DIM;
    using L = OpLayout<DIM, P>;
    constexpr int NP = Q::NP, NFP = Q::NFP, NFC = Q::NFC, RG = Q::RG, ES = Q::ES, NCH = Q::NCH, G = Q::kGroup;
    constexpr int JJ = DIM * DIM, TW = Q::TW, NPERM = Sizes<DIM, P>::NPERM;
    constexpr bool kNeedU = MODE == kModeMid || MODE == kModeFinal;
    constexpr bool kFinal = MODE == kModeFinal || MODE == kModeEuler;
    __shared__ __align__(16) float sQ[Q::kWaves][G * ES];
    __shared__ float sOp[Q::kFrag];              // operator registers, read as they are used
    __shared__ uint32_t sTab[NFC * NPERM * TW];  // neighbour nodes (bytes) per (its face, permutation)
    __shared__ double sRed[256 / 16][5];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (uniform: group addresses stay scalar)
    const Physics<float> ph = a.ph;
    for (int x = tid; x < NFC * NPERM * TW; x += 256) {
        const int row = x / TW, w = x - row * TW, fp = row / NPERM, pc = row - fp * NPERM;
        uint32_t v = 0;
        for (int k = 0; k < 4 && 4 * w + k < NFP; ++k)
            v |= static_cast<uint32_t>(a.iops[L::kMask + fp * NFP + a.iops[L::kPerm + pc * NFP + 4 * w + k]]) << (8 * k);
        sTab[x] = v;
    }
    for (int x = tid; x < Q::kFrag; x += 256) sOp[x] = a.vfrag[x];
    __syncthreads();

    float* const W = sQ[wave];
    double res[5] = {0, 0, 0, 0, 0};
    // contiguous range of groups per wave; the blocks of one XCD take adjacent ranges
    const int64_t nw = static_cast<int64_t>(gridDim.x) * Q::kWaves;
    const int64_t wi = xcdRemap(blockIdx.x, gridDim.x) * Q::kWaves + wave;
    const int64_t g0 = wi * nGroups / nw, g1 = (wi + 1) * nGroups / nw;
    const char* const qbase = reinterpret_cast<const char*>(a.qin);

    // what a group needs first (its loads one behind another; loading them a group ahead measured no gain)
    struct Group {
        float q[NCH][4];
        int nb[NFC];
        uint32_t cd;  // of the 4 faces
        float fg[NFC];  // h = Fscale / 2: h (v0.n) on lane 0, h n on lanes 1..3 (rounded once from FP64)
        float J[DIM];   // dxi_r/dx of the lane's direction
    };
    auto loadGroup = [&](int64_t grp, Group& n) __attribute__((always_inline)) {
        int lane = tid & 63;
        asm volatile("" : "+v"(lane));
        const int el = lane >> 2, f = lane & 3;
        const int64_t e0 = grp * G;
        const int nE = static_cast<int>((a.K - e0) < G ? (a.K - e0) : G);
        const int e = el < nE ? el : 0;
        const float* qg = a.qin + e0 * NP * 4;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int x = lane + 64 * c;
            loadNode<4>(qg + (x < nE * NP ? x : 0) * 4, n.q[c]);
        }
        const int32_t* nbg = a.nbr + e0 * NFC;
        const uint8_t* cdg = a.code + e0 * NFC;
        const int4 v = reinterpret_cast<const int4*>(nbg)[e];
        n.nb[0] = v.x, n.nb[1] = v.y, n.nb[2] = v.z, n.nb[3] = v.w;
        n.cd = reinterpret_cast<const uint32_t*>(cdg)[e];
        const float* fgg = a.fgeo + e0 * NFC * 4;
#pragma unroll
        for (int k = 0; k < NFC; ++k) n.fg[k] = fgg[(e * NFC + k) * 4 + ((f + 3) & 3)];
        const float* gg = a.geo + e0 * JJ;
#pragma unroll
        for (int r = 0; r < DIM; ++r) n.J[r] = gg[e * JJ + r * DIM + (f >= 1 ? f - 1 : 0)];
    };
    for (int64_t grp = g0; grp < g1; ++grp) {
        Group cur;
        loadGroup(grp, cur);
        // (opaque, so that what follows from the lane is not kept in registers over the loop)
        int lane = tid & 63;
        asm volatile("" : "+v"(lane));
        const int el = lane >> 2, f = lane & 3;
        const float v0l = f == 0 ? 0.0f : f == 1 ? ph.v0[0] : f == 2 ? ph.v0[1] : ph.v0[2];
        const float pl = f == 0 ? 1.0f : 0.0f;  // 1 on the pressure's lane
        const bool dirLane = f >= 1;
        const int64_t e0 = grp * G;
        const int nE = static_cast<int>((a.K - e0) < G ? (a.K - e0) : G);
        const int64_t e = e0 + (el < nE ? el : 0);  // this lane's element (clamped)
        int nb[NFC], cd[NFC];
        float fg[NFC], J[DIM];
#pragma unroll
        for (int k = 0; k < NFC; ++k) {
            nb[k] = cur.nb[k];
            cd[k] = (cur.cd >> (8 * k)) & 0xff;
            fg[k] = cur.fg[k];
        }
#pragma unroll
        for (int r = 0; r < DIM; ++r) J[r] = dirLane ? cur.J[r] : 0.0f;
        // ---- stage input into lanes ----
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int x = lane + 64 * c;
            if (x < nE * NP) storeNode<4>(&W[(x / NP) * ES + (x % NP) * 4], cur.q[c]);
        }
        waveSync();
        float q[NP];
#pragma unroll
        for (int j = 0; j < NP; ++j) q[j] = W[el * ES + j * 4 + f];
        // ---- exterior values of all face nodes ----
        float qp[NFC * NFP];
#pragma unroll
        for (int k = 0; k < NFC; ++k) {
            const int row = ((cd[k] & 3) * NPERM + (cd[k] >> 2)) * TW;
            uint32_t t[TW];
#pragma unroll
            for (int w = 0; w < TW; ++w) t[w] = sTab[row + w];
            const uint32_t src = static_cast<uint32_t>(nb[k] >= 0 ? nb[k] : static_cast<int>(e)) * (NP * 16u) + 4 * f;
#pragma unroll
            for (int x = 0; x < NFP; ++x) {
                const uint32_t nn = (t[x >> 2] >> (8 * (x & 3))) & 0xff;
                qp[k * NFP + x] = *reinterpret_cast<const float*>(qbase + (src + 16 * nn));
            }
            if (nb[k] <= -3) {  // learned face: the exterior states in this face's own node order
                const float* g = a.ghost + static_cast<int64_t>(-3 - nb[k]) * NFP * 4 + f;
#pragma unroll
                for (int x = 0; x < NFP; ++x) qp[k * NFP + x] = g[4 * x];
            }
        }
        // (the scheduler is kept from moving loads and products of one phase into another: with all
        // phases' registers live at once it spills)
        __builtin_amdgcn_sched_barrier(0);
        // ---- volume products and flux-Jacobian fold (see stageKernel): sum_r a_r Dq_r for every
        //      field, rc2 div v for p, grad p / rho0 for v; 4 nodes of all directions at a time ----
        mf4 R[RG];
        {
            float ar[DIM], wp[DIM];
#pragma unroll
            for (int r = 0; r < DIM; ++r) {
                ar[r] = quadSum(J[r] * v0l);
                wp[r] = ph.irho0 * J[r];
            }
            const float wd = pl * ph.rc2;
            staticFor<RG>([&](auto gc) {
                constexpr int g = decltype(gc)::value;
                __builtin_amdgcn_sched_barrier(0);
                mf4 D[DIM];
#pragma unroll
                for (int r = 0; r < DIM; ++r) D[r] = mf4{0.0f, 0.0f, 0.0f, 0.0f};
                float op = 0.0f;
                staticFor<NP * DIM>([&](auto tc) {
                    constexpr int j = decltype(tc)::value / DIM, r = decltype(tc)::value % DIM;
                    constexpr int slot = (g * NP + j) * DIM + r;
                    if constexpr (slot % 16 == 0 || decltype(tc)::value == 0) op = sOp[slot / 16 * 64 + lane];
                    D[r] = quadMma<slot % 16>(op, q[j], D[r]);
                });
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float dv = 0.0f, s = wp[0] * quadFirst(D[0][i]);  // (first: one lane-move multiply)
#pragma unroll
                    for (int r = 0; r < DIM; ++r) {
                        const float d = D[r][i];
                        dv += J[r] * d;
                        s += ar[r] * d;
                        if (r > 0) s += wp[r] * quadFirst(d);
                    }
                    s += wd * quadSum(dv);
                    asm volatile("" : "+v"(s));  // (folded here, not after the products of all nodes)
                    R[g][i] = s;
                }
            });
        }
        __builtin_amdgcn_sched_barrier(0);
        // ---- RK operands of this lane's nodes (consumed at the end) ----
        float pu[NCH][4], pacc[NCH][4];
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int x = lane + 64 * c;
            const int at = (x < nE * NP ? x : 0) * 4;
            if constexpr (kNeedU) {
                loadNodeNT<4>(a.u + e0 * NP * 4 + at, pu[c]);
                loadNodeNT<4>(a.acc + e0 * NP * 4 + at, pacc[c]);
            } else if constexpr (MODE == kModeFirst || MODE == kModeEuler) {
                loadNode<4>(a.qin + e0 * NP * 4 + at, pu[c]);
            }
        }
        // ---- numerical fluxes into the lift products ----
        staticFor<NFC>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            __builtin_amdgcn_sched_barrier(0);
            const float hn = f == 0 ? 0.0f : fg[k];
            const float h = __builtin_amdgcn_sqrtf(quadSum(hn * hn));
            // interior (and learned) faces: n.F((q- + q+)/2) + (c0/2)(q- - q+), scaled by fs
            float wA = quadFirst(fg[k]), wD = h * ph.c0, gl = hn, s = 1.0f, wB = pl * ph.rc2, wC = ph.irho0 * hn;
            if (nb[k] == -1 || nb[k] == -2) {
                const float fs = 2.0f * h, nl = hn / h, vn0 = wA / h;
                gl = nl;
                s = wD = 0.0f;
                if (nb[k] == -2) {
                    wA = vn0 * fs;
                    wB = -vn0 * nl * fs;
                    wC = nl * ph.irho0 * fs;
                } else {
                    const float ac = 0.25f * fs * (ph.c0 + vn0), vl = vn0 < 0.0f ? 0.0f : -0.25f * fs * vn0;
                    wA = f == 0 ? ac : -vl;
                    wB = f == 0 ? ph.c0 * ph.rho0 * ac : (ac + vl) * nl;
                    wC = nl * ac * ph.irc0;
                }
            }
            float pi[NFP];
            staticFor<NFP>([&](auto xc) {
                constexpr int x = decltype(xc)::value, own = faceNode<P>(k, x), fa = k * NFP + x;
                const float qm = q[own], qe = qp[fa];
                const float qs = qm + s * qe;
                const float nv = quadSum(gl * qs);
                float v = wC * quadFirst(qs);
                v += wA * qs;
                v += wD * (qm - qe);  // (the jump as such: small where the solution is smooth)
                pi[x] = v + wB * nv;
            });
            // (the face's fluxes before its products, so that their lane moves overlap)
#pragma unroll
            for (int x = 0; x < NFP; ++x) asm volatile("" : "+v"(pi[x]));
            float op = 0.0f;
            staticFor<NFP * RG>([&](auto tc) {
                constexpr int x = decltype(tc)::value / RG, g = decltype(tc)::value % RG;
                constexpr int slot = (k * NFP + x) * RG + g;
                if constexpr (slot % 16 == 0 || decltype(tc)::value == 0) op = sOp[(Q::VR + slot / 16) * 64 + lane];
                R[g] = quadMma<slot % 16>(op, pi[x], R[g]);
            });
        });
        // ---- right-hand sides back to node vectors ----
        __builtin_amdgcn_sched_barrier(0);
        waveSync();
#pragma unroll
        for (int j = 0; j < NP; ++j) W[el * ES + j * 4 + f] = R[j / 4][j % 4];
        waveSync();
        const float dt = a.dt;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int x = lane + 64 * c;
            if (x >= nE * NP) continue;
            const int64_t gb = e0 * NP * 4;  // (scalar)
            float rhs[4];
            loadNode<4>(&W[(x / NP) * ES + (x % NP) * 4], rhs);
            if constexpr (MODE == kModeRHS) {
                float o[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) o[k] = dt * rhs[k];
                storeNode<4>(a.qout + gb + x * 4, o);
            } else if constexpr (MODE == kModeFirst || MODE == kModeMid) {
                const float half = (MODE == kModeMid && a.stage == kStageRK3) ? 1.0f : 0.5f;
                float accn[4], qn[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float kk = dt * rhs[k];
                    accn[k] = MODE == kModeFirst ? kk : pacc[c][k] + 2.0f * kk;
                    qn[k] = pu[c][k] + half * kk;
                }
                storeNodeNT<4>(a.acc + gb + x * 4, accn);
                storeNode<4>(a.qout + gb + x * 4, qn);
            } else {
                float plo[4], ps[4], unew[4], lnew[4];
                loadNodeNT<4>(a.ulo + gb + x * 4, plo);
                if (a.snap) loadNodeNT<4>(a.snap + gb + x * 4, ps);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float kk = dt * rhs[k];
                    const float delta = (MODE == kModeFinal) ? (pacc[c][k] + kk) / 6.0f : kk;
                    float s_, e_, t_, e2;
                    twoSum(plo[k], delta, t_, e2);
                    twoSum(pu[c][k], t_, s_, e_);
                    twoSum(s_, e_ + e2, unew[k], lnew[k]);
                }
                storeNodeNT<4>(a.uout + gb + x * 4, unew);
                storeNodeNT<4>(a.ulo + gb + x * 4, lnew);
                if (!allFinite<4>(unew)) a.stateBad[0] = 1;
                if (a.snap) {
                    double d[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        d[k] = (static_cast<double>(unew[k]) + static_cast<double>(lnew[k])) - static_cast<double>(ps[k]);
                    const double ic2 = static_cast<double>(ph.ic2);
                    const double u0 = static_cast<double>(unew[0]) + static_cast<double>(lnew[0]);
                    const double sp = static_cast<double>(ps[0]) * ic2 - u0 * ic2;
                    res[0] += d[0] * d[0];
                    res[1] += sp * sp;
                    res[2] += d[1] * d[1];
                    res[3] += d[2] * d[2];
                    res[4] += d[3] * d[3];
                }
            }
        }
        waveSync();  // the next group's staging overwrites the wave's LDS
    }
    if constexpr (kFinal) {
        if (a.snap) blockResiduals<256>(res, sRed, a.resPartial + static_cast<int64_t>(blockIdx.x) * 5);
    }
}

}  // namespace dgk
