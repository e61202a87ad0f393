// Matrix-core stage kernel of tetrahedra of order 4 and 5 in FP64 and order 4 in mixed precision: both
// contractions of a stage on v_mfma_f64_16x16x4_f64 / v_mfma_f32_16x16x4_f32 (nodal form of
// getElStiffVector and getElFlux, src/Mesh.cpp:734-751, :822-839),
//   rhs = [Dw_1 | Dw_2 | Dw_3 | -LIFT] . [G_1; G_2; G_3; Fscale pi],  G_r = sum_x (dxi_r/dx_x) F_x(q).
//
// A block takes 16 elements (matrix column = element) and has one wave per 16 rows (element nodes),
// which multiplies all fields. The stage input is staged in LDS as it lies in memory; a lane reads the
// fields of one node of one element, the B operands of the node's products of all fields. FP32
// multiplies q and applies the flux Jacobian to the products; in FP64 the registers of that spill,
// and the Jacobian is folded into the operands (by every wave for itself: 45 VALU instructions against
// 12-15 products of 64 cycles). Operator fragments stream from L2 (one load per 4-5 products). The
// numerical fluxes are computed one thread per face node, 12 (order 4) or 16 (order 5) face nodes of
// each element at a time, with the neighbours' traces one pass ahead: two faces at a time take 71 KB
// of LDS in FP64 at order 5 and leave 2 blocks per CU instead of 3 (131 against 120 us per stage). A
// persistent block that loads its next 16 elements early measured 125 us there, and no gain in FP32.
//
// Why: the thread-per-node kernel reads each operator value and each state value once per output
// node and field from L1 and LDS; at order 5 the operator does not fit the LDS. FP64 runs on the
// matrix cores at the VALU's rate, but a fragment serves 16 outputs. us per RK4 step, before > now:
//   FP64  24,576 order 5, 5 fields 773 > 464 (4: 713 > 351);  63,888 order 4, 4 fields 813 > 463
//   mixed 162,000 order 4, 5 fields 1080 > 865 (4: 862 > 636)
// What bounds it now: the order-5 FP64 stage of 120 us has 51 us of products (48% of the cycles) and
// 62 us of memory traffic; blocks start together and stay in step, so that the two overlap little.
#pragma once
#include "dg_kernels.hpp"

namespace dgk {

// Smallest stride >= n with which the 16 elements x 4 (FP32; FP64: 2) consecutive values that a wave
// (half a wave) reads at once fall in different LDS banks: an odd multiple of 4 (2) values.
template <typename T>
__host__ __device__ constexpr int tetMMStride(int n) {
    const int m = sizeof(T) == 4 ? 4 : 2, k = (n + m - 1) / m;
    return m * (k % 2 ? k : k + 1);
}

template <typename T, int P, int NF>
struct TetMM {
    using S = Sizes<3, P>;
    static constexpr int NP = S::NP, NFP = S::NFP, NFT = S::NFT;
    static constexpr int G = 16;                     // elements per block
    static constexpr int MT = (NP + 15) / 16;        // row tiles = waves
    static constexpr int BS = 64 * MT;
    static constexpr int KS = (NP + 3) / 4;          // k-steps per direction
    static constexpr int PR = 4 * MT;                // face nodes per pass: one per thread
    static constexpr int H = (NFT + PR - 1) / PR;    // passes over the face nodes
    static constexpr int KSL = MT;                   // k-steps per pass
    static constexpr int QE = tetMMStride<T>(NF * 4 * KS);  // element stride of the staged input
    static constexpr int PE = tetMMStride<T>(NF * PR);      // and of the fluxes of a pass
    static constexpr int kFrag = MT * (3 * KS + H * KSL) * 64;  // operator fragment values
    static constexpr int kLds = static_cast<int>(sizeof(T)) * G * (QE + PE + 9 + 16) + 8 * G * 4 +
                                4 * OpLayout<3, P>::kITotal + 8 * 5 * (BS / 16);
    // the flux Jacobian on the derivatives (once per node, 3 NF accumulators) instead of on the operands
    // (once per node and wave): in FP64 the registers of that spill
    static constexpr bool kFoldAfter = sizeof(T) == 4;
    static constexpr int kWaves = sizeof(T) == 4 ? 4 : 3;  // per SIMD
    static_assert(kWaves * 4 / MT * (kLds + 1024) <= 160 * 1024);
};

template <typename T, int P, int NF, int MODE>
__global__ __launch_bounds__((TetMM<T, P, NF>::BS), (TetMM<T, P, NF>::kWaves)) void stageKernelTetMM(StageArgs<T> a) {
    using B = TetMM<T, P, NF>;
    using L = OpLayout<3, P>;
    constexpr int NP = B::NP, NFP = B::NFP, G = B::G, BS = B::BS, KS = B::KS, KSL = B::KSL, H = B::H, PR = B::PR;
    constexpr int QE = B::QE, PE = B::PE, EV = NP * NF;
    constexpr bool COMP = sizeof(T) == 4;  // mixed precision: compensated state
    constexpr int VW = 16 / sizeof(T);
    using V = typename MfmaTraits<T>::V;
    typedef T T4 __attribute__((ext_vector_type(4)));
    constexpr int kStIt = (G * NP * NF / VW + BS - 1) / BS;  // staged 16-byte words per thread
    constexpr int kNodeIt = (G * NP + BS - 1) / BS;         // element nodes per thread
    constexpr bool kFinal = MODE == kModeFinal || MODE == kModeEuler;
    __shared__ __align__(16) T sQ[G * QE];  // stage input, later the right-hand side
    __shared__ __align__(16) T sP[G * PE];  // Fscale * numerical flux of a pass
    __shared__ T sJ[G * 9];
    __shared__ __align__(16) T sFg[G * 4][4];
    __shared__ int sNb[G * 4];
    __shared__ int sCd[G * 4];
    __shared__ int32_t sI[L::kITotal];
    __shared__ double sRed[BS / 16][5];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const Physics<T> ph = a.ph;
    const int64_t grp = xcdRemap(blockIdx.x, gridDim.x);
    const int64_t e0 = grp * G;
    const int nE = static_cast<int>((a.K - e0) < G ? (a.K - e0) : G);
    const T* const qg = a.qin + e0 * NP * NF;

    // ---- staging ----
    {
        typedef T W __attribute__((ext_vector_type(VW)));
        const int nw = nE * NP * NF;
        W st[kStIt];
#pragma unroll
        for (int c = 0; c < kStIt; ++c) {
            const int x = VW * (tid + c * BS);
            // (a block starts at a multiple of 16 bytes; a rest of less than 16 is loaded by values)
            if (x + VW <= nw) {
                st[c] = *reinterpret_cast<const W*>(qg + x);
            } else {
#pragma unroll
                for (int k = 0; k < VW; ++k) st[c][k] = x + k < nw ? qg[x + k] : T(0);
            }
        }
        for (int x = tid; x < L::kITotal; x += BS) sI[x] = a.iops[x];
        for (int x = tid; x < G * 9; x += BS) sJ[x] = a.geo[e0 * 9 + (x < nE * 9 ? x : x % 9)];
        for (int x = tid; x < G * 4; x += BS) {
            const bool in = x < nE * 4;
            const int64_t ef = e0 * 4 + (in ? x : x % 4);  // past the end: the first element's, without flux
            sNb[x] = in ? a.nbr[ef] : -1;
            sCd[x] = a.code[ef];
            const T4 f = reinterpret_cast<const T4*>(a.fgeo)[ef];
            sFg[x][0] = f.x;
            sFg[x][1] = f.y;
            sFg[x][2] = f.z;
            sFg[x][3] = in ? f.w : T(0);
        }
#pragma unroll
        for (int c = 0; c < kStIt; ++c) {
            const int y = VW * (tid + c * BS), el = y / EV, rem = y - el * EV;
            if (y >= G * EV) continue;
            T* dst = &sQ[el * QE + rem];
            if constexpr (EV % VW == 0 && QE % VW == 0) {
                *reinterpret_cast<W*>(dst) = st[c];
            } else {
#pragma unroll
                for (int k = 0; k < VW; ++k)
                    if (G * EV % VW == 0 || y + k < G * EV) dst[rem + k < EV ? k : k + QE - EV] = st[c][k];
            }
        }
        // padding of the k-steps: finite, its operator values are zero
        if constexpr (4 * KS > NP)
            for (int x = tid; x < G * (4 * KS - NP) * NF; x += BS) {
                const int el = x / ((4 * KS - NP) * NF);
                sQ[el * QE + EV + x - el * (4 * KS - NP) * NF] = T(0);
            }
    }
    __syncthreads();

    // ---- fluxes of the face nodes [h PR, (h + 1) PR) of an element, one per thread ----
    T qp[NF];
    const int fel = tid / PR, fk = tid % PR;
    auto gather = [&](int h) __attribute__((always_inline)) {
        const int fa = h * PR + fk;
        const T* src = qg;  // a valid address for idle threads and boundary faces
        if (fa < B::NFT) {
            const int f = fa / NFP, an = fa - f * NFP, nb = sNb[fel * 4 + f], cd = sCd[fel * 4 + f];
            const int nn = sI[L::kMask + (cd & 3) * NFP + sI[L::kPerm + (cd >> 2) * NFP + an]];
            if (nb >= 0) src = a.qin + (static_cast<int64_t>(nb) * NP + nn) * NF;
        }
        loadNode<NF>(src, qp);
    };
    auto fluxes = [&](int h) __attribute__((always_inline)) {
        const int fa = h * PR + fk;
        T pi[NF], fs = T(0);
#pragma unroll
        for (int k = 0; k < NF; ++k) pi[k] = T(0);
        if (fa < B::NFT) {
            const int f = fa / NFP, own = sI[L::kMask + fa], ef = fel * 4 + f, nb = sNb[ef];
            T qm[NF];
#pragma unroll
            for (int k = 0; k < NF; ++k) qm[k] = sQ[fel * QE + own * NF + k];
            const T n[3] = {sFg[ef][0], sFg[ef][1], sFg[ef][2]};
            fs = sFg[ef][3];
            numericalFlux<3, NF>(ph, n, nb, qm, qp, pi);  // (no learned faces at these orders)
        }
#pragma unroll
        for (int k = 0; k < NF; ++k) sP[fel * PE + fk * NF + k] = fs * pi[k];
    };
    gather(0);

    // ---- volume products: this wave's 16 nodes, all fields ----
    const int col = lane & 15, kq = lane >> 4;
    const T* aw = a.vfrag + static_cast<int64_t>(wave) * (3 * KS + H * KSL) * 64 + lane;
    V acc[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = V{0, 0, 0, 0};
    const T* qc = &sQ[col * QE + kq * NF];
    const T* J = &sJ[col * 9];  // of the column's element
    // value of the flux in direction r at one node, or of its derivative
    auto fold = [&](int r, const T (&q)[NF], T (&g)[NF]) __attribute__((always_inline)) {
        const T ar = J[r * 3] * ph.v0[0] + J[r * 3 + 1] * ph.v0[1] + J[r * 3 + 2] * ph.v0[2];
        const T jv = J[r * 3] * q[1] + J[r * 3 + 1] * q[2] + J[r * 3 + 2] * q[3], pr = q[0] * ph.irho0;
        g[0] = ar * q[0] + ph.rc2 * jv;
#pragma unroll
        for (int x = 0; x < 3; ++x) g[1 + x] = ar * q[1 + x] + J[r * 3 + x] * pr;
        if constexpr (NF == 5) g[4] = ar * q[4] + ph.rho0 * jv;
    };
    if constexpr (B::kFoldAfter) {
        V Dq[3][NF];
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int f = 0; f < NF; ++f) Dq[r][f] = V{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            T q[NF], A[3];
#pragma unroll
            for (int r = 0; r < 3; ++r) A[r] = aw[(ks * 3 + r) * 64];
#pragma unroll
            for (int f = 0; f < NF; ++f) q[f] = qc[4 * ks * NF + f];
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int f = 0; f < NF; ++f) Dq[r][f] = MfmaTraits<T>::mma(A[r], q[f], Dq[r][f]);
        }
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                T q[NF], g[NF];
#pragma unroll
                for (int f = 0; f < NF; ++f) q[f] = Dq[r][f][k];
                fold(r, q, g);
#pragma unroll
                for (int f = 0; f < NF; ++f) acc[f][k] += g[f];
            }
    } else {
#pragma unroll 2
        for (int ks = 0; ks < KS; ++ks) {
            T q[NF], A[3];
#pragma unroll
            for (int r = 0; r < 3; ++r) A[r] = aw[(ks * 3 + r) * 64];
#pragma unroll
            for (int f = 0; f < NF; ++f) q[f] = qc[4 * ks * NF + f];
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                T g[NF];
                fold(r, q, g);
#pragma unroll
                for (int f = 0; f < NF; ++f) acc[f] = MfmaTraits<T>::mma(A[r], g[f], acc[f]);
            }
        }
    }
    // ---- lift products, a pass of face nodes at a time ----
    T up[kNodeIt][NF], ap[kNodeIt][NF];  // registers of the update, loaded behind the last products
#pragma unroll
    for (int h = 0; h < H; ++h) {
        if (h > 0) __syncthreads();  // the last pass's products have read sP
        T A[KSL];
#pragma unroll
        for (int ks = 0; ks < KSL; ++ks) A[ks] = aw[(3 * KS + h * KSL + ks) * 64];
        fluxes(h);
        __syncthreads();
        if (h + 1 < H) gather(h + 1);
        if constexpr (MODE == kModeMid || MODE == kModeFinal) {
            if (h + 1 == H)
#pragma unroll
                for (int c = 0; c < kNodeIt; ++c) {
                    const int x = tid + c * BS;
                    const int64_t base = (e0 * NP + (x < nE * NP ? x : 0)) * NF;
                    loadNodeNT<NF>(a.u + base, up[c]);
                    loadNodeNT<NF>(a.acc + base, ap[c]);
                }
        }
        const T* pc = &sP[col * PE + kq * NF];
#pragma unroll
        for (int ks = 0; ks < KSL; ++ks)
#pragma unroll
            for (int f = 0; f < NF; ++f) acc[f] = MfmaTraits<T>::mma(A[ks], pc[4 * ks * NF + f], acc[f]);
    }
    // (every read of sQ lies before the last pass's barrier)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int node = 16 * wave + MfmaTraits<T>::row(lane, r);
        if (node < NP)
#pragma unroll
            for (int f = 0; f < NF; ++f) sQ[col * QE + node * NF + f] = acc[f][r];
    }
    __syncthreads();

    // ---- register update, one thread per element node ----
    double res[5] = {0, 0, 0, 0, 0};
    const T dt = a.dt;
#pragma unroll
    for (int c = 0; c < kNodeIt; ++c) {
        const int x = tid + c * BS;
        if (x >= nE * NP) continue;
        const int el = x / NP, i = x - el * NP;
        const int64_t base = (e0 * NP + x) * NF;
        T kk[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) kk[f] = dt * sQ[el * QE + i * NF + f];
        if constexpr (MODE == kModeRHS) {
            storeNode<NF>(a.qout + base, kk);
        } else if constexpr (MODE == kModeFirst || MODE == kModeMid) {
            const T half = (MODE == kModeMid && a.stage == kStageRK3) ? T(1) : T(0.5);
            T accn[NF], qn[NF];
            if constexpr (MODE == kModeFirst) loadNode<NF>(a.qin + base, up[c]);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                accn[f] = MODE == kModeFirst ? kk[f] : ap[c][f] + T(2) * kk[f];
                qn[f] = up[c][f] + half * kk[f];
            }
            storeNodeNT<NF>(a.acc + base, accn);
            storeNode<NF>(a.qout + base, qn);
        } else {
            T ps[NF], plo[NF], unew[NF], lnew[NF];
            if constexpr (MODE == kModeEuler) loadNode<NF>(a.qin + base, up[c]);
            if constexpr (COMP) loadNodeNT<NF>(a.ulo + base, plo);
            if (a.snap) loadNodeNT<NF>(a.snap + base, ps);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const T delta = MODE == kModeFinal ? (ap[c][f] + kk[f]) / T(6) : kk[f];
                if constexpr (COMP) {
                    T s, e, t, e2;
                    twoSum(plo[f], delta, t, e2);
                    twoSum(up[c][f], t, s, e);
                    twoSum(s, e + e2, unew[f], lnew[f]);
                } else {
                    unew[f] = up[c][f] + delta;
                    lnew[f] = T(0);
                }
            }
            storeNodeNT<NF>(a.uout + base, unew);
            if constexpr (COMP) storeNodeNT<NF>(a.ulo + base, lnew);
            if (!allFinite<NF>(unew)) a.stateBad[0] = 1;
            if (a.snap) {
                double d[4];
#pragma unroll
                for (int f = 0; f < 4; ++f)
                    d[f] = (static_cast<double>(unew[f]) + lnew[f]) - static_cast<double>(ps[f]);
                const double ic2 = static_cast<double>(ph.ic2);
                const double sp = ps[0] * ic2 - (static_cast<double>(unew[0]) + lnew[0]) * ic2;
                res[0] += d[0] * d[0];
                res[1] += sp * sp;
                res[2] += d[1] * d[1];
                res[3] += d[2] * d[2];
                res[4] += d[3] * d[3];
            }
        }
    }
    if constexpr (kFinal) {
        if (a.snap) blockResiduals<BS>(res, sRed, a.resPartial + static_cast<int64_t>(blockIdx.x) * 5);
    }
}

}  // namespace dgk
