// FP64 matrix-core stage kernel for tetrahedra: both contractions of a stage on
// v_mfma_f64_16x16x4_f64 (nodal form of getElStiffVector and getElFlux, src/Mesh.cpp:734-751,
// :822-839),
//   rhs = [Dw_1 | Dw_2 | Dw_3 | -LIFT] . [G_1; G_2; G_3; Fscale pi],  G_r = sum_x (dxi_r/dx_x) F_x(q).
//
// A block takes 16 elements (matrix column = element) and has one wave per 16 rows (element nodes),
// which multiplies all fields. The stage input is staged in LDS field-major per element; a lane then
// reads the fields of one node of one element, folds the flux Jacobian into them in registers and
// has the B operands of the node's products of all fields (every wave does this for itself: 45 VALU
// instructions against 12-15 matrix instructions of 64 cycles). Operator fragments stream from L2
// (one 512-byte load per 4-5 products). The numerical fluxes are computed one thread per face node,
// 12 (order 4) or 16 (order 5) face nodes of each element at a time, with the neighbours' traces one
// pass ahead: two faces at a time take 71 KB of LDS at order 5 and leave 2 blocks per CU instead of 3
// (131 against 120 us per stage), and a persistent block that loads its next 16 elements early has
// registers for 2 as well (125 us).
//
// Why: the thread-per-node kernel reads each operator value and each state value once per output
// node and field from L1 and LDS; at order 5 the operator does not fit the LDS. MFMA runs FP64 at
// the VALU's rate, but a fragment serves 16 outputs. RK4 step of 24,576 elements of order 5,
// 5 fields: 775 -> 479 us (a stage 205 -> 120, its floors 62 of memory and 51 of matrix products);
// 63,888 of order 4, 4 fields: 815 -> 482 us. What bounds it now: matrix products (48% of the
// cycles) and VALU (15%) of one SIMD take turns, and the staging and update of all blocks of a CU
// overlap with them only in part.
#pragma once
#include "dg_kernels.hpp"

namespace dgk {

// Smallest stride >= n that is twice an odd number of doubles: 16 elements x 2 consecutive doubles
// read by half a wave then fall in different LDS banks.
__host__ __device__ constexpr int f64Stride(int n) { return n % 4 == 2 ? n : n + 2 - n % 4 + (n % 4 == 3 ? 4 : 0); }

template <int P, int NF>
struct F64Shape {
    using S = Sizes<3, P>;
    static constexpr int NP = S::NP, NFP = S::NFP, NFT = S::NFT;
    static constexpr int G = 16;                     // elements per block
    static constexpr int MT = (NP + 15) / 16;        // row tiles = waves
    static constexpr int BS = 64 * MT;
    static constexpr int KS = (NP + 3) / 4;          // k-steps per direction
    static constexpr int PR = 4 * MT;                // face nodes per pass: one per thread
    static constexpr int H = (NFT + PR - 1) / PR;    // passes over the face nodes
    static constexpr int KSL = MT;                   // k-steps per pass
    static constexpr int QS = 4 * KS, QE = f64Stride(NF * QS);
    static constexpr int PS = PR, PE = f64Stride(NF * PS);
    static constexpr int kFrag = MT * (3 * KS + H * KSL) * 64;  // operator fragment values
    static constexpr int kLds = 8 * G * (QE + PE + 9 + 16) + 8 * G * 4 + 4 * OpLayout<3, P>::kITotal + 8 * 5 * (BS / 16);
    static constexpr int kWaves = 3;  // per SIMD: 3 blocks per CU at order 5, 4 at order 4
    static_assert(kWaves * 4 / MT * (kLds + 1024) <= 160 * 1024);
};

template <int P, int NF, int MODE>
__global__ __launch_bounds__((F64Shape<P, NF>::BS), (F64Shape<P, NF>::kWaves)) void stageKernelF64(StageArgs<double> a) {
    using B = F64Shape<P, NF>;
    using L = OpLayout<3, P>;
    constexpr int NP = B::NP, NFP = B::NFP, G = B::G, BS = B::BS, KS = B::KS, KSL = B::KSL, H = B::H, PR = B::PR;
    constexpr int QS = B::QS, QE = B::QE, PS = B::PS, PE = B::PE;
    constexpr int kStIt = (G * NP * NF / 2 + BS - 1) / BS;  // staged 16-byte words per thread
    constexpr int kNodeIt = (G * NP + BS - 1) / BS;         // element nodes per thread
    constexpr bool kFinal = MODE == kModeFinal || MODE == kModeEuler;
    __shared__ double sQ[G * QE];  // stage input, later the right-hand side
    __shared__ double sP[G * PE];  // Fscale * numerical flux of a pass
    __shared__ double sJ[G * 9];
    __shared__ __align__(32) double sFg[G * 4][4];
    __shared__ int sNb[G * 4];
    __shared__ int sCd[G * 4];
    __shared__ int32_t sI[L::kITotal];
    __shared__ double sRed[BS / 16][5];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const Physics<double> ph = a.ph;
    const int64_t grp = xcdRemap(blockIdx.x, gridDim.x);
    const int64_t e0 = grp * G;
    const int nE = static_cast<int>((a.K - e0) < G ? (a.K - e0) : G);
    const double* const qg = a.qin + e0 * NP * NF;

    // ---- staging ----
    {
        typedef double D2 __attribute__((ext_vector_type(2)));
        const int nw = nE * NP * NF;
        D2 st[kStIt];
#pragma unroll
        for (int c = 0; c < kStIt; ++c) {
            const int x = 2 * (tid + c * BS);
            // (a group starts at a multiple of 16 bytes; the last word of a short odd group by itself)
            if (x + 1 < nw) st[c] = *reinterpret_cast<const D2*>(qg + x);
            else st[c] = D2{x < nw ? qg[x] : 0.0, 0.0};
        }
        for (int x = tid; x < L::kITotal; x += BS) sI[x] = a.iops[x];
        for (int x = tid; x < G * 9; x += BS) sJ[x] = a.geo[e0 * 9 + (x < nE * 9 ? x : x % 9)];
        for (int x = tid; x < G * 4; x += BS) {
            const bool in = x < nE * 4;
            const int64_t ef = e0 * 4 + (in ? x : x % 4);  // past the end: the first element's, without flux
            sNb[x] = in ? a.nbr[ef] : -1;
            sCd[x] = a.code[ef];
            const double4 f = reinterpret_cast<const double4*>(a.fgeo)[ef];
            sFg[x][0] = f.x;
            sFg[x][1] = f.y;
            sFg[x][2] = f.z;
            sFg[x][3] = in ? f.w : 0.0;
        }
#pragma unroll
        for (int c = 0; c < kStIt; ++c)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int y = 2 * (tid + c * BS) + k;
                if (y < G * NP * NF) {
                    const int el = y / (NP * NF), rem = y - el * (NP * NF), node = rem / NF, f = rem - node * NF;
                    sQ[el * QE + f * QS + node] = st[c][k];
                }
            }
        // padding of the k-steps: finite, its operator values are zero
        if constexpr (QS > NP)
            for (int x = tid; x < G * NF * (QS - NP); x += BS) {
                const int row = x / (QS - NP), el = row / NF;
                sQ[el * QE + (row - el * NF) * QS + NP + x % (QS - NP)] = 0.0;
            }
    }
    __syncthreads();

    // ---- fluxes of the face nodes [h PR, (h + 1) PR) of an element, one per thread ----
    double qp[NF];
    const int fel = tid / PR, fk = tid % PR;
    auto gather = [&](int h) __attribute__((always_inline)) {
        const int fa = h * PR + fk;
        const double* src = qg;  // a valid address for idle threads and boundary faces
        if (fa < B::NFT) {
            const int f = fa / NFP, an = fa - f * NFP, nb = sNb[fel * 4 + f], cd = sCd[fel * 4 + f];
            const int nn = sI[L::kMask + (cd & 3) * NFP + sI[L::kPerm + (cd >> 2) * NFP + an]];
            if (nb >= 0) src = a.qin + (static_cast<int64_t>(nb) * NP + nn) * NF;
        }
        loadNode<NF>(src, qp);
    };
    auto fluxes = [&](int h) __attribute__((always_inline)) {
        const int fa = h * PR + fk;
        double pi[NF], fs = 0.0;
#pragma unroll
        for (int k = 0; k < NF; ++k) pi[k] = 0.0;
        if (fa < B::NFT) {
            const int f = fa / NFP, own = sI[L::kMask + fa], ef = fel * 4 + f, nb = sNb[ef];
            double qm[NF];
#pragma unroll
            for (int k = 0; k < NF; ++k) qm[k] = sQ[fel * QE + k * QS + own];
            const double n[3] = {sFg[ef][0], sFg[ef][1], sFg[ef][2]};
            fs = sFg[ef][3];
            numericalFlux<3, NF>(ph, n, nb, qm, qp, pi);  // (no learned faces at these orders)
        }
#pragma unroll
        for (int k = 0; k < NF; ++k) sP[fel * PE + k * PS + fk] = fs * pi[k];
    };
    gather(0);

    // ---- volume products: this wave's 16 nodes, all fields ----
    const int col = lane & 15, kq = lane >> 4;
    const double* aw = a.vfrag + static_cast<int64_t>(wave) * (3 * KS + H * KSL) * 64 + lane;
    md4 acc[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = md4{0.0, 0.0, 0.0, 0.0};
    {
        double J[3][3], ar[3];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            ar[r] = 0.0;
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                J[r][x] = sJ[col * 9 + r * 3 + x];
                ar[r] += J[r][x] * ph.v0[x];
            }
        }
        const double* qc = &sQ[col * QE + kq];
#pragma unroll 2
        for (int ks = 0; ks < KS; ++ks) {
            double q[NF], A[3];
#pragma unroll
            for (int r = 0; r < 3; ++r) A[r] = aw[(ks * 3 + r) * 64];
#pragma unroll
            for (int f = 0; f < NF; ++f) q[f] = qc[f * QS + 4 * ks];
            const double pr = q[0] * ph.irho0;
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const double jv = J[r][0] * q[1] + J[r][1] * q[2] + J[r][2] * q[3];
                double g[NF];
                g[0] = ar[r] * q[0] + ph.rc2 * jv;
#pragma unroll
                for (int x = 0; x < 3; ++x) g[1 + x] = ar[r] * q[1 + x] + J[r][x] * pr;
                if constexpr (NF == 5) g[4] = ar[r] * q[4] + ph.rho0 * jv;
#pragma unroll
                for (int f = 0; f < NF; ++f) acc[f] = MfmaTraits<double>::mma(A[r], g[f], acc[f]);
            }
        }
    }
    // ---- lift products, a pass of face nodes at a time ----
    double up[kNodeIt][NF], ap[kNodeIt][NF];  // registers of the update, loaded behind the last products
#pragma unroll
    for (int h = 0; h < H; ++h) {
        if (h > 0) __syncthreads();  // the last pass's products have read sP
        double A[KSL];
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
        const double* pc = &sP[col * PE + kq];
#pragma unroll
        for (int ks = 0; ks < KSL; ++ks)
#pragma unroll
            for (int f = 0; f < NF; ++f) acc[f] = MfmaTraits<double>::mma(A[ks], pc[f * PS + 4 * ks], acc[f]);
    }
    // (every read of sQ lies before the last pass's barrier)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int node = 16 * wave + MfmaTraits<double>::row(lane, r);
        if (node < NP)
#pragma unroll
            for (int f = 0; f < NF; ++f) sQ[col * QE + f * QS + node] = acc[f][r];
    }
    __syncthreads();

    // ---- register update, one thread per element node ----
    double res[5] = {0, 0, 0, 0, 0};
    const double dt = a.dt;
#pragma unroll
    for (int c = 0; c < kNodeIt; ++c) {
        const int x = tid + c * BS;
        if (x >= nE * NP) continue;
        const int el = x / NP, i = x - el * NP;
        const int64_t base = (e0 * NP + x) * NF;
        double kk[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) kk[f] = dt * sQ[el * QE + f * QS + i];
        if constexpr (MODE == kModeRHS) {
            storeNode<NF>(a.qout + base, kk);
        } else if constexpr (MODE == kModeFirst || MODE == kModeMid) {
            const double half = (MODE == kModeMid && a.stage == kStageRK3) ? 1.0 : 0.5;
            double accn[NF], qn[NF];
            if constexpr (MODE == kModeFirst) loadNode<NF>(a.qin + base, up[c]);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                accn[f] = MODE == kModeFirst ? kk[f] : ap[c][f] + 2.0 * kk[f];
                qn[f] = up[c][f] + half * kk[f];
            }
            storeNodeNT<NF>(a.acc + base, accn);
            storeNode<NF>(a.qout + base, qn);
        } else {
            double ps[NF], unew[NF];
            if constexpr (MODE == kModeEuler) loadNode<NF>(a.qin + base, up[c]);
            if (a.snap) loadNodeNT<NF>(a.snap + base, ps);
#pragma unroll
            for (int f = 0; f < NF; ++f) unew[f] = up[c][f] + (MODE == kModeFinal ? (ap[c][f] + kk[f]) / 6.0 : kk[f]);
            storeNodeNT<NF>(a.uout + base, unew);
            if (!allFinite<NF>(unew)) a.stateBad[0] = 1;
            if (a.snap) {
                double d[4];
#pragma unroll
                for (int f = 0; f < 4; ++f) d[f] = unew[f] - ps[f];
                const double sp = ps[0] * ph.ic2 - unew[0] * ph.ic2;
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
