// Resident time loop for grids small enough to stay on the chip (reference loop:
// src/solver.cpp:311-584, :66-302): one launch runs many steps, every block keeps its elements'
// state, accumulator, operators and geometry in registers and LDS, and only the stage inputs that
// neighbouring blocks read as traces go through memory.
//
// What bounds it: the latency of one exchange per stage, not bandwidth or arithmetic. With a launch
// per stage a 2D step costs four kernel launches of 4-7 us each with cold caches plus the end-of-step
// kernel (8-10 us), whatever the grid's size.
//
// Exchange: every face node whose exterior value belongs to another block has a mailbox (two, used
// in turn). The owner of the exterior value stores it there as soon as its stage is done; the
// reader polls the mailbox itself, so a trace takes one store and one load and no flag, fence or
// block-wide wait lies between. An empty mailbox holds kEmpty words (a NaN pattern no arithmetic
// produces); every value is checked, so the order in which they arrive does not matter. Of a double
// the check looks at the high word only, since a low word may hold any bits: it relies on the aligned
// 8 bytes of a double becoming visible at once, although they are part of a 16-byte store. The reader
// empties the mailbox again, and has that store acknowledged before it sends its own next trace
// of the same face node; the owner writes the same mailbox two epochs later, after it received
// that trace, so a mailbox is always empty when it is written.
//
// Learned faces (DG_BC_LEARNED, mixed precision): further blocks of the launch evaluate the closure network for 16
// faces each. To the block that owns such a face they are one more neighbour: they receive its trace
// in an inbox and answer into the mailboxes of its face nodes. (Evaluated by the owning block itself
// the network's registers came on top of the block's state: its spills made 1,000-block grids slower
// than a launch per stage.)
//
// The blocks wait for one another, so the launch is cooperative (all blocks resident, or it
// fails). Every wait is bounded by a clock all the same (it also ends where a state contains the
// kEmpty pattern): a thread that waits too long sets the chunk's outcome to kAborted, every block
// leaves, and the state in memory is still the one at the start of the chunk: blocks write it back
// only once all of them have finished (kDone).
//
// Residual partials and the state at observer nodes are stored per step and reduced after the
// chunk by residentPostKernel, in the order of postKernel.
#pragma once
#include "dg_closure.hpp"
#include "dg_kernels.hpp"

namespace dgk {

enum : int { kPending = 0, kDone = 1, kAborted = 2 };
enum : int { kResRows = 0, kResSpread = 1, kResDense = 2, kResTight = 3, kResShapes = 4 };

constexpr uint32_t kEmpty = 0xffffffffu;

template <typename T>
struct ResidentArgs {
    T* __restrict__ u;
    T* __restrict__ ulo;
    const T* __restrict__ snap;  // residual snapshot, or null without residuals
    T* mail;                     // two sets of mailboxes of NF values, [K][NFT] for the face nodes, then
    int mailBytes;               //   [learned faces][NFP] inboxes; empty at the start of a chunk; and the
                                 //   bytes of one set
    const int64_t* __restrict__ learned;  // the learned faces (element * NFC + face),
    int nLearned;                         //   their number and the network (packClosure)
    const u32x4_t* __restrict__ net;
    int blocks;                           // blocks of elements; the others evaluate learned faces
    const T* __restrict__ geo;
    const T* __restrict__ fgeo;
    const float* __restrict__ fgeoH;  // (FP32) [K][NFC][4] h n, h (v0.n) with h = Fscale / 2, rounded once
    const int32_t* __restrict__ nbr;
    const uint8_t* __restrict__ code;
    const T* __restrict__ ops;
    const int32_t* __restrict__ iops;
    int* outcome;                          // [chunks], kPending at the start of a batch
    int* done;                             // [chunks] blocks that finished the chunk
    double* __restrict__ resPartial;       // [steps][blocks][5]
    const int32_t* __restrict__ obsOff;    // [blocks + 1] observer entries of each block,
    const int32_t* __restrict__ obsEntry;  //   pairs (thread, slot), threads ascending
    double* __restrict__ obsVal;           // [steps][slots][4]
    const double* __restrict__ srcVal;     // [slots of the batch][nsrc][2]: value, 1 = overwrite
    int* nonfinite;                        // first slot with a non-finite state, or -1
    int64_t K;
    int64_t slot0;       // slot of the chunk's first step in the batch
    int64_t batchSteps;  // steps of the batch
    uint64_t patience;   // longest wait, in ticks of the 100 MHz clock
    T dt;
    int steps;           // steps of the chunk
    int chunk;
    int slots;
    int euler;
    Physics<T> ph;
};

// Shapes of the blocks, the first that the chip holds for a grid:
//   kResRows: a block takes only as many elements as have their face nodes covered by one thread each,
//     and a thread keeps its node's operator rows in registers (where they fit beside its state in
//     256), which shortens the chain of a stage: 2 blocks per CU;
//   kResSpread: the same elements per block, operators in LDS: 4 blocks per CU (FP64 tetrahedra and
//     order 1: 3);
//   kResDense: as many elements as have their nodes covered, several face nodes per thread;
//   kResTight: the same in FP32 at 5 blocks per CU (it spills 8 to 76 registers with 4 fields and 37 to
//     106 with 5).
// Measured against a launch per stage (us per step, 4 fields, one observer; start > resident):
//   triangles p=3 mixed: 200 elements 24.4 > 8.6, 8,000 26.6 > 9.6, 18,000 28.8 > 13.7;
//   FP64 26.5 > 10.5, 31.5 > 14.4, 38.6 > 23.7; p=1 mixed 40,000 25.8 > 12.8;
//   tetrahedra p=2 mixed: 160 29.0 > 10.4, 4,400 29.6 > 11.3; FP64 32.1 > 15.2, 33.5 > 18.6;
//   p=3 mixed: 8,000 38.0 > 24.1, FP64 54.3 > 41.3;
//   learned walls: triangles p=4 mixed 200 42.0 > 19.6, 20,000 54.7 > 26.5; tetrahedra p=3 mixed
//   160 45.6 > 22.7, 8,000 56.7 > 29.4.
// The largest grids of a shape, 4 / 5 fields:
//   mixed kResDense: triangles p=1 86,528 30.6 > 24.8 / 39.2 > 32.0, p=3 25,538 32.0 > 18.5 / 39.2 > 23.1,
//   tetrahedra p=3 10,368 45.0 > 27.1 / 55.8 > 37.3;
//   mixed kResTight: triangles p=2 53,138 35.8 > 30.2 / 46.9 > 41.7, p=3 31,752 35.8 > 27.4 / 46.1 > 37.9,
//   p=5 15,138 40.0 > 22.6 / 52.4 > 29.6, tetrahedra p=3 13,182 50.6 > 38.7 / 63.3 > 51.9 (triangles of
//   order 1 lose there: pickResident);
//   FP64: triangles p=1 31,752 30.1 > 21.8 / 34.9 > 29.4, p=3 21,218 45.4 > 26.1 / 60.1 > 35.4, tetrahedra
//   p=2 6,000 34.8 > 23.8 / 38.9 > 31.4, p=3 7,986 56.1 > 40.1 / 72.2 > 56.7.
template <int DIM, int P, int NF, typename T, int SHAPE>
struct ResidentShape {
    using S = Sizes<DIM, P>;
    static constexpr bool kFp64 = sizeof(T) == 8;
    static constexpr int EB = kBlock / (SHAPE < kResDense && S::NFT > S::NP ? S::NFT : S::NP);
    static constexpr int kFIt = (EB * S::NFT + kBlock - 1) / kBlock;  // face nodes per thread
    static constexpr int kRowRegs = (S::NP * DIM + S::NFT) * static_cast<int>(sizeof(T)) / 4;
    static constexpr bool kOpsReg = SHAPE == kResRows && kRowRegs <= (!kFp64 ? 96 : NF == 4 ? 64 : 44);
    // waves per SIMD asked for: bounds the registers so that this many blocks stay on a CU
    static constexpr int kWaves = SHAPE == kResRows ? 2 : kFp64 && (SHAPE == kResDense || DIM == 3 || P == 1) ? 3 : SHAPE == kResTight ? 5 : 4;
    // Not built where it lost to a launch per stage, its registers spilled: dense blocks with three
    // face nodes per thread (tetrahedra p=2, 13,000 elements, FP64: 47 against 45 us per step, 5
    // fields 82 against 57) or of FP64 triangles of order 1, and spread ones of 5 FP64 fields on
    // tetrahedra of order 1 (13,000 elements: 72 against 34)
    static constexpr bool kBuilt = SHAPE == kResDense    ? kFIt <= 2 && !(kFp64 && P == 1)
                                   : SHAPE == kResTight  ? kFIt <= 2 && !kFp64
                                   : SHAPE == kResSpread ? !(kFp64 && DIM == 3 && P == 1 && NF == 5)
                                                         : true;
};

// Device-scope (SC1: past the L2 of the XCD) accesses of one mailbox: 4 values at index 4 * box as
// 16-byte accesses and, with 5 fields, the fifth in a plane of its own behind those of all boxes.
constexpr int kSc1 = 16;
typedef uint32_t Raw4 __attribute__((ext_vector_type(4)));
typedef uint32_t Raw2 __attribute__((ext_vector_type(2)));

// Both sets of mailboxes as one buffer; `set` below is the set's offset in bytes.
template <typename T>
__device__ inline __amdgpu_buffer_rsrc_t mailBuffer(T* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(p, 0, bytes, 0x00027000);
}

template <int NF, typename T>
__device__ inline void loadMail(__amdgpu_buffer_rsrc_t r, int set, int fifth, int box, T (&v)[NF]) {
    const Raw4 x = __builtin_amdgcn_raw_buffer_load_b128(r, box * 4 * static_cast<int>(sizeof(T)), set, kSc1);
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t w = x[k];  // (a bit cast of the vector element itself reads element 0)
            v[k] = __builtin_bit_cast(float, w);
        }
        if constexpr (NF == 5)
            v[4] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, box * 4, set + fifth, kSc1));
    } else {
        const Raw4 y = __builtin_amdgcn_raw_buffer_load_b128(r, box * 32 + 16, set, kSc1);
        v[0] = __builtin_bit_cast(double, Raw2{x[0], x[1]});
        v[1] = __builtin_bit_cast(double, Raw2{x[2], x[3]});
        v[2] = __builtin_bit_cast(double, Raw2{y[0], y[1]});
        v[3] = __builtin_bit_cast(double, Raw2{y[2], y[3]});
        if constexpr (NF == 5) {
            const Raw2 z = __builtin_amdgcn_raw_buffer_load_b64(r, box * 8, set + fifth, kSc1);
            v[4] = __builtin_bit_cast(double, z);
        }
    }
}

template <int NF, typename T>
__device__ inline void storeMail(__amdgpu_buffer_rsrc_t r, int set, int fifth, int box, const T (&v)[NF]) {
    if constexpr (sizeof(T) == 4) {
        Raw4 x;
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = __builtin_bit_cast(uint32_t, v[k]);
        __builtin_amdgcn_raw_buffer_store_b128(x, r, box * 16, set, kSc1);
        if constexpr (NF == 5)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v[4]), r, box * 4, set + fifth, kSc1);
    } else {
        Raw2 w[NF];
#pragma unroll
        for (int k = 0; k < NF; ++k) w[k] = __builtin_bit_cast(Raw2, v[k]);
        __builtin_amdgcn_raw_buffer_store_b128(Raw4{w[0].x, w[0].y, w[1].x, w[1].y}, r, box * 32, set, kSc1);
        __builtin_amdgcn_raw_buffer_store_b128(Raw4{w[2].x, w[2].y, w[3].x, w[3].y}, r, box * 32 + 16, set, kSc1);
        if constexpr (NF == 5) __builtin_amdgcn_raw_buffer_store_b64(w[4], r, box * 8, set + fifth, kSc1);
    }
}

// Whether every value of a mailbox has arrived.
template <int NF, typename T>
__device__ inline bool arrived(const T (&v)[NF]) {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < NF; ++k) {
        if constexpr (sizeof(T) == 4)
            ok = ok && __builtin_bit_cast(uint32_t, v[k]) != kEmpty;
        else
            ok = ok && static_cast<uint32_t>(__builtin_bit_cast(uint64_t, v[k]) >> 32) != kEmpty;
    }
    return ok;
}

template <typename T>
__device__ inline T emptyValue() {
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float, kEmpty);
    else return __builtin_bit_cast(double, ~uint64_t(0));
}

// All of this thread's vector memory operations are complete (stores acknowledged by memory).
__device__ inline void waitStores() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    asm volatile("" ::: "memory");
}

__device__ inline int deviceLoad(const int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Whether to give up a wait that began at t0: the chunk was aborted, or is now for lack of patience.
__device__ inline bool giveUp(int* outcome, uint64_t t0, uint64_t patience) {
    if (deviceLoad(outcome) == kAborted) return true;
    if (patience > 0 && __builtin_amdgcn_s_memrealtime() - t0 <= patience) return false;
    int expect = kPending;
    __hip_atomic_compare_exchange_strong(outcome, &expect, static_cast<int>(kAborted), __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

template <int DIM, int P, int NF, typename T, bool COMP, int SHAPE>
__global__ __launch_bounds__(kBlock, (ResidentShape<DIM, P, NF, T, SHAPE>::kWaves)) void residentKernel(ResidentArgs<T> a,
                                                                                                     SourceArgs s) {
    using S = Sizes<DIM, P>;
    using L = OpLayout<DIM, P>;
    using R = ResidentShape<DIM, P, NF, T, SHAPE>;
    using V4 = typename Vec4<T>::V;
    constexpr int NP = S::NP, NFP = S::NFP, NFC = S::NFC, NFT = S::NFT, EB = R::EB, JJ = DIM * DIM;
    constexpr int kFIt = R::kFIt;
    constexpr int QS = ldsStride(NP * NF), FS = ldsStride(NFT * NF);
    constexpr int kOpsN = R::kOpsReg ? 1 : L::kN;  // Dw and LIFT; FP64 as two 32-bit planes (see stageKernel)
    constexpr bool kPlanes = sizeof(T) == 8;
    // the stage input and the scaled fluxes of the elements, or the network's exchange
    constexpr int kQF = EB * (QS + FS), kNetLds = static_cast<int>(sizeof(dgc::ClosureLds) / sizeof(T));
    __shared__ __align__(32) T sQF[kQF > kNetLds ? kQF : kNetLds];
    T* const sQ = sQF;
    T* const sF = sQF + EB * QS;
    __shared__ T sJ[EB * JJ];
    __shared__ __align__(32) T sN[EB * NFC * 8];  // unit normal, Fscale; h n, h (v0.n) with h = Fscale / 2
    __shared__ __align__(16) T sOps[kOpsN];
    __shared__ double sRed[kBlock / 16][5];
    __shared__ int sAbort;  // not 0: a thread of the block gave up (learned faces: in epoch sAbort - 1)

    if (a.chunk > 0 && a.outcome[a.chunk - 1] != kDone) {  // an earlier chunk of the batch was aborted
        if (threadIdx.x == 0) a.outcome[a.chunk] = kAborted;
        return;
    }
    const int tid = threadIdx.x;
    int* const outcome = &a.outcome[a.chunk];
    const __amdgpu_buffer_rsrc_t mail = mailBuffer(a.mail, 2 * a.mailBytes);
    const int inbox0 = static_cast<int>(a.K) * NFT;
    const int fifth = (inbox0 + a.nLearned * NFP) * 4 * static_cast<int>(sizeof(T));
    T none[NF];
#pragma unroll
    for (int k = 0; k < NF; ++k) none[k] = emptyValue<T>();
    const int nst = a.euler ? 1 : 4;
    if (tid == 0) sAbort = 0;

    if (static_cast<int>(blockIdx.x) >= a.blocks) {
        // ---- a block of learned faces: trace in, exterior state out, once per stage ----
        if constexpr (sizeof(T) == 4) {  // (FP64 grids with learned faces launch per stage: closureWaveKernel)
            dgc::ClosureLds& lds = *reinterpret_cast<dgc::ClosureLds*>(sQF);
            const int node = tid & 15, idx = (static_cast<int>(blockIdx.x) - a.blocks) * dgc::kTileFaces + (tid >> 4);
            const bool mine = idx < a.nLearned && node < NFP;
            const int lf = idx < a.nLearned ? idx : a.nLearned - 1;
            const int64_t ef = a.learned[lf];
            const int fa = static_cast<int>(ef % NFC) * NFP + (node < NFP ? node : 0);
            const int in = inbox0 + lf * NFP + (node < NFP ? node : 0), out = static_cast<int>(ef / NFC) * NFT + fa;
            const T n[3] = {a.fgeo[ef * 4], a.fgeo[ef * 4 + 1], DIM == 3 ? a.fgeo[ef * 4 + 2] : T(0)};
            const dgc::ClosureNet w = dgc::loadClosureNet(a.net, tid >> 6, tid & 63);
            __syncthreads();
            for (int epoch = 0; epoch < a.steps * nst; ++epoch) {
                T qm[NF], qp[NF];
                const int set = (epoch & 1) * a.mailBytes;
                if (mine) {
                    loadMail<NF>(mail, set, fifth, in, qm);
                    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
                    for (int tries = 1; !arrived<NF>(qm); ++tries) {
                        if ((tries % 64 == 0 || a.patience == 0) && giveUp(outcome, t0, a.patience)) {
                            sAbort = epoch + 1;
                            break;
                        }
                        loadMail<NF>(mail, set, fifth, in, qm);
                    }
                    storeMail<NF>(mail, set, fifth, in, none);
                } else {
#pragma unroll
                    for (int k = 0; k < NF; ++k) qm[k] = T(0);
                }
                dgc::closureExterior<DIM, NFP, NF>(w, lds, a.ph, n, qm, qp);
                // (this epoch's value is set before the barriers inside, so all threads leave or none:
                // one already polling for the next epoch may write that epoch's here)
                if (sAbort == epoch + 1) return;
                waitStores();
                if (mine) storeMail<NF>(mail, set, fifth, out, qp);
            }
        }
        return;
    }

    const int nblk = a.blocks;
    const int bi = static_cast<int>(xcdRemap(blockIdx.x, nblk));
    const int64_t e0 = static_cast<int64_t>(bi) * EB;
    const int nE = static_cast<int>((a.K - e0) < EB ? (a.K - e0) : EB);
    const bool active = tid < nE * NP;
    const int el = active ? tid / NP : 0, i = active ? tid - el * NP : 0;
    const int64_t base = (e0 * NP + (active ? tid : 0)) * NF;
    uint32_t* const sOpsW = reinterpret_cast<uint32_t*>(sOps);

    // ---- once per chunk: state, geometry, operators, the addresses of this thread's face nodes ----
    T u[NF], ulo[NF], acc[NF], q[NF];
    loadNode<NF>(a.u + base, u);
#pragma unroll
    for (int k = 0; k < NF; ++k) {
        ulo[k] = T(0);
        acc[k] = T(0);
        q[k] = u[k];
    }
    if constexpr (COMP) loadNode<NF>(a.ulo + base, ulo);
    T rowD[R::kOpsReg ? NP * DIM : 1], rowL[R::kOpsReg ? NFT : 1];
    if constexpr (R::kOpsReg) {
#pragma unroll
        for (int j = 0; j < NP; ++j)
#pragma unroll
            for (int r = 0; r < DIM; ++r) rowD[j * DIM + r] = a.ops[L::kDw + (j * NP + i) * DIM + r];
#pragma unroll
        for (int fa = 0; fa < NFT; ++fa) rowL[fa] = a.ops[L::kL + fa * NP + i];
    } else {
        for (int x = tid; x < kOpsN; x += kBlock) {
            const T v = a.ops[x];
            if constexpr (kPlanes) {
                const uint64_t b = __builtin_bit_cast(uint64_t, static_cast<double>(v));
                sOpsW[x] = static_cast<uint32_t>(b);
                sOpsW[kOpsN + x] = static_cast<uint32_t>(b >> 32);
            } else {
                sOps[x] = v;
            }
        }
    }
    auto opAt = [&](int k) -> T {
        if constexpr (kPlanes)
            return __builtin_bit_cast(double, Raw2{sOpsW[k], sOpsW[kOpsN + k]});
        else
            return sOps[k];
    };
    for (int x = tid; x < nE * JJ; x += kBlock) sJ[x] = a.geo[e0 * JJ + x];
    for (int x = tid; x < nE * NFC; x += kBlock) {
        const V4 n = reinterpret_cast<const V4*>(a.fgeo + e0 * NFC * 4)[x];
        V4 hn;
        if constexpr (sizeof(T) == 4) {
            // (products of rounded factors would leave a constant error per face: 10-25% more error in
            // the velocities of 2D runs)
            hn = reinterpret_cast<const V4*>(a.fgeoH + e0 * NFC * 4)[x];
        } else {
            const T h = T(0.5) * n.w;
            hn.x = h * n.x;
            hn.y = h * n.y;
            hn.z = h * n.z;
            hn.w = a.ph.v0[0] * hn.x + a.ph.v0[1] * hn.y + a.ph.v0[2] * hn.z;
        }
        reinterpret_cast<V4*>(sN)[2 * x] = n;
        reinterpret_cast<V4*>(sN)[2 * x + 1] = hn;
    }
    // face nodes: own value and face row in LDS; the exterior value in LDS (same block), in this
    // node's mailbox (fExt; the own value goes to fSend, the mailbox of the node opposite), or none
    // (boundary)
    enum : int { kIdle = 0, kLocal = 1, kRemote = 2, kReflect = 3, kAbsorb = 4 };
    int fKind[kFIt], fOwn[kFIt], fRow[kFIt], fExt[kFIt], fSend[kFIt], fOut[kFIt];
#pragma unroll
    for (int c = 0; c < kFIt; ++c) {
        const int it = tid + c * kBlock;
        fKind[c] = kIdle;
        fOwn[c] = fRow[c] = fExt[c] = fSend[c] = fOut[c] = 0;
        if (it < nE * NFT) {
            const int fe = it / NFT, fa = it - fe * NFT, f = fa / NFP, an = fa - f * NFP;
            const int64_t ef = (e0 + fe) * NFC + f;
            const int nb = a.nbr[ef], cd = a.code[ef];
            fOwn[c] = fe * QS + a.iops[L::kMask + f * NFP + an] * NF;
            fRow[c] = (fe * NFC + f) * 8;
            fOut[c] = fe * FS + fa * NF;
            if (nb >= 0) {
                const int opp = (cd & 3) * NFP + a.iops[L::kPerm + (cd >> 2) * NFP + an];  // its face node
                const int64_t lb = nb - e0;
                const bool local = lb >= 0 && lb < nE;
                fKind[c] = local ? kLocal : kRemote;
                fExt[c] = local ? static_cast<int>(lb) * QS + a.iops[L::kMask + opp] * NF
                                : static_cast<int>(e0 + fe) * NFT + fa;
                fSend[c] = nb * NFT + opp;
            } else if (nb <= -3) {  // learned: the block that evaluates face -3 - nb
                fKind[c] = kRemote;
                fExt[c] = static_cast<int>(e0 + fe) * NFT + fa;
                fSend[c] = inbox0 + (-3 - nb) * NFP + an;
            } else {
                fKind[c] = nb == -2 ? kReflect : kAbsorb;
            }
        }
    }
    // this thread's observer entries and source node
    int ob0 = 0, ob1 = 0;
    for (int x = a.obsOff[bi]; x < a.obsOff[bi + 1]; ++x) {
        const int t = a.obsEntry[2 * x];
        if (t < tid) ob0 = x + 1;
        if (t <= tid) ob1 = x + 1;
    }
    if (ob0 == 0) ob0 = a.obsOff[bi];
    int srcLast = -1, srcFirst = 0, srcCount = 0;  // last covering source, the list of all (definition order)
    if (active && s.nnodes > 0) {
        const int64_t node = e0 * NP + tid;
        int64_t lo = 0, hi = s.nnodes;
        while (lo < hi) {
            const int64_t m = (lo + hi) / 2;
            if (s.nodes[m] < node) lo = m + 1;
            else hi = m;
        }
        if (lo < s.nnodes && s.nodes[lo] == node) {
            srcLast = s.lastSrc[lo];
            srcFirst = static_cast<int>(s.coverOff[lo]);
            srcCount = static_cast<int>(s.coverOff[lo + 1]) - srcFirst;
        }
    }
    T qm[kFIt][NF];  // this thread's face nodes: own values of the current stage input
    auto sendTraces = [&](int epoch) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < kFIt; ++c) loadNode<NF>(&sQ[fOwn[c]], qm[c]);
        waitStores();  // the mailboxes emptied in the last stage
#pragma unroll
        for (int c = 0; c < kFIt; ++c)
            if (fKind[c] == kRemote) storeMail<NF>(mail, (epoch & 1) * a.mailBytes, fifth, fSend[c], qm[c]);
    };
    int epoch = 0;
    if (active) storeNode<NF>(&sQ[el * QS + i * NF], q);
    __syncthreads();
    sendTraces(epoch);

    int pendingStep = -1;  // step whose residual rows in sRed are still to be summed
    for (int step = 0; step < a.steps; ++step) {
        const int64_t slot = a.slot0 + step;
        for (int st = 0; st < nst; ++st) {
            const bool last = st == nst - 1;
            // ---- volume contraction and flux-Jacobian fold of the own state ----
            T rhs[NF];
            {
                T Dq[DIM][NF];
#pragma unroll
                for (int r = 0; r < DIM; ++r)
#pragma unroll
                    for (int k = 0; k < NF; ++k) Dq[r][k] = T(0);
                const T* q0 = &sQ[el * QS];
                constexpr int kUnroll = R::kOpsReg ? NP : 4;
#pragma unroll kUnroll
                for (int j = 0; j < NP; ++j) {
                    T qj[NF];
#pragma unroll
                    for (int k = 0; k < NF; ++k) qj[k] = q0[j * NF + k];
#pragma unroll
                    for (int r = 0; r < DIM; ++r) {
                        T d;
                        if constexpr (R::kOpsReg) d = rowD[j * DIM + r];
                        else d = opAt(L::kDw + (j * NP + i) * DIM + r);
#pragma unroll
                        for (int k = 0; k < NF; ++k) Dq[r][k] += d * qj[k];
                    }
                }
                const T* J = &sJ[el * JJ];
                T ar[DIM];
#pragma unroll
                for (int r = 0; r < DIM; ++r) {
                    T v = T(0);
#pragma unroll
                    for (int x = 0; x < DIM; ++x) v += J[r * DIM + x] * a.ph.v0[x];
                    ar[r] = v;
                }
                T sdiv = T(0);
#pragma unroll
                for (int r = 0; r < DIM; ++r)
#pragma unroll
                    for (int x = 0; x < DIM; ++x) sdiv += J[r * DIM + x] * Dq[r][1 + x];
#pragma unroll
                for (int k = 0; k < NF; ++k) {
                    T v = T(0);
#pragma unroll
                    for (int r = 0; r < DIM; ++r) v += ar[r] * Dq[r][k];
                    rhs[k] = v;
                }
                rhs[0] += a.ph.rc2 * sdiv;
                if constexpr (NF == 5) rhs[4] += a.ph.rho0 * sdiv;
#pragma unroll
                for (int kv = 0; kv < DIM; ++kv) {
                    T g = T(0);
#pragma unroll
                    for (int r = 0; r < DIM; ++r) g += J[r * DIM + kv] * Dq[r][0];
                    rhs[1 + kv] += a.ph.irho0 * g;
                }
            }
            // operands of the step's end, fetched while the neighbours finish
            bool srcAct = false;
            double srcVal = 0.0;
            if (last) {
                if (srcLast >= 0 && slot + 1 < a.batchSteps) {
                    // the last covering source that is active (see evalSourceRound)
                    const double* sv = a.srcVal + (slot + 1) * s.nsrc * 2;
                    srcVal = sv[2 * srcLast];
                    srcAct = sv[2 * srcLast + 1] != 0.0;
                    for (int k = srcFirst + srcCount - 2; !srcAct && k >= srcFirst; --k) {
                        srcVal = sv[2 * s.coverSrc[k]];
                        srcAct = sv[2 * s.coverSrc[k] + 1] != 0.0;
                    }
                }
            }

            // ---- exterior values and fluxes ----
            T qp[kFIt][NF];
            bool ok = true;
#pragma unroll
            for (int c = 0; c < kFIt; ++c) {
                if (fKind[c] == kRemote) {
                    loadMail<NF>(mail, (epoch & 1) * a.mailBytes, fifth, fExt[c], qp[c]);
                    ok = ok && arrived<NF>(qp[c]);
                } else {
                    loadNode<NF>(&sQ[fKind[c] == kLocal ? fExt[c] : 0], qp[c]);
                }
            }
            if (!ok) {
                const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
                for (int tries = 1; !ok; ++tries) {
                    ok = true;
#pragma unroll
                    for (int c = 0; c < kFIt; ++c)
                        if (fKind[c] == kRemote) {
                            loadMail<NF>(mail, (epoch & 1) * a.mailBytes, fifth, fExt[c], qp[c]);
                            ok = ok && arrived<NF>(qp[c]);
                        }
                    if (!ok && (tries % 64 == 0 || a.patience == 0) && giveUp(outcome, t0, a.patience)) {
                        sAbort = 1;
                        break;
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < kFIt; ++c) {
                if (fKind[c] == kIdle) continue;
                const T* nf = &sN[fRow[c]];
                T pi[NF];
                if (fKind[c] == kLocal || fKind[c] == kRemote) {
                    if (fKind[c] == kRemote) storeMail<NF>(mail, (epoch & 1) * a.mailBytes, fifth, fExt[c], none);
                    const T hn[3] = {nf[4], nf[5], nf[6]};
                    const T hv = nf[7], cf = nf[3] * (T(0.5) * a.ph.c0);
                    T qs[NF], qd[NF];
#pragma unroll
                    for (int k = 0; k < NF; ++k) {
                        qs[k] = qm[c][k] + qp[c][k];
                        qd[k] = qm[c][k] - qp[c][k];
                    }
                    const T nvs = hn[0] * qs[1] + hn[1] * qs[2] + hn[2] * qs[3];
                    const T t = a.ph.irho0 * qs[0];
                    pi[0] = hv * qs[0] + a.ph.rc2 * nvs + cf * qd[0];
#pragma unroll
                    for (int x = 0; x < 3; ++x) pi[1 + x] = hv * qs[1 + x] + hn[x] * t + cf * qd[1 + x];
                    if constexpr (NF == 5) pi[4] = hv * qs[4] + a.ph.rho0 * nvs + cf * qd[4];
                } else {
                    const T nv[3] = {nf[0], nf[1], nf[2]};
                    numericalFlux<DIM, NF>(a.ph, nv, fKind[c] == kReflect ? -2 : -1, qm[c], qp[c], pi);
#pragma unroll
                    for (int k = 0; k < NF; ++k) pi[k] *= nf[3];
                }
#pragma unroll
                for (int k = 0; k < NF; ++k) sF[fOut[c] + k] = pi[k];
            }
            __syncthreads();
            if (sAbort) return;
            if (pendingStep >= 0) {
                if (tid < 5) {
                    double v = 0.0;
                    for (int r = 0; r < kBlock / 16; ++r) v += sRed[r][tid];
                    a.resPartial[(static_cast<int64_t>(pendingStep) * nblk + blockIdx.x) * 5 + tid] = v;
                }
                pendingStep = -1;
            }

            // ---- lift and register update ----
            {
                const T* f0 = &sF[el * FS];
                constexpr int kUnroll = R::kOpsReg ? NFT : 4;
#pragma unroll kUnroll
                for (int fa = 0; fa < NFT; ++fa) {
                    T l;
                    if constexpr (R::kOpsReg) l = rowL[fa];
                    else l = opAt(L::kL + fa * NP + i);
#pragma unroll
                    for (int k = 0; k < NF; ++k) rhs[k] -= l * f0[fa * NF + k];
                }
            }
            T lnew[NF], unew[NF];
            if (!last) {
                const T half = st == 2 ? T(1) : T(0.5);
#pragma unroll
                for (int k = 0; k < NF; ++k) {
                    const T kk = a.dt * rhs[k];
                    acc[k] = st == 0 ? kk : acc[k] + T(2) * kk;
                    q[k] = u[k] + half * kk;
                }
            } else {
#pragma unroll
                for (int k = 0; k < NF; ++k) {
                    const T kk = a.dt * rhs[k];
                    const T delta = a.euler ? kk : (acc[k] + kk) / T(6);
                    if constexpr (COMP) {
                        T sum, e, t, e2;
                        twoSum(ulo[k], delta, t, e2);
                        twoSum(u[k], t, sum, e);
                        twoSum(sum, e + e2, unew[k], lnew[k]);
                    } else {
                        unew[k] = u[k] + delta;
                        lnew[k] = T(0);
                    }
                    u[k] = unew[k];
                    ulo[k] = lnew[k];
                }
                // the next step starts from the overwritten state; its records from the computed one
                if (srcAct) {
                    const T hi = static_cast<T>(srcVal);
                    u[0] = hi;
                    if constexpr (COMP) ulo[0] = static_cast<T>(srcVal - static_cast<double>(hi));
                    if constexpr (NF == 5) {
                        const double rv = srcVal * s.ic2;
                        const T rh = static_cast<T>(rv);
                        u[4] = rh;
                        if constexpr (COMP) ulo[4] = static_cast<T>(rv - static_cast<double>(rh));
                    }
                }
#pragma unroll
                for (int k = 0; k < NF; ++k) q[k] = u[k];
            }
            if (active) storeNode<NF>(&sQ[el * QS + i * NF], q);
            __syncthreads();
            if (!last || step + 1 < a.steps) sendTraces(++epoch);

            // ---- the step's records, while the traces travel ----
            if (last) {
                T ps[NF];
                if (a.snap) loadNode<NF>(a.snap + base, ps);
                if (active && !allFinite<NF>(unew))
                    atomicMin(reinterpret_cast<unsigned*>(a.nonfinite), static_cast<unsigned>(slot));
                for (int x = ob0; x < ob1; ++x) {
                    const int64_t at = static_cast<int64_t>(step) * a.slots + a.obsEntry[2 * x + 1];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        double v = static_cast<double>(unew[k]);
                        if constexpr (COMP) v += static_cast<double>(lnew[k]);
                        a.obsVal[at * 4 + k] = v;
                    }
                }
                if (a.snap) {
                    double res[5] = {0, 0, 0, 0, 0};
                    if (active) {
                        double d[4], sv[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            sv[k] = static_cast<double>(ps[k]);
                            d[k] = (static_cast<double>(unew[k]) + static_cast<double>(lnew[k])) - sv[k];
                        }
                        const double ic2 = static_cast<double>(a.ph.ic2);
                        const double un = static_cast<double>(unew[0]) + static_cast<double>(lnew[0]);
                        const double sp = sv[0] * ic2 - un * ic2;
                        res[0] = d[0] * d[0];
                        res[1] = sp * sp;
                        res[2] = d[1] * d[1];
                        res[3] = d[2] * d[2];
                        res[4] = d[3] * d[3];
                    }
#pragma unroll
                    for (int k = 0; k < 5; ++k) {
                        const double v = rowSum16(res[k]);
                        if ((tid & 15) == 0) sRed[tid >> 4][k] = v;
                    }
                    pendingStep = step;
                }
            }
        }
    }
    // ---- write back once every block has finished ----
    __syncthreads();
    if (pendingStep >= 0 && tid < 5) {
        double v = 0.0;
        for (int r = 0; r < kBlock / 16; ++r) v += sRed[r][tid];
        a.resPartial[(static_cast<int64_t>(pendingStep) * nblk + blockIdx.x) * 5 + tid] = v;
    }
    if (tid == 0) {
        const int n = __hip_atomic_fetch_add(&a.done[a.chunk], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (n == nblk - 1) {
            int expect = kPending;
            __hip_atomic_compare_exchange_strong(outcome, &expect, static_cast<int>(kDone), __ATOMIC_RELAXED,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
        int got;
        while ((got = deviceLoad(outcome)) == kPending) (void)giveUp(outcome, t0, a.patience);
        if (got != kDone) sAbort = 1;
    }
    __syncthreads();
    if (sAbort || !active) return;
    storeNode<NF>(a.u + base, u);
    if constexpr (COMP) storeNode<NF>(a.ulo + base, ulo);
}

struct ResidentPostArgs {
    const double* resPartial;  // [steps][nblocks][5]
    int64_t nblocks;
    double invN;
    const double* obsVal;      // [steps][slots][4]
    const double* obsW;        // [slots] weights, 0 for padding
    const int32_t* obsSrc;     // [slots] the slot holding the value (padding: its segment's first)
    const int32_t* obsSeg0;    // [nobs + 1]
    int nseg, nobs, slots;
    double* resRing;
    double* obsRing;
    int* nonfinite;
    const int* outcome;        // the chunk's
    int64_t slot0;
    int computeResiduals;
};

// Residuals and observers of a chunk, one block per step: the sums of postKernel in its order.
[[maybe_unused]] static __global__ __launch_bounds__(kPostBlock) void residentPostKernel(ResidentPostArgs p) {
    constexpr int NW = kPostBlock / 64;
    constexpr int kSegChunk = NW;  // segments per pass
    __shared__ double red[NW][5];
    __shared__ double sSeg[kSegChunk][5];
    if (*p.outcome != kDone) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t step = blockIdx.x, slot = p.slot0 + step;
    double acc[5] = {0, 0, 0, 0, 0};
    if (p.computeResiduals)
        for (int64_t b = tid; b < p.nblocks; b += kPostBlock)
#pragma unroll
            for (int k = 0; k < 5; ++k) acc[k] += p.resPartial[(step * p.nblocks + b) * 5 + k];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        double v = acc[k];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
        if (lane == 0) red[wave][k] = v;
    }
    __syncthreads();
    if (tid < 5) {
        double v = 0.0;
        for (int w = 0; w < NW; ++w) v += red[w][tid];
        v *= p.invN;
        p.resRing[slot * 5 + tid] = v;
        if (!isfinite(v)) atomicMin(reinterpret_cast<unsigned*>(p.nonfinite), static_cast<unsigned>(slot));
    }
    // observers: one wave per segment, the segments of a pass summed in order by the observer's thread
    int o = 0;          // (thread 0) the observer being summed
    double ob[5] = {0, 0, 0, 0, 0};
    for (int sg0 = 0; sg0 < p.nseg || (sg0 == 0 && p.nobs > 0); sg0 += kSegChunk) {
        const int sg = sg0 + wave;
        double v[5] = {0, 0, 0, 0, 0};
        if (sg < p.nseg) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int x = sg * 256 + lane + 64 * q;
                const double w = p.obsW[x];
                const double* val = p.obsVal + (step * p.slots + p.obsSrc[x]) * 4;
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] += val[k] * w;
                v[4] += w;
            }
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_down(v[k], off, 64);
                if (lane == 0) sSeg[wave][k] = v[k];
            }
        }
        __syncthreads();
        if (tid == 0) {
            for (int x = sg0; x < sg0 + kSegChunk && x < p.nseg; ++x) {
                while (o < p.nobs && p.obsSeg0[o + 1] <= x) {
                    for (int k = 0; k < 4; ++k) p.obsRing[(slot * p.nobs + o) * 4 + k] = ob[k] / ob[4];
                    for (int k = 0; k < 5; ++k) ob[k] = 0.0;
                    ++o;
                }
                for (int k = 0; k < 5; ++k) ob[k] += sSeg[x - sg0][k];
            }
            if (sg0 + kSegChunk >= p.nseg)
                for (; o < p.nobs; ++o) {
                    for (int k = 0; k < 4; ++k) p.obsRing[(slot * p.nobs + o) * 4 + k] = ob[k] / ob[4];
                    for (int k = 0; k < 5; ++k) ob[k] = 0.0;
                }
        }
        __syncthreads();
    }
}

// Value and activity of every source at the steps of a batch (the resident kernel reads them; the
// evaluation of a sine there would cost all its waves the registers).
[[maybe_unused]] static __global__ __launch_bounds__(256) void residentSourceKernel(SourceArgs s, int64_t steps,
                                                                                    double* __restrict__ out) {
    const int64_t x = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (x >= steps * s.nsrc) return;
    const int64_t slot = x / s.nsrc;
    double v = 0.0;
    const bool on = sourceValue(s, static_cast<int>(x - slot * s.nsrc), slot, s.tTable[slot], v);
    out[2 * x] = v;
    out[2 * x + 1] = on ? 1.0 : 0.0;
}

// Empties the mailboxes for a chunk; before the first chunk of a batch also its outcomes and counts.
[[maybe_unused]] static __global__ __launch_bounds__(256) void residentResetKernel(uint4* mail, int64_t words, int* outcome,
                                                                                   int* done, int chunks) {
    const int64_t x = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (x < words) mail[x] = uint4{kEmpty, kEmpty, kEmpty, kEmpty};
    if (x < chunks) outcome[x] = kPending, done[x] = 0;
}

// Defined in dg_resident.hip, where the instances are built. Elements per block and resident blocks
// per CU of the kernel for (dim, p, nf, precision); 0 when none is built.
int residentElements(int dim, int p, int shape);
int residentBlocksPerCu(int dim, int p, int nf, bool fp64, int shape);
template <typename T>
hipError_t launchResident(int dim, int p, int nf, int shape, ResidentArgs<T> a, SourceArgs s, unsigned grid, hipStream_t st);

}  // namespace dgk
