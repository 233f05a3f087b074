// Block-level GEMM: one problem per workgroup, waves on a PM x PN x PK grid.
//
// This is the MI355X form of KAMI's communication-avoiding block GEMM
// (src/block_gemm/KAMI/{1d,2d,3d}/fp64/block_gemm_{1d,2d,3d}_double_mma.cu and the
// fp16 variants).  The partition names keep the reference's meaning:
//   1D  (PM = P, PN = 1, PK = 1): each wave owns M/P rows of A, held in registers for
//       the whole product (the reference's a_frags, F64-1D:73-102); B is the only
//       operand that crosses waves and it goes through LDS (F64-1D:148-185).
//   2D  (PM = PN = P, PK = 1): wave (r, c) owns C(r, c); A rows are shared along a wave
//       row and B columns along a wave column through LDS (F64-2D:156-186).
//   3D  (PK > 1): as 2D, and K is split over a depth axis; the PK partial C tiles are
//       reduced on the device through LDS (the reference sums slabs on the host,
//       F64-3D:324-333).
// Differences from the reference that are deliberate:
//   * operands shared between waves are staged into LDS once per K stage with 16-byte
//     coalesced loads, not written by an owner wave from its registers, and the stage
//     buffers are double-buffered so one barrier per stage suffices (the reference's
//     2D kernel is missing its post-MMA barrier, F64-2D:188-212);
//   * the wave64 MFMA atoms of kami_device.hpp replace mma.sync m16n8k8 / m16n8k16;
//   * alpha and beta are honoured (the reference ignores them, F64-1D:55 vs :205-208);
//   * `iters` repeats the whole product into the same accumulators, which is the
//     reference's resident-repeat NUM_ITER loop (F64-1D:140); iters = 1 is a plain GEMM.
#pragma once

#include "kami_device.hpp"

namespace kami {

constexpr int cmin(int a, int b) { return a < b ? a : b; }
constexpr int cmax(int a, int b) { return a > b ? a : b; }

// B_: B is stored N x K, or K x N.  Then its K rows go to LDS as they are and the reads turn
// them.  (Turning them in the writes instead cost eight 2-byte or two 8-byte conflicting stores a piece:
// FP16 256^3 x 1024 183 us against 114.5, 224^3 x 2048 246 against 177, FP64 128^3 x 4096 431
// against 376, 64 x 64 x 512 x 2048 273 against 226; N x K 111, 187, 335 and 209.)
// Many repeated products on one stage of 2-byte values are another matter: the reads are
// repeated and the writes are not, and a turned fragment is two reads of half a row where a row of
// K is one.  They turn the rows in the writes (TURNED, from turn_iters on): 64^3 x 1024, 400 times,
// BF16 104 us against 164, 128 x 128 x 32 x 1024, 279 times, 158 against 238, 256^3 x 1024, 8
// times, 318 against 403.
enum BStage : int { kStageNK, kStageRows, kStageTurned };
template <class AT, int BM_, int BN_, int BK_, int PM_, int PN_, int PK_, int KS_, int B_ = kStageNK>
struct BlockGeom {
    static constexpr bool SRC_KN = B_ != kStageNK;    // K rows in memory
    static constexpr bool KN = B_ == kStageRows;      // K rows in LDS
    static constexpr bool TURNED = B_ == kStageTurned;
    using AsKN = BlockGeom<AT, BM_, BN_, BK_, PM_, PN_, PK_, KS_, kStageRows>;
    using AsTurned = BlockGeom<AT, BM_, BN_, BK_, PM_, PN_, PK_, KS_, kStageTurned>;
    static constexpr int BM = BM_, BN = BN_, BK = BK_;
    static constexpr int PM = PM_, PN = PN_, PK = PK_, KS = KS_;
    static constexpr int WAVES = PM * PN * PK;
    static constexpr int NT = WAVES * kWave;
    static constexpr int TM = BM / PM, TN = BN / PN;
    // atom edge (16, or 32 for the 32 x 32 atoms) and accumulators per lane
    static constexpr int DIM = AtomShape<AT>::DIM, NACC = AtomShape<AT>::NACC;
    static constexpr int IM = TM / DIM, JN = TN / DIM;
    static constexpr int NS = BK / KS;
    static constexpr int KSW = KS / PK;
    static constexpr int KSTEPS = KSW / AT::KSTEP;
    static constexpr int ELT = (int)sizeof(typename AT::in_t);
    static constexpr int VE = 16 / ELT;  // elements per 16-byte staging chunk
    static constexpr bool A_PRIV = (PN == 1);
    static constexpr int NBUF = (NS == 1) ? 1 : 2;
    // FP64 over several stages: the bound of a piece that is always within it is left out, since
    // the loads and writes of a stage are otherwise a branch each (3D 128^3 x 1024 115 us with
    // the branches, 102 without; a single stage is faster with them, 64^3 in 1D 26.2, 27.6)
    static constexpr bool WHOLE = ELT == 8 && NS > 1;
    static constexpr int ROWB = lds_row_bytes(KS * ELT, AT::FRAG_BYTES);  // conflict-free reads
    static constexpr int A_LDS = A_PRIV ? 0 : BM * ROWB;
    // K x N: bytes between staged K rows, and the extra bytes after every eight of 2-byte
    // values.  FP64 reads 8 bytes a lane, 16 columns of rows 2 g + e by lane group g: a row of
    // 64 mod 128 bytes puts two groups on different banks.  2-byte values are read by
    // transposing reads, four rows of 32 bytes by lane group g: rows 32 mod 64 bytes apart, and
    // the groups' rows half the banks apart.
    static constexpr int KROW = BN * ELT + (ELT == 8 ? 64 : BN * ELT % 64 == 0 ? 32 : 0);
    static constexpr int KGAP = ELT == 8 ? 0 : 128;
    static constexpr int B_LDS = KN ? KS * KROW + KS / 8 * KGAP : BN * ROWB;
    __device__ static constexpr int krow(int k) { return k * KROW + (k >> 3) * KGAP; }
    static constexpr int STAGE_LDS = A_LDS + B_LDS;
    static constexpr int STAGING = NBUF * STAGE_LDS;
    static constexpr int ACC_ELT = (int)sizeof(typename AT::acc_t);
    static constexpr int RED_ROW_BYTES = PK * PM * PN * JN * NACC * 64 * ACC_ELT;
    static constexpr int RED_ROWS = (PK > 1) ? cmin(IM, cmax(1, STAGING / RED_ROW_BYTES)) : 1;
    static constexpr int RED_ROUNDS = (IM + RED_ROWS - 1) / RED_ROWS;
    static constexpr int RED_LDS = (PK > 1) ? RED_ROWS * RED_ROW_BYTES : 0;
    static constexpr int LDS = cmax(STAGING, RED_LDS);
    static constexpr int CA = A_PRIV ? 0 : BM * KS / VE;  // 16-byte chunks of an A stage
    static constexpr int CB = BN * KS / VE;               // 16-byte chunks of a B stage
    static constexpr int NA = (CA + NT - 1) / NT;
    static constexpr int NBC = (CB + NT - 1) / NT;

    static_assert(BM % PM == 0 && BN % PN == 0 && BK % KS == 0 && KS % PK == 0, "tiling");
    static_assert(TM % DIM == 0 && TN % DIM == 0, "wave tile must be a multiple of the atom");
    static_assert(KSW % AT::KSTEP == 0, "wave K slice must be a multiple of the atom K step");
    static_assert((KS * ELT) % 16 == 0 && (BN * ELT) % 16 == 0, "16-byte staging");
    static_assert(NT <= 1024, "workgroup too large");
    static_assert(LDS <= 160 * 1024, "LDS budget of one workgroup");
};

struct BlockArgs {
    const void* A;
    const void* B;
    void* C;
    int64_t sa, sb, sc;       // per-problem strides (elements)
    int64_t lda, ldb, ldc;    // leading dimensions (elements)
    double alpha, beta;
    int32_t iters;
    int32_t b_kn;             // 1: B stored K x N (the launcher picks the kernel)
};

// B fragment of column atom jn at K step ks of the K slice of wave (pn, pk), from the stage at
// bb; kk is the lane's byte offset in a row of K.  The address is formed as the fragments of A
// are: with the row's part first, the 256^3 resident forms keep an address per fragment and
// spill 60 registers (FP16 x 1024, 8 times, 596 us against 246).  K x N rows: a lane's values
// are AT::KV rows of one column.  K step 8: the upper lane groups' values are not used, and they
// read the lower groups' rows so as to stay in the stage.
template <class AT, class G>
__device__ __forceinline__ typename AT::frag_t stage_b_fragment(const unsigned char* bb, int lane, int pn,
                                                                int pk, int jn, int ks, int kk) {
    using frag_t = typename AT::frag_t;
    if constexpr (!G::KN) {
        return bitcast<frag_t>(load_raw<AT::FRAG_BYTES>(
            bb + (pn * G::TN + jn * G::DIM + (lane % G::DIM)) * G::ROWB + kk));
    } else {
        const int col = pn * G::TN + lane % G::DIM, grp = lane / G::DIM;
        constexpr int GROUPS = cmin(64 / G::DIM, AT::KSTEP / AT::KV);
        const unsigned char* q = bb + G::krow(pk * G::KSW + AT::KV * (grp % GROUPS));
        const int step = G::krow(ks * AT::KSTEP) + jn * G::DIM * G::ELT;
        if constexpr (G::ELT == 8) {
            q += col * 8 + step;
            return frag_t{*reinterpret_cast<const double*>(q), *reinterpret_cast<const double*>(q + G::KROW)};
        } else {
            const int l = lane & 15;
            q += (l >> 2) * G::KROW + (col - l) * 2 + 8 * (l & 3) + step;
            const u2_t lo = lds_read_turned(q);
            if constexpr (AT::KV == 4) {
                return bitcast<frag_t>(lo);
            } else {
                const u2_t hi = lds_read_turned(q + 4 * G::KROW);
                return bitcast<frag_t>(u4_t{lo[0], lo[1], hi[0], hi[1]});
            }
        }
    }
}

// Waves a SIMD is to hold, at most, where a call moves more than the caches hold.  1D instances
// of 2-byte values write more than they read, and with fewer problems in flight and the registers
// spent on longer runs of loads the writes to memory go faster: operands not in the caches, 64 x
// 64 x 32 x 4096 with 4 waves 23.2 us uncapped, 20.0 with 3 a SIMD; 128 x 128 x 16 x 2048 with 8
// 35.4, 30.8; 64^3 x 4096 25.8, 24.8; 128 x 128 x 32 x 4096 with 4 (K x N) 72.8, 64.1.  8: no
// such form.  Smaller problems want all the waves they can have (16^3 4.2 us, 4.5 with 3), and so
// do the 2D instances (BF16 64^3 51 us, 58).
template <class AT, class G>
constexpr int waves_per_simd() {
    if (G::ELT == 8 || G::PN > 1 || G::PK > 1 || G::BM < 64 || G::TURNED) return 8;
    const int want = G::IM * G::JN * G::NACC >= 128 ? 2 : 3, own = (G::WAVES + 3) / 4;
    return (want + own - 1) / own * own;  // whole workgroups
}
// Below that the writes stay in the caches and every wave helps (64 x 64 x 16 x 2048 with 4 waves
// 9.3 us, capped 11.1; 128 x 128 x 16 x 1024 14.0, 15.1; 84 MB of 64 x 64 x 16 16.6, 17.6, but 100
// MB of 64 x 64 x 32 24.2, 21.3, and 84 MB of 128 x 128 x 32 with eight waves 20.6, 18.8).  From
// many repetitions on the products bound it: their fragments want the registers whatever the size
// (64^3 x 2048, 32 times, 29.4 us, capped 24.5), as long as two workgroups fit a CU (192 x 192 x 16
// x 8192 with 12 waves, 32 times, 324 us, 412 capped to one).  Where LDS holds no second workgroup
// anyway the cap takes no waves away.
constexpr int64_t cap_bytes(int waves) { return waves >= 8 ? 80000000 : 100000000; }
constexpr int kCapIters = 8;
template <class AT, class G>
bool cap_pays(int64_t bytes, int iters) {
    if (2 * G::LDS > 160 * 1024) return true;
    return iters > kCapIters ? waves_per_simd<AT, G>() >= 2 * ((G::WAVES + 3) / 4) : bytes >= cap_bytes(G::WAVES);
}

// KFENCE > 0: a scheduling fence after every KFENCE K steps of a stage, so the
// compiler does not hoist the B fragment loads of a whole long stage ahead of the MFMAs
// (used by the resident forms, whose single stage covers all of K).  With 2 the wave's rows of A
// are loaded once B's have arrived: the address unit takes their fragments four lanes a
// clock, and B, which every wave waits for, would queue behind them (256^3 x 1024, twice,
// 119 us against 127; 192^3 x 2048 113 against 116).
//
// SP > 1: the wave tiles of the full BN columns do not fit the register file, so the
// problem's columns are computed in SP passes of G::BN = BN / SP columns each (B rows and
// C columns of pass sp start at sp * G::BN); A is read again in every pass.
// MOST: waves a SIMD holds, at most (waves_per_simd).
template <class AT, class G, int KFENCE = 0, int SP = 1, int MOST = 8>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu((G::WAVES + 3) / 4, MOST)))
block_gemm_kernel(BlockArgs args) {
    using in_t = typename AT::in_t;
    using acc_t = typename AT::acc_t;
    using out_t = typename AT::out_t;
    using frag_t = typename AT::frag_t;
    using accv_t = typename AT::accv_t;
    constexpr int FB = AT::FRAG_BYTES;

    __shared__ __attribute__((aligned(16))) unsigned char smem[G::LDS];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    // wave grid coordinates: depth fastest, then column, then row
    const int pk = wave % G::PK;
    const int pn = (wave / G::PK) % G::PN;
    const int pm = wave / (G::PK * G::PN);

    const int64_t prob = blockIdx.x;
    const int64_t lda = args.lda, ldb = args.ldb, ldc = args.ldc;
    const in_t* __restrict__ A = reinterpret_cast<const in_t*>(args.A) + prob * args.sa;
#pragma unroll 1
    for (int sp = 0; sp < SP; ++sp) {
    if (sp > 0) __syncthreads();  // the previous pass is done with LDS
    const in_t* __restrict__ B = reinterpret_cast<const in_t*>(args.B) + prob * args.sb +
                                 (int64_t)sp * G::BN * (G::SRC_KN ? 1 : ldb);
    out_t* __restrict__ C = reinterpret_cast<out_t*>(args.C) + prob * args.sc + sp * G::BN;

    accv_t acc[G::IM][G::JN];
#pragma unroll
    for (int i = 0; i < G::IM; ++i)
#pragma unroll
        for (int j = 0; j < G::JN; ++j)
#pragma unroll
            for (int v = 0; v < G::NACC; ++v) acc[i][j][v] = 0;

    // ---- staging of the shared operands (global -> registers -> LDS) ----
    u4_t stA[G::NA > 0 ? G::NA : 1];
    u4_t stB[G::NBC];
    auto load_stage = [&](int s) {
        const int k0 = s * G::KS;
        if constexpr (!G::A_PRIV) {
            constexpr int CPR = G::KS / G::VE;
#pragma unroll
            for (int i = 0; i < G::NA; ++i) {
                const int c = tid + i * G::NT;
                if ((G::WHOLE && G::CA % G::NT == 0) || c < G::CA) {
                    const int r = c / CPR, cc = c % CPR;
                    stA[i] = load_raw<16>(A + r * lda + k0 + cc * G::VE);
                }
            }
        }
        if constexpr (!G::SRC_KN) {
            constexpr int CPR = G::KS / G::VE;
#pragma unroll
            for (int i = 0; i < G::NBC; ++i) {
                const int c = tid + i * G::NT;
                if ((G::WHOLE && G::CB % G::NT == 0) || c < G::CB) {
                    const int r = c / CPR, cc = c % CPR;
                    stB[i] = load_raw<16>(B + r * ldb + k0 + cc * G::VE);
                }
            }
        } else {
            constexpr int CPR = G::BN / G::VE;
#pragma unroll
            for (int i = 0; i < G::NBC; ++i) {
                const int c = tid + i * G::NT;
                if ((G::WHOLE && G::CB % G::NT == 0) || c < G::CB) {
                    const int kr = c / CPR, jc = c % CPR;
                    stB[i] = load_raw<16>(B + (int64_t)(k0 + kr) * ldb + jc * G::VE);
                }
            }
        }
    };
    auto write_stage = [&](int buf) {
        unsigned char* base = smem + buf * G::STAGE_LDS;
        if constexpr (!G::A_PRIV) {
            constexpr int CPR = G::KS / G::VE;
#pragma unroll
            for (int i = 0; i < G::NA; ++i) {
                const int c = tid + i * G::NT;
                if ((G::WHOLE && G::CA % G::NT == 0) || c < G::CA) {
                    const int r = c / CPR, cc = c % CPR;
                    store_raw<16>(base + r * G::ROWB + cc * 16, stA[i]);
                }
            }
        }
        unsigned char* bb = base + G::A_LDS;
        constexpr int CPR = (G::SRC_KN ? G::BN : G::KS) / G::VE;
#pragma unroll
        for (int i = 0; i < G::NBC; ++i) {
            const int c = tid + i * G::NT;
            if ((G::WHOLE && G::CB % G::NT == 0) || c < G::CB) {
                const int r = c / CPR, cc = c % CPR;
                if constexpr (G::TURNED) {
                    const in_t* e = reinterpret_cast<const in_t*>(&stB[i]);
#pragma unroll
                    for (int q = 0; q < G::VE; ++q)
                        *reinterpret_cast<in_t*>(bb + (cc * G::VE + q) * G::ROWB + r * G::ELT) = e[q];
                } else {
                    store_raw<16>(bb + (G::KN ? G::krow(r) : r * G::ROWB) + cc * 16, stB[i]);
                }
            }
        }
    };

    // ---- register-resident A (1D): each wave loads its own rows in fragment layout ----
    constexpr int AIM = G::A_PRIV ? G::IM : 1;
    constexpr int AKS = G::A_PRIV ? G::KSTEPS : 1;
    frag_t a_cur[AIM][AKS];
    frag_t a_nxt[(G::A_PRIV && G::NS > 1) ? AIM : 1][(G::A_PRIV && G::NS > 1) ? AKS : 1];
    auto load_a = [&](int s, frag_t (&dst)[AIM][AKS]) {
        if constexpr (G::A_PRIV) {
            const int kb = s * G::KS + pk * G::KSW + AT::KV * (lane / G::DIM);
#pragma unroll
            for (int im = 0; im < G::IM; ++im) {
                const in_t* row = A + (int64_t)(pm * G::TM + im * G::DIM + (lane % G::DIM)) * lda + kb;
#pragma unroll
                for (int ks = 0; ks < G::KSTEPS; ++ks)
                    dst[im][ks] = bitcast<frag_t>(load_raw<FB>(row + ks * AT::KSTEP));
            }
        }
    };

    auto compute = [&](int buf) {
        const unsigned char* base = smem + buf * G::STAGE_LDS;
        const unsigned char* bb = base + G::A_LDS;
        const int kin = pk * G::KSW + AT::KV * (lane / G::DIM);
#pragma unroll
        for (int ks = 0; ks < G::KSTEPS; ++ks) {
            const int kk = (kin + ks * AT::KSTEP) * G::ELT;
            // A fragments of this K step stay live; B fragments are streamed one column
            // atom at a time so the accumulators keep most of the register file.
            frag_t af[G::IM];
#pragma unroll
            for (int im = 0; im < G::IM; ++im) {
                if constexpr (G::A_PRIV) {
                    af[im] = a_cur[im][ks];
                } else {
                    af[im] = bitcast<frag_t>(
                        load_raw<FB>(base + (pm * G::TM + im * G::DIM + (lane % G::DIM)) * G::ROWB + kk));
                }
            }
            if constexpr (AT::NSUB == 1) {
#pragma unroll
                for (int jn = 0; jn < G::JN; ++jn) {
                    const frag_t bf = stage_b_fragment<AT, G>(bb, lane, pn, pk, jn, ks, kk);
#pragma unroll
                    for (int im = 0; im < G::IM; ++im) AT::mma(acc[im][jn], af[im], bf);
                }
            } else {
                // several instructions per fragment: issue sub-step e for every atom
                // before sub-step e + 1 so consecutive MFMAs never share an accumulator
                frag_t bf[G::JN];
#pragma unroll
                for (int jn = 0; jn < G::JN; ++jn)
                    bf[jn] = stage_b_fragment<AT, G>(bb, lane, pn, pk, jn, ks, kk);
#pragma unroll
                for (int e = 0; e < AT::NSUB; ++e)
#pragma unroll
                    for (int jn = 0; jn < G::JN; ++jn)
#pragma unroll
                        for (int im = 0; im < G::IM; ++im) AT::mma_sub(acc[im][jn], af[im], bf[jn], e);
            }
            if constexpr (KFENCE > 0)
                if ((ks + 1) % KFENCE == 0) __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- main loop ----
    constexpr bool A_LATE = KFENCE == 2;
    load_stage(0);
    if constexpr (!A_LATE) load_a(0, a_cur);
    // the arguments that products and stores need, while the loads are on their way: fetched where
    // they are used they are waited for behind those (128 x 128 x 32 x 512 in four waves 8.1 us,
    // 7.9; 192 x 192 x 16 x 64 in 2D 0.96 of the time).  Smaller tiles on wave grids lose by it
    // (32^3 in 2 x 2 waves, 1000 times, 1.07), FP64 neither way.
    if constexpr (G::ELT == 2 && (G::PN == 1 ? G::BM >= 64 : G::BM >= 192))
        asm volatile("" ::"s"(args.iters), "s"(args.alpha), "s"(args.beta));
    write_stage(0);
    __syncthreads();
    if constexpr (A_LATE) load_a(0, a_cur);
    if constexpr (G::NS == 1) {
        for (int it = 0; it < args.iters; ++it) compute(0);
    } else {
        int g = 0;
        for (int it = 0; it < args.iters; ++it) {
#pragma unroll 1
            for (int s = 0; s < G::NS; ++s, ++g) {
                const bool has_next = (s + 1 < G::NS) || (it + 1 < args.iters);
                const int sn = (s + 1 == G::NS) ? 0 : s + 1;
                if (has_next) {
                    load_stage(sn);
                    if constexpr (G::A_PRIV) load_a(sn, a_nxt);
                }
                compute(g & 1);
                if (has_next) {
                    write_stage((g & 1) ^ 1);
                    if constexpr (G::A_PRIV) {
#pragma unroll
                        for (int im = 0; im < AIM; ++im)
#pragma unroll
                            for (int ks = 0; ks < AKS; ++ks) a_cur[im][ks] = a_nxt[im][ks];
                    }
                }
                __syncthreads();
            }
        }
    }

    // ---- 3D: reduce the PK partial tiles through LDS; atom (im, jn) is finalised by
    //      depth (im * JN + jn) % PK, summing depths in ascending order ----
    if constexpr (G::PK > 1) {
        acc_t* red = reinterpret_cast<acc_t*>(smem);
#pragma unroll
        for (int r = 0; r < G::RED_ROUNDS; ++r) {
            __syncthreads();
#pragma unroll
            for (int im = r * G::RED_ROWS; im < cmin((r + 1) * G::RED_ROWS, G::IM); ++im)
#pragma unroll
                for (int jn = 0; jn < G::JN; ++jn) {
                    if ((im * G::JN + jn) % G::PK != pk) {
                        const int slot =
                            (((pk * G::PM + pm) * G::PN + pn) * G::RED_ROWS + (im - r * G::RED_ROWS)) *
                                G::JN + jn;
#pragma unroll
                        for (int v = 0; v < G::NACC; ++v)
                            red[slot * (G::NACC * 64) + v * 64 + lane] = acc[im][jn][v];
                    }
                }
            __syncthreads();
#pragma unroll
            for (int im = r * G::RED_ROWS; im < cmin((r + 1) * G::RED_ROWS, G::IM); ++im)
#pragma unroll
                for (int jn = 0; jn < G::JN; ++jn) {
                    if ((im * G::JN + jn) % G::PK == pk) {
                        accv_t tot;
#pragma unroll
                        for (int q = 0; q < G::PK; ++q) {
                            accv_t x;
                            if (q == pk) {
                                x = acc[im][jn];
                            } else {
                                const int slot =
                                    (((q * G::PM + pm) * G::PN + pn) * G::RED_ROWS +
                                     (im - r * G::RED_ROWS)) * G::JN + jn;
#pragma unroll
                                for (int v = 0; v < G::NACC; ++v)
                                    x[v] = red[slot * (G::NACC * 64) + v * 64 + lane];
                            }
                            if (q == 0) tot = x; else tot += x;
                        }
                        acc[im][jn] = tot;
                    }
                }
        }
    }

    // ---- epilogue: C = alpha * acc + beta * C ----
    const acc_t alpha = (acc_t)args.alpha;
    const acc_t beta = (acc_t)args.beta;
#pragma unroll
    for (int im = 0; im < G::IM; ++im)
#pragma unroll
        for (int jn = 0; jn < G::JN; ++jn) {
            if (G::PK > 1 && (im * G::JN + jn) % G::PK != pk) continue;
            const int col = pn * G::TN + jn * G::DIM + (lane % G::DIM);
#pragma unroll
            for (int v = 0; v < G::NACC; ++v) {
                const int row = pm * G::TM + im * G::DIM + AT::out_row(lane, v);
                out_t* dst = C + (int64_t)row * ldc + col;
                acc_t val = alpha * acc[im][jn][v];
                if (beta != (acc_t)0) val += beta * (acc_t)(*dst);
                *dst = (out_t)val;
            }
        }
    }  // column passes
}

template <class AT, class G, int KFENCE, int SP, int MOST = 8>
hipError_t launch_block_gemm_as(const BlockArgs& args, int64_t count, hipStream_t stream) {
    if constexpr (MOST == 8 && KFENCE < 2 && waves_per_simd<AT, G>() < 8) {  // (resident forms repeat)
        constexpr int64_t problem = (int64_t)(G::BM + G::BN * SP) * G::BK * G::ELT + (int64_t)G::BM * G::BN * SP * 4;
        if (cap_pays<AT, G>(count * problem, args.iters))
            return launch_block_gemm_as<AT, G, KFENCE, SP, waves_per_simd<AT, G>()>(args, count, stream);
    }
    hipLaunchKernelGGL((block_gemm_kernel<AT, G, KFENCE, SP, MOST>), dim3((unsigned)count), dim3(G::NT), 0, stream,
                       args);
    return hipGetLastError();
}

// Repetitions from which 2-byte K x N rows in one stage are turned in the writes, once, and not
// in the reads, every time; the conflicting writes cost more the more columns there are (turned in
// the writes against the reads, 4096 problems: 64^3 8 times 28.1 us, 26.8, 16 times 35.1, 36.5;
// 128^3 8 times 125, 110, 16 times 172, 195, 32 times 313, 358; 256 x 256 x 32 16 times 302, 265,
// x 1024 128 times 321, 343).  Several stages are written again for every repetition and stay
// rows (128 x 128 x 512 x 256, 64 times, 0.41 of the time with turned writes).
constexpr int turn_iters(int columns) { return columns / 8; }

template <class AT, class G, int KFENCE = 0, int SP = 1>
hipError_t launch_block_gemm(const BlockArgs& args, int64_t count, hipStream_t stream) {
    // FP64 in one stage on a wave grid: a fragment's two rows are two reads, by every wave row, which
    // costs more than the conflicting writes once the CUs hold several problems of 64 columns (2D
    // 64^3 x 1024 23.8 us turned in the writes, 25.8 in the reads, x 64 5.2, 4.8; 32^3 x 1024 4.9,
    // 4.5; 1D, where a wave reads all of B either way, 64^3 x 1024 29.2 and 26.3)
    constexpr bool grid64 = G::ELT == 8 && G::PN > 1 && G::BN >= 64;
    if constexpr (G::NS == 1 && (G::ELT == 2 || grid64))
        if (args.b_kn && (grid64 ? count > 512 : args.iters >= turn_iters(G::BN * SP)))
            return launch_block_gemm_as<AT, typename G::AsTurned, KFENCE, SP>(args, count, stream);
    if (args.b_kn) return launch_block_gemm_as<AT, typename G::AsKN, KFENCE, SP>(args, count, stream);
    return launch_block_gemm_as<AT, G, KFENCE, SP>(args, count, stream);
}

// A resident form, which is taken for repeated products only (2-byte K x N: three or more), and
// turns in the writes for any: with rows in LDS the instances of 16 waves and FP64's spill.
template <class AT, class G>
hipError_t launch_resident(const BlockArgs& args, int64_t count, hipStream_t stream) {
    if (args.b_kn) return launch_block_gemm_as<AT, typename G::AsTurned, 2, 1>(args, count, stream);
    return launch_block_gemm_as<AT, G, 2, 1>(args, count, stream);
}

}  // namespace kami
