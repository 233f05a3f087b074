// Batched GEMM over problems of uneven size: one launch over a device queue of wave tiles,
// per-size-bucket tile variants chosen by an autotuner.
//
// Reference: batched_gemm_{1d,2d,3d}_double_mma (src/batched_gemm/KAMI/1d/
// batched_gemm_1d_double_mma.cu:59-218) runs one uniform-size problem per CTA at fixed
// strides (:71-74) with the partition picked per size by the sweep script
// (scripts/fp64_batched_GH200.sh:96-123).  Here:
//   * problems carry their own {m, n, k, lda, ldb, ldc, A, B, C} (the kami_problem array);
//   * every problem is cut into output tiles; a tile is one 64-byte queue entry holding
//     its own operand pointers, strides, extents and variant (WorkItem);
//   * an entry is cut into wave tiles of up to 64 x 32 (2-byte inputs: 64 x 64; WaveUnit, 8
//     bytes each).  A wave computes one of them alone, staged through LDS of its own, so there is no barrier
//     and no shared counter: the hardware's dispatcher hands out the workgroups, longest
//     problems first, and one wave's loads hide behind the products of the others;
//   * units are laid out so that neighbouring tiles run on one XCD at the same time;
//   * the variant of a tile is the tile shape and wave partition of its size bucket,
//     picked by timing candidates on the device at plan creation (or from priors);
//   * one execution is one kernel launch, also for plans made with use_graph: replaying a
//     captured graph of that one kernel took 18.5 us of a caller's loop where the launch
//     takes 8.9 us (100 FP64 problems of 16 to 256).
// M, N and K must be multiples of 16.
//
// What bounds it: 20000 problems of 16 to 256 (3.58 GB FP64, 1.19 GB FP16 with FP32 C) run
// in 788 us and 275 us, 4.5 and 4.3 TB/s of the algorithmic bytes; FP64 moves 3.97 GB, at the rate
// of a copy (5 TB/s).
// The persistent form this replaced (workgroups popping tiles of up to 128 x 128 from an atomic
// counter, LDS stages shared by four waves, one barrier a stage, a one-thread kernel to clear
// the counter) took 1027 us and 398 us: two workgroups a CU and their barriers left too little
// in flight.
#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <vector>

#include "kami_internal.hpp"

namespace kami {

// One queue entry = one output tile, carrying everything its loads and stores need, so
// the kernel never goes back to the problem table.
struct WorkItem {
    const void* A;  // first element of the tile's rows of A
    const void* B;  // first element of the tile's rows of B (n x K) or columns (K x n)
    void* C;        // first element of the tile in C
    int64_t lda, ldb, ldc;
    int32_t mlim, nlim;  // rows / columns of C from the tile origin to the problem edge
    int32_t k, variant;
};
static_assert(sizeof(WorkItem) == 64, "queue entry layout");

// Consecutive queue entries dealt to one XCD at a time: a power of two up to
// 1 << kQueueShift.
constexpr int kQueueShift = 3;

// Tile variants.  Index = variant id stored in the work items.
//   0: 64 x 64 tile      1: 32 x 32 tile      2: 64 x 64 tile, wave tiles of 16 x 32
//   3: 128 x 64 tile     4: 128 x 128 tile (FP64)     5: 64 x 128 tile (FP64)
// Wave tiles are as large as kCapM and kCapN allow except where noted.
constexpr int kVariants = 6;
static_assert(kVariants == kBatchedVariants, "tuning-cache variant range");
static const int kVariantTM[kVariants] = {64, 32, 64, 128, 128, 64};
static const int kVariantTN[kVariants] = {64, 32, 64, 64, 128, 128};
static const int kVariantSM[kVariants] = {4, 4, 1, 4, 4, 4};  // atoms of a wave tile, at most
static const int kVariantSN[kVariants] = {4, 4, 2, 4, 4, 4};

// Variants a precision offers: 4 and 5 are FP64's.
inline int variants_of(int prec) { return prec == KAMI_PREC_F64 ? kVariants : 4; }

// One wave's share of a queue entry: the im x jn atoms (16 x 16) of C whose first atom is
// (ra, ca), counted in atoms from the entry's origin.  im = 0: nothing to do.
struct WaveUnit {
    uint32_t item;
    uint8_t ra, ca, im, jn;
};
static_assert(sizeof(WaveUnit) == 8, "wave unit layout");
// Wave tiles in atoms, largest first.  A larger tile reads A's and B's lines less often, and
// fewer of its waves fit a SIMD.  A precision starts at first_cap or, where larger_pays, at the
// one before: 2-byte inputs at 64 x 32 or 64 x 64 (256^3 x 1024 141 us, 115; 320^3 x 1024 280, 227;
// 20000 problems of 16 to 256 291, 276, and 304 with 32 x 32; 20000 of 16 to 64 21.7, 23.8), FP64
// at 32 x 32 or 64 x 32 (20000 of 16 to 256 807, 788; 128^3 x 4096 387, 372; 256^3 x 1024 636, 609;
// 64^3 x 8192 148, 155; with 64 x 64 169 there and 614 at 256^3).
constexpr int kCaps = 5;
static const int kCapM[kCaps] = {4, 4, 2, 1, 1}, kCapN[kCaps] = {4, 2, 2, 2, 1};
constexpr int first_cap(int elt) { return elt == 8 ? 2 : 1; }
constexpr int kWavesPerGroup = 4;
constexpr int kXcds = 8;  // workgroup L runs on XCD L mod 8

// Where the unit of wave w of workgroup L of `groups` lies
__host__ __device__ inline int64_t unit_at(int64_t L, int64_t groups, int w) {
    return (L % kXcds * (groups / kXcds) + L / kXcds) * kWavesPerGroup + w;
}

struct BatchArgs {
    const WorkItem* items;
    const WaveUnit* units;
    int64_t n_units;  // a multiple of kWavesPerGroup x kXcds
    double alpha, beta;
    int cap;  // the largest wave tile is kCapM[cap] x kCapN[cap] atoms
};

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Raw buffer descriptors over a wave tile's operands.  A lane offset at or past
// kBufferRange reads as zero, so pieces past K need no branch.
constexpr int kBufferRange = 0x7FFFFFF0;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, kBufferRange,
                                             0x00020000);
}
__device__ __forceinline__ u4_t buffer_load16(__amdgpu_buffer_rsrc_t r, int off, int soff) {
    return __builtin_bit_cast(u4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0));
}
__device__ __forceinline__ double buffer_load8(__amdgpu_buffer_rsrc_t r, int off, int soff) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0));
}

#define KAMI_GLOBAL __attribute__((address_space(1)))

// A wave tile of IM x JN atoms computed by one wave on its own: no barrier, so the waves of a
// CU run apart and one wave's loads hide behind the others' products.  A stage is one
// 128-byte line of every row of the tile (16 FP64 or 64 FP16 / BF16 values of K, two
// fragments).  Loading fragments straight from memory would put 16 rows under 16
// consecutive lanes, which the address unit takes 4 lanes a clock (64 clocks an
// instruction); so eight lanes load a row's line (16 clocks) and the lines are turned into
// fragments through LDS of the wave's own.
template <class AT, bool KN, int IM, int JN>
struct WaveTile {
    using frag_t = typename AT::frag_t;
    using acc_t = typename AT::acc_t;
    using out_t = typename AT::out_t;
    using accv_t = typename AT::accv_t;
    static constexpr int ELT = (int)sizeof(typename AT::in_t);
    static constexpr bool F64 = ELT == 8;
    static constexpr int VE = 16 / ELT;
    static constexpr int KS = 128 / ELT, NF = KS / AT::KSTEP;
    static_assert(NF == 2 && AT::FRAG_BYTES == 16, "a stage row is two 64-byte fragment groups");
    // K x N operands: FP64 fragments are loaded straight (16 lanes read 16 consecutive
    // columns); rows of 2-byte values are turned by transposing LDS reads
    static constexpr bool TURN = KN && !F64;
    static constexpr int PPR = JN == 3 ? 8 : JN * 2;  // lanes of a K row, a 16-byte piece each
    static constexpr int TROW = PPR * 16 + 16;        // bytes of a staged K row
    static constexpr int NA = IM * 2, NB = TURN ? PPR : JN * 2;  // 16-byte pieces of a lane
    static_assert(!TURN || KS == 64, "NB loads of 64 / PPR rows are a stage");
    static constexpr int A_LDS = IM * 16 * 128;
    static constexpr int LDS = A_LDS + (!KN ? JN * 16 * 128 : TURN ? KS * TROW : 0);

    struct Stage {
        u4_t a[NA], b[NB];
    };

    const __amdgpu_buffer_rsrc_t ra, rb;
    const int lane, grp, lda, ldb, k;
    unsigned char* const lds;
    int aoff, boff;  // the lane's byte offsets in the first stage
    // LDS offsets.  Piece p of row r lies in slot p ^ 2 ((r / 4) mod 4) of the row's eight, so
    // that the 32 lanes of a read pass (16 rows, two neighbouring pieces) and the rows of a
    // write fall on different banks.
    int woff, roff;

    __device__ __forceinline__ WaveTile(const WorkItem& w, const WaveUnit& u, unsigned char* lds_)
        : ra(tile_rsrc(static_cast<const char*>(w.A) + (int64_t)u.ra * 16 * w.lda * ELT)),
          rb(tile_rsrc(static_cast<const char*>(w.B) + (int64_t)u.ca * 16 * (KN ? 1 : w.ldb) * ELT)),
          lane(threadIdx.x & 63), grp(lane >> 4), lda((int)w.lda), ldb((int)w.ldb), k(w.k), lds(lds_) {
        aoff = ((lane >> 3) * lda + (lane & 7) * VE) * ELT;
        if constexpr (!KN)
            boff = ((lane >> 3) * ldb + (lane & 7) * VE) * ELT;
        else if constexpr (F64)
            boff = (2 * grp * ldb + (lane & 15)) * ELT;  // sub-step e takes row k = 2 grp + e
        else
            boff = (lane / PPR * ldb + (lane % PPR) * 8) * ELT;
        woff = (lane >> 3) * 128 + (((lane & 7) ^ ((lane >> 5) << 1)) << 4);
        roff = (lane & 15) * 128 + ((grp ^ (((lane >> 2) & 3) << 1)) << 4);
    }

    // Stage c of K's (k + KS - 1) / KS.  (FP64 stages never pass K, a multiple of 16: with its
    // two comparisons left out 256^3 x 100, K x N, took 73.7 us instead of 68.5.)
    __device__ __forceinline__ void load(Stage& s, int c) const {
        // pieces past K lie out of the descriptor's range; the scalar offsets stay inside
        // the operand
        const int k0 = c * KS, kb = k0 < k ? k0 : 0;
        const bool ok = F64 ? k0 < k : k0 + (lane & 7) * VE < k;
        const int ao = ok ? aoff : kBufferRange, bo = ok ? boff : kBufferRange;
#pragma unroll
        for (int i = 0; i < NA; ++i) s.a[i] = buffer_load16(ra, ao, (i * 8 * lda + kb) * ELT);
        if constexpr (!KN) {
#pragma unroll
            for (int j = 0; j < NB; ++j) s.b[j] = buffer_load16(rb, bo, (j * 8 * ldb + kb) * ELT);
        } else if constexpr (F64) {
#pragma unroll
            for (int t = 0; t < NF; ++t)
#pragma unroll
                for (int j = 0; j < JN; ++j) {
                    const int so = ((kb + t * AT::KSTEP) * ldb + j * 16) * ELT;
                    const d2_t x = {buffer_load8(rb, bo, so), buffer_load8(rb, bo, so + ldb * ELT)};
                    s.b[j * NF + t] = bitcast<u4_t>(x);
                }
        } else {
            constexpr int RPL = 64 / PPR;  // K rows of one load instruction
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int r = k0 + i * RPL;
                const bool live = r + lane / PPR < k && (JN != 3 || lane % PPR < 2 * JN);
                s.b[i] = buffer_load16(rb, live ? boff : kBufferRange,
                                       (r < k ? r : 0) * ldb * ELT);
            }
        }
    }

    // Stage registers to LDS (a wave's LDS accesses complete in order: no wait between the
    // reads of one stage and the writes of the next)
    __device__ __forceinline__ void write(const Stage& s) const {
#pragma unroll
        for (int i = 0; i < NA; ++i) store_raw<16>(lds + (woff ^ ((i & 1) * 64)) + i * 1024, s.a[i]);
        if constexpr (!KN) {
#pragma unroll
            for (int j = 0; j < NB; ++j)
                store_raw<16>(lds + A_LDS + (woff ^ ((j & 1) * 64)) + j * 1024, s.b[j]);
        } else if constexpr (TURN) {
#pragma unroll
            for (int i = 0; i < NB; ++i)
                store_raw<16>(lds + A_LDS + (i * (64 / PPR) + lane / PPR) * TROW + (lane % PPR) * 16, s.b[i]);
        }
    }

    // FP64 K x N: B's fragments as loaded, kept while the stage's registers are loaded again
    struct Held {
        u4_t b[KN && F64 ? NB : 1];
        __device__ __forceinline__ explicit Held(const Stage& s) {
            if constexpr (KN && F64)
#pragma unroll
                for (int j = 0; j < NB; ++j) b[j] = s.b[j];
        }
    };

    // Products of the stage in LDS, one fragment (half a line) at a time
    __device__ __forceinline__ void mma(const Held& held, accv_t (&acc)[IM][JN]) const {
#pragma unroll
        for (int t = 0; t < NF; ++t) {
            frag_t a[IM], b[JN];
#pragma unroll
            for (int i = 0; i < IM; ++i)
                a[i] = bitcast<frag_t>(load_raw<16>(lds + (roff ^ (t * 64)) + i * 2048));
            if constexpr (TURN) {
                const unsigned char* p = lds + A_LDS + (8 * grp + ((lane & 15) >> 2)) * TROW + 8 * (lane & 3);
#pragma unroll
                for (int j = 0; j < JN; ++j) {
                    const u2_t lo = lds_read_turned(p + t * 32 * TROW + j * 32);
                    const u2_t hi = lds_read_turned(p + (t * 32 + 4) * TROW + j * 32);
                    b[j] = bitcast<frag_t>(u4_t{lo[0], lo[1], hi[0], hi[1]});
                }
            } else {
#pragma unroll
                for (int j = 0; j < JN; ++j) {
                    if constexpr (KN)
                        b[j] = bitcast<frag_t>(held.b[j * NF + t]);
                    else
                        b[j] = bitcast<frag_t>(load_raw<16>(lds + A_LDS + (roff ^ (t * 64)) + j * 2048));
                }
            }
#pragma unroll
            for (int e = 0; e < AT::NSUB; ++e)
#pragma unroll
                for (int j = 0; j < JN; ++j)
#pragma unroll
                    for (int i = 0; i < IM; ++i) AT::mma_sub(acc[i][j], a[i], b[j], e);
        }
    }

    __device__ __forceinline__ void run(const WorkItem& w, const WaveUnit& u, double alpha_d,
                                        double beta_d) const {
        accv_t acc[IM][JN];
#pragma unroll
        for (int i = 0; i < IM; ++i)
#pragma unroll
            for (int j = 0; j < JN; ++j) acc[i][j] = accv_t{0, 0, 0, 0};
        // Stage c - 1 in LDS, stage c in registers or on its way; the last one after the loop.
        // (Straight-line stages: a branch around a load would make the compiler wait for every
        // load in flight where the paths meet.)
        Stage s;
        const int n = (k + KS - 1) / KS;
        load(s, 0);
        for (int c = 1; c < n; ++c) {
            write(s);
            wave_lds_order();
            const Held held(s);
            load(s, c);
            __builtin_amdgcn_sched_barrier(0);
            mma(held, acc);
            wave_lds_order();
            __builtin_amdgcn_sched_barrier(0);
        }
        write(s);
        wave_lds_order();
        mma(Held(s), acc);
        const acc_t alpha = (acc_t)alpha_d, beta = (acc_t)beta_d;
        KAMI_GLOBAL out_t* C = (KAMI_GLOBAL out_t*)w.C + ((int64_t)u.ra * 16 * w.ldc + u.ca * 16);
#pragma unroll
        for (int i = 0; i < IM; ++i)
#pragma unroll
            for (int j = 0; j < JN; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    KAMI_GLOBAL out_t* dst = C + (int64_t)(i * 16 + AT::out_row(lane, v)) * w.ldc + j * 16 + (lane & 15);
                    acc_t val = alpha * acc[i][j][v];
                    if (beta != (acc_t)0) val += beta * (acc_t)(*dst);
                    *dst = (out_t)val;
                }
    }
};

// MM x NN: atoms of a wave tile, at most: the smaller the tile, the more waves a SIMD holds (2 x 2
// four, 4 x 2 three, 4 x 4 two).  One wave per unit; a workgroup is four consecutive units
// (neighbouring wave tiles of one problem share its lines of A and B in the CU's L1).
template <class AT, bool KN, int MM, int NN>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(MM == 2 ? 4 : NN == 2 ? 3 : 2)))
batched_wave_kernel(BatchArgs args) {
    constexpr int LDS_WAVE = WaveTile<AT, KN, MM, NN>::LDS;
    __shared__ __attribute__((aligned(16))) unsigned char smem[kWavesPerGroup * LDS_WAVE];
    const int wave = uni(threadIdx.x >> 6);
    unsigned char* const lds = smem + wave * LDS_WAVE;
    const WaveUnit u = load_uniform(args.units + unit_at(blockIdx.x, gridDim.x, wave));
    if (u.im == 0) return;
    const WorkItem w = load_uniform(args.items + u.item);
    auto run = [&](auto im, auto jn) {
        WaveTile<AT, KN, decltype(im)::value, decltype(jn)::value>(w, u, lds).run(w, u, args.alpha, args.beta);
    };
    auto run_rows = [&](auto im) {
        // Returns leave 116 registers where branches past each other leave 160 (4 x 2: 20000
        // problems of 16 to 64 45.0 us against 47.5), but 208 against 166 with 4 x 4 (320^3 x
        // 1024 231 against 226).
        if constexpr (NN == 2) {
            if (u.jn == 1) return run(im, std::integral_constant<int, 1>{});
            if (u.jn == 2) return run(im, std::integral_constant<int, 2>{});
        } else {
            if (u.jn == 1)
                run(im, std::integral_constant<int, 1>{});
            else if (u.jn == 2)
                run(im, std::integral_constant<int, 2>{});
            if (u.jn == 3) run(im, std::integral_constant<int, 3>{});
            if (u.jn == 4) run(im, std::integral_constant<int, 4>{});
        }
    };
    if (u.im == 1) return run_rows(std::integral_constant<int, 1>{});
    if (u.im == 2) return run_rows(std::integral_constant<int, 2>{});
    if constexpr (MM > 2) {
        if (u.im == 3) return run_rows(std::integral_constant<int, 3>{});
        return run_rows(std::integral_constant<int, 4>{});
    }
}

static int size_class(int x) { return x <= 32 ? 0 : x <= 64 ? 1 : x <= 128 ? 2 : x <= 256 ? 3 : 4; }
static int bucket_of(const kami_problem& p) {
    return (size_class(p.m) * 5 + size_class(p.n)) * 5 + size_class(p.k);
}

// Prior variant of a bucket: the largest tile that the problem fills, following the
// reference's choice of fewer, larger warps for larger sizes
// (scripts/fp64_batched_GH200.sh:7-14).  The tile is what the queue counts and deals out;
// every prior's wave tiles are the queue's largest.
static int prior_variant(int prec, int bucket) {
    const int cm = bucket / 25, cn = (bucket / 5) % 5;
    if (cm == 0 && cn == 0) return 1;
    if (prec == KAMI_PREC_F64) {
        if (cm >= 2 && cn >= 2) return 4;
        if (cm >= 2) return 3;
        if (cn >= 2) return 5;
        return 0;
    }
    if (cm >= 3 && cn >= 2) return 3;
    return 0;
}


// Workgroups of one execution: one per kWavesPerGroup units.
static int64_t batched_groups(int64_t n_units) { return n_units / kWavesPerGroup; }

// A dispatch holds fewer than 2^32 work-items; longer queues take several.
constexpr int64_t kMaxGroups = (int64_t)1 << 23;

template <class AT, int MM, int NN>
static void launch_kernel(const BatchArgs& a, bool kn, dim3 grid, hipStream_t s) {
    if (kn)
        hipLaunchKernelGGL((batched_wave_kernel<AT, true, MM, NN>), grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((batched_wave_kernel<AT, false, MM, NN>), grid, dim3(256), 0, s, a);
}

template <class AT>
static hipError_t launch_for(BatchArgs a, bool kn, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int64_t left = batched_groups(a.n_units); left > 0 && e == hipSuccess; left -= kMaxGroups) {
        const dim3 grid((unsigned)std::min(left, kMaxGroups));
        if (kCapM[a.cap] <= 2) {
            launch_kernel<AT, 2, 2>(a, kn, grid, s);
        } else if (kCapN[a.cap] == 2) {
            launch_kernel<AT, 4, 2>(a, kn, grid, s);
        } else if constexpr (sizeof(typename AT::in_t) == 2) {
            launch_kernel<AT, 4, 4>(a, kn, grid, s);
        }
        e = hipGetLastError();
        a.units += kMaxGroups * kWavesPerGroup;
    }
    return e;
}

// log2 of the entries dealt to one of `takers` XCDs at a time: as many as leave every XCD
// three deals or more, from 2 to 1 << kQueueShift.
static int32_t queue_shift(int64_t n_items, int takers) {
    const int64_t per = n_items / (3 * (int64_t)std::max(takers, 1));
    int32_t sh = 1;
    while (sh < kQueueShift && (int64_t(2) << sh) <= per) ++sh;
    return sh;
}

static hipError_t launch_batched(int prec, const BatchArgs& a, bool kn, hipStream_t s) {
    if (prec == KAMI_PREC_F64) return launch_for<AtomF64>(a, kn, s);
    if (prec == KAMI_PREC_F16_F32) return launch_for<AtomF16x32>(a, kn, s);
    return launch_for<AtomBF16x32>(a, kn, s);
}

// The wave tiles of one queue entry, two by two so that four consecutive ones form a
// square (they share lines of A and B).
struct UnitCursor {
    int rows = 0, cols = 0;  // wave tiles of the entry
    int r = 0, c = 0;        // next one
    int am = 0, an = 0;      // atoms of the entry
    int sm = 1, sn = 1;      // atoms of a wave tile
    bool done = true;
    static int strips(int atoms, int most) { return (atoms + most - 1) / most; }
    void start(const WorkItem& w, int cap) {
        am = std::min(w.mlim, kVariantTM[w.variant]) / 16;
        an = std::min(w.nlim, kVariantTN[w.variant]) / 16;
        // as few strips as the cap allows, of nearly equal height
        rows = strips(am, std::min(kCapM[cap], kVariantSM[w.variant]));
        cols = strips(an, std::min(kCapN[cap], kVariantSN[w.variant]));
        sm = strips(am, rows);
        sn = strips(an, cols);
        r = c = 0;
        done = false;
    }
    WaveUnit take(uint32_t item) {
        const WaveUnit u{item, (uint8_t)(r * sm), (uint8_t)(c * sn),
                         (uint8_t)std::min(sm, am - r * sm), (uint8_t)std::min(sn, an - c * sn)};
        if ((c & 1) == 0 && c + 1 < cols) {
            ++c;
        } else if ((r & 1) == 0 && r + 1 < rows) {
            ++r;
            c &= ~1;
        } else if ((c | 1) + 1 < cols) {
            c = (c | 1) + 1;
            r &= ~1;
        } else {
            r = (r | 1) + 1;
            c = 0;
            done = r >= rows;
        }
        return u;
    }
};

// Wave tiles of all entries for the cap, rounded up to a workgroup for every XCD.
static int64_t count_units(const WorkItem* items, int64_t n_items, int cap) {
    int64_t n = 0;
    UnitCursor u;
    for (int64_t i = 0; i < n_items; ++i) {
        u.start(items[i], cap);
        n += (int64_t)u.rows * u.cols;
    }
    constexpr int64_t kRound = kWavesPerGroup * kXcds;
    return (n + kRound - 1) / kRound * kRound;
}

// Fewest wave tiles that fill the chip (four a SIMD); below that the wave tiles are made
// smaller, down to 16 x 16, until there are as many.  FP64, problems of 16 to 256:
// 8 of them 6.0 us against 9.9 with 32 x 32 tiles, 100 9.1 against 13.5, 300 14.7 against
// 17.2 (and 17.2 with 2048 here); FP16 is bound by the launch itself there.
constexpr int64_t kFullUnits = 4096;

// Whether the wave tiles one size larger than first_cap's pay, of which there would be `larger`
// instead of `first`: they have to fill the chip twice over (two waves a SIMD for 2-byte inputs,
// three for FP64; FP16 256^3 x 200, 3200 of them, 34.5 us against 32.4, FP64 K x N 128^3 x 600,
// 4800 of them, 68.0 against 63.7), be fewer by a quarter at least, or little
// is read less often, and run long enough to hide their loads with fewer waves: a mean K by work of
// 128 for 2-byte inputs (two stages; 128^3 x 8192 201 us either way, 144^3 x 4096 192 against
// 205), 96 for FP64 (six; 96^3 x 4096 192 against 198, 64^3 x 8192 155 against 148).  FP64 K x N
// reads B eight bytes a lane, again for every row of tiles: in long queues of wide problems the
// larger ones pay whatever K (256 x 256 x 16 x 2000 217 against 254, 1024 x 256 x 32 x 500 285 against
// 343; but x 100 50 against 47, 128 x 128 x 32 x 2000 86 against 81).
static bool larger_pays(const WorkItem* items, int64_t n_items, int elt, bool b_kn, int64_t larger, int64_t first) {
    if (larger < 2 * 1024 * (elt == 8 ? 3 : 2) || 4 * larger > 3 * first) return false;
    const double least = elt == 8 ? 96 : 128;
    double work = 0, work_k = 0, work_n = 0;
    for (int64_t i = 0; i < n_items; ++i) {
        const WorkItem& w = items[i];
        const double f = (double)std::min(w.mlim, kVariantTM[w.variant]) * std::min(w.nlim, kVariantTN[w.variant]) * w.k;
        work += f;
        work_k += f * w.k;
        work_n += f * w.nlim;  // columns to the problem's edge
    }
    const bool wide_kn = elt == 8 && b_kn && larger >= 14 * 1024 && work_n > 160 * work;
    return wide_kn || work_k >= least * work;
}

static int wave_cap(const WorkItem* items, int64_t n_items, int elt, bool b_kn, int64_t* n_units) {
    int cap = first_cap(elt);
    const int64_t larger = count_units(items, n_items, cap - 1);
    if (larger_pays(items, n_items, elt, b_kn, larger, count_units(items, n_items, cap))) {
        *n_units = larger;
        return cap - 1;
    }
    while ((*n_units = count_units(items, n_items, cap)) < kFullUnits && cap + 1 < kCaps) ++cap;
    return cap;
}

// The wave units of a launch.  Workgroup L runs on XCD L mod kXcds; every XCD takes
// deals of consecutive entries (neighbouring tiles of a problem, or problems of nearly
// equal cost), so the tiles that share rows of A or columns of B run on one XCD at the
// same time and its L2 serves all but the first reader.  An XCD's units lie together, in
// the order of its workgroups (unit_at), so the line one workgroup reads its units from
// serves the next three as well.
static void build_units(const WorkItem* items, int64_t n_items, int cap, int64_t n_units, WaveUnit* out) {
    struct {
        int64_t item = 0, end = 0;
        UnitCursor u;
    } x[kXcds];
    const int64_t deal = (int64_t)1 << queue_shift(n_items, kXcds);
    int64_t next = 0;
    auto more = [&](int q) {  // the next unit of XCD q's stream, dealing again when needed
        if (!x[q].u.done) return true;
        if (++x[q].item >= x[q].end) {
            if (next >= n_items) {
                x[q].item = x[q].end;
                return false;
            }
            x[q].item = next;
            x[q].end = next = std::min(n_items, next + deal);
        }
        x[q].u.start(items[x[q].item], cap);
        return true;
    };
    const int64_t groups = batched_groups(n_units);
    for (int64_t first = 0; first < groups; first += kMaxGroups) {  // dispatch by dispatch
        const int64_t here = std::min(groups - first, kMaxGroups);
        WaveUnit* const base = out + first * kWavesPerGroup;
        for (int64_t L = 0; L < here; ++L) {
            const int q = (int)(L % kXcds);
            for (int w = 0; w < kWavesPerGroup; ++w) {
                int t = 0;
                while (t < kXcds && !more((q + t) % kXcds)) ++t;  // an empty stream takes from another
                base[unit_at(L, here, w)] = t < kXcds ? x[(q + t) % kXcds].u.take((uint32_t)x[(q + t) % kXcds].item)
                                                      : WaveUnit{0, 0, 0, 0, 0};
            }
        }
    }
}

// Queue entries of the problems: every problem cut into tiles of its bucket's variant,
// each entry carrying the tile's own operand pointers.  Problems are ordered longest
// first (by m n k) so the tail of the queue holds the cheapest work, and a problem's tiles
// stay consecutive in row-major order, so that build_units can put the tiles that share
// rows of A or columns of B on one XCD together.
// Queue entries of `count` problems (bucket[p] their size bucket), written to out[];
// `order` is room for `count` indices.  Equal-cost problems keep their input order
// (an index tie-break instead of a stable sort, which may allocate).
static int64_t count_items(const kami_problem* probs, int64_t count, const int* bucket,
                           const int* variant_of_bucket) {
    int64_t n = 0;
    for (int64_t p = 0; p < count; ++p) {
        const int v = variant_of_bucket[bucket[p]];
        n += (int64_t)((probs[p].m + kVariantTM[v] - 1) / kVariantTM[v]) *
             ((probs[p].n + kVariantTN[v] - 1) / kVariantTN[v]);
    }
    return n;
}

static void build_items(const kami_problem* probs, int64_t count, const int* bucket,
                        const int* variant_of_bucket, int ei, int eo, bool b_kn, int64_t* order,
                        WorkItem* out) {
    for (int64_t p = 0; p < count; ++p) order[p] = p;
    std::sort(order, order + count, [&](int64_t a, int64_t b) {
        const kami_problem &P = probs[a], &Q = probs[b];
        const int64_t ca = (int64_t)P.m * P.n * P.k, cb = (int64_t)Q.m * Q.n * Q.k;
        return ca != cb ? ca > cb : a < b;
    });
    int64_t i = 0;
    for (int64_t q = 0; q < count; ++q) {
        const int64_t p = order[q];
        const kami_problem& P = probs[p];
        const int v = variant_of_bucket[bucket[p]];
        const int tm = kVariantTM[v], tn = kVariantTN[v];
        for (int r = 0; r < P.m; r += tm)
            for (int c = 0; c < P.n; c += tn) {
                WorkItem& w = out[i++];
                w.A = static_cast<const char*>(P.A) + (int64_t)r * P.lda * ei;
                w.B = static_cast<const char*>(P.B) + (b_kn ? (int64_t)c : (int64_t)c * P.ldb) * ei;
                w.C = static_cast<char*>(P.C) + ((int64_t)r * P.ldc + c) * eo;
                w.lda = P.lda;
                w.ldb = P.ldb;
                w.ldc = P.ldc;
                w.mlim = P.m - r;
                w.nlim = P.n - c;
                w.k = P.k;
                w.variant = v;
            }
    }
}

static void build_items(const std::vector<kami_problem>& probs, const std::vector<int>& bucket,
                        const int* variant_of_bucket, int ei, int eo, bool b_kn,
                        std::vector<WorkItem>& items) {
    const int64_t count = (int64_t)probs.size();
    std::vector<int64_t> order(probs.size());
    items.resize((size_t)count_items(probs.data(), count, bucket.data(), variant_of_bucket));
    build_items(probs.data(), count, bucket.data(), variant_of_bucket, ei, eo, b_kn, order.data(),
                items.data());
}

// Validates one problem of a batch and fills in packed leading dimensions.
static kami_status check_problem(kami_problem& p, int b_layout, int ei, int eo) {
    if (p.m <= 0 || p.n <= 0 || p.k <= 0 || p.m % 16 || p.n % 16 || p.k % 16) return KAMI_EINVAL;
    if (!p.A || !p.B || !p.C) return KAMI_EINVAL;
    if (!p.lda) p.lda = p.k;
    if (!p.ldb) p.ldb = b_layout == KAMI_B_NK ? p.k : p.n;
    if (!p.ldc) p.ldc = p.n;
    if (p.lda < p.k || p.ldb < (b_layout == KAMI_B_NK ? p.k : p.n) || p.ldc < p.n)
        return KAMI_EINVAL;
    if (!span_fits(p.m, p.lda, ei) || !span_fits(b_layout == KAMI_B_NK ? p.n : p.k, p.ldb, ei) ||
        !span_fits(p.m, p.ldc, eo))
        return KAMI_EINVAL;
    if ((p.lda * ei) % 16 || (p.ldb * ei) % 16 || ((uintptr_t)p.A % 16) || ((uintptr_t)p.B % 16) ||
        ((uintptr_t)p.C % eo))
        return KAMI_EINVAL;
    // Operand pieces are addressed by 32-bit byte offsets from the tile's origin
    // (WaveTile::load): the farthest piece of any tile must end below kBufferRange.
    const int64_t a_span = ((int64_t)(std::min(p.m, 128) - 1) * p.lda + p.k) * ei;
    const int64_t b_span = b_layout == KAMI_B_NK
                               ? ((int64_t)(std::min(p.n, 128) - 1) * p.ldb + p.k) * ei
                               : ((int64_t)(p.k - 1) * p.ldb + std::min(p.n, 128)) * ei;
    if (a_span > kBufferRange || b_span > kBufferRange) return KAMI_ENOTSUP;
    return KAMI_OK;
}

// Tile variant of every size bucket without timing: the tuning cache's choice, else the
// prior.
static void untimed_variants(int precision, int (&variant_of_bucket)[125]) {
    for (int b = 0; b < 125; ++b) {
        const int tuned = batched_tuned_variant(precision, b);
        variant_of_bucket[b] =
            tuned >= 0 && tuned < variants_of(precision) ? tuned : prior_variant(precision, b);
    }
}

static kami_status upload(const void* host, size_t bytes, void** dev) {
    hipError_t e = hipMalloc(dev, bytes ? bytes : 16);
    if (e != hipSuccess) {
        g_last_hip = (int32_t)e;
        return KAMI_ENOMEM;
    }
    if (bytes) {
        e = hipMemcpy(*dev, host, bytes, hipMemcpyHostToDevice);
        if (e != hipSuccess) return hip_fail(e);
    }
    return KAMI_OK;
}

// A queue on the device: the entries, and behind them their wave units.
struct DeviceQueue {
    void* mem = nullptr;
    int64_t n_items = 0, n_units = 0;
    int cap = 0;
    const WorkItem* items() const { return static_cast<const WorkItem*>(mem); }
    const WaveUnit* units() const { return reinterpret_cast<const WaveUnit*>(items() + n_items); }
};

static kami_status upload_queue(const std::vector<WorkItem>& items, int elt, bool b_kn, DeviceQueue* q) {
    const int64_t n = (int64_t)items.size();
    if (n > UINT32_MAX) return KAMI_ENOMEM;  // 256 GiB of entries
    int64_t n_units = 0;
    const int cap = wave_cap(items.data(), n, elt, b_kn, &n_units);
    const size_t item_bytes = (size_t)n * sizeof(WorkItem), bytes = item_bytes + (size_t)n_units * sizeof(WaveUnit);
    std::unique_ptr<unsigned char[]> host(new (std::nothrow) unsigned char[bytes]);
    if (!host) return KAMI_ENOMEM;
    std::memcpy(host.get(), items.data(), item_bytes);
    build_units(items.data(), n, cap, n_units, reinterpret_cast<WaveUnit*>(host.get() + item_bytes));
    q->n_items = n;
    q->n_units = n_units;
    q->cap = cap;
    return upload(host.get(), bytes, &q->mem);
}

// ---- one-shot execution without allocation ----
// The queue of kami_batched_gemm_static lives in `scratch`, a file-scope device array
// (each device holds its own copy until the process ends): up to kStaticItems queue
// entries, and behind them their wave units, at most kStaticUnits (16 wave tiles of
// 32 x 32 in an entry of 128 x 128; smaller wave tiles only while there are fewer than
// kFullUnits).  Host code reaches a device's copy only through the address
// hipGetSymbolAddress returns with that device current (the array's name is a host-side
// stand-in, not a device address).  The host side stages the problems, their order and
// the queue in static arrays, so the call makes no allocation of device or host memory; a
// mutex keeps two host threads from sharing the staging.
constexpr int64_t kStaticItems = 32768;  // 2 MiB of queue entries
constexpr int64_t kStaticUnits = 16 * kStaticItems;
constexpr size_t kStaticBytes = kStaticItems * sizeof(WorkItem) + kStaticUnits * sizeof(WaveUnit);
static_assert(4 * kFullUnits + kWavesPerGroup * kXcds <= kStaticUnits, "small wave tiles fit");
static __device__ __align__(256) unsigned char scratch[kStaticBytes];

struct StaticStaging {
    std::mutex mu;
    unsigned char* dev_ptr[kMaxCachedDevices] = {};  // scratch of each device
    kami_problem probs[kStaticItems];  // a problem holds at least one entry
    int bucket[kStaticItems];
    int64_t order[kStaticItems];
    alignas(16) unsigned char queue[kStaticBytes];  // entries, then units
};
static StaticStaging g_static;

// scratch of the current device (caller holds g_static.mu)
static kami_status static_scratch(unsigned char** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    if (dev < 0 || dev >= kMaxCachedDevices) return KAMI_ENOTSUP;
    if (!g_static.dev_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e);
        g_static.dev_ptr[dev] = static_cast<unsigned char*>(p);
    }
    *out = g_static.dev_ptr[dev];
    return KAMI_OK;
}

}  // namespace kami

struct kami_batched_plan {
    int prec = 0;
    int64_t problems = 0;
    int64_t n_items = 0;
    double flops = 0;
    int b_kn = 0;
    double alpha = 1.0, beta = 0.0;
    kami::DeviceQueue queue;
    std::vector<int> bucket_ids;      // non-empty buckets, ascending
    std::vector<int> bucket_variant;  // chosen variant per non-empty bucket
};

namespace kami {

static void free_plan(kami_batched_plan* p) {
    if (!p) return;
    if (p->queue.mem) (void)hipFree(p->queue.mem);
    delete p;
}

}  // namespace kami

using namespace kami;

extern "C" {

kami_status kami_batched_plan_create(const kami_problem* probs, int64_t count, int32_t precision,
                                     const kami_batched_opts* opts, void* stream,
                                     kami_batched_plan** out) {
    if (!probs || !out || count <= 0 || count > 0x7fffffffLL) return KAMI_EINVAL;
    if (precision != KAMI_PREC_F64 && precision != KAMI_PREC_F16_F32 &&
        precision != KAMI_PREC_BF16_F32)
        return KAMI_ENOTSUP;
    kami_batched_opts o;
    std::memset(&o, 0, sizeof(o));
    o.alpha = 1.0;
    if (opts) o = *opts;
    if (o.b_layout != KAMI_B_NK && o.b_layout != KAMI_B_KN) return KAMI_EINVAL;
    if (o.autotune && o.beta != 0.0) return KAMI_EINVAL;  // tuning runs overwrite C
    const int ei = elt_in(precision), eo = elt_out(precision);
    std::vector<kami_problem> hp(probs, probs + count);
    double flops = 0;
    for (auto& p : hp) {
        const kami_status pst = check_problem(p, o.b_layout, ei, eo);
        if (pst != KAMI_OK) return pst;
        flops += 2.0 * p.m * p.n * (double)p.k;
    }
    kami_status st = device_check();
    if (st != KAMI_OK) return st;
    hipStream_t s = (hipStream_t)stream;

    kami_batched_plan* plan = new (std::nothrow) kami_batched_plan();
    if (!plan) return KAMI_ENOMEM;
    plan->prec = precision;
    plan->problems = count;
    plan->flops = flops;
    plan->b_kn = o.b_layout == KAMI_B_KN;
    plan->alpha = o.alpha;
    plan->beta = o.beta;

    std::vector<int> bucket(hp.size());
    int variant_of_bucket[125];
    bool used[125] = {false};
    for (size_t i = 0; i < hp.size(); ++i) {
        bucket[i] = bucket_of(hp[i]);
        used[bucket[i]] = true;
    }
    untimed_variants(precision, variant_of_bucket);

    hipError_t e = hipSuccess;
    if (o.autotune) {
        // time every variant on up to 256 problems of each bucket, keep the fastest.  The
        // sample is repeated until it carries at least kTuneProblems problems so that every
        // variant is timed at full occupancy (a small sample would be latency-bound and
        // favour the smallest tiles); the repeats write identical values to the same C
        // (tuning requires beta = 0).
        constexpr size_t kTuneProblems = 4096;
        hipEvent_t e0, e1;
        e = hipEventCreate(&e0);
        if (e == hipSuccess) e = hipEventCreate(&e1);
        if (e != hipSuccess) {
            free_plan(plan);
            return hip_fail(e);
        }
        for (int b = 0; b < 125 && st == KAMI_OK; ++b) {
            if (!used[b]) continue;
            std::vector<kami_problem> sample;
            std::vector<int> sb;
            for (size_t i = 0; i < hp.size() && sample.size() < 256; ++i)
                if (bucket[i] == b) {
                    sample.push_back(hp[i]);
                    sb.push_back(0);
                }
            const size_t distinct = sample.size();
            for (size_t i = 0; sample.size() < kTuneProblems; ++i) {
                sample.push_back(sample[i % distinct]);
                sb.push_back(0);
            }
            float best = 1e30f;
            for (int v = 0; v < variants_of(precision); ++v) {
                int vb[1] = {v};
                std::vector<WorkItem> items;
                build_items(sample, sb, vb, ei, eo, plan->b_kn, items);
                DeviceQueue q;
                st = upload_queue(items, ei, plan->b_kn, &q);
                if (st != KAMI_OK) {
                    if (q.mem) (void)hipFree(q.mem);
                    break;
                }
                BatchArgs a{q.items(), q.units(), q.n_units, o.alpha, 0.0, q.cap};
                e = launch_batched(precision, a, plan->b_kn, s);  // warm-up
                if (e == hipSuccess) e = hipEventRecord(e0, s);
                for (int rep = 0; rep < 3 && e == hipSuccess; ++rep)
                    e = launch_batched(precision, a, plan->b_kn, s);
                if (e == hipSuccess) e = hipEventRecord(e1, s);
                if (e == hipSuccess) e = hipEventSynchronize(e1);
                float ms = 0;
                if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
                (void)hipFree(q.mem);
                if (e != hipSuccess) {
                    st = hip_fail(e);
                    break;
                }
                if (ms < best) {
                    best = ms;
                    variant_of_bucket[b] = v;
                }
            }
            if (st == KAMI_OK) set_batched_tuned_variant(precision, b, variant_of_bucket[b]);
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        if (st != KAMI_OK) {
            free_plan(plan);
            return st;
        }
    }

    std::vector<WorkItem> items;
    build_items(hp, bucket, variant_of_bucket, ei, eo, plan->b_kn, items);
    plan->n_items = (int64_t)items.size();
    st = upload_queue(items, ei, plan->b_kn, &plan->queue);
    if (st != KAMI_OK) {
        free_plan(plan);
        return st;
    }
    for (int b = 0; b < 125; ++b)
        if (used[b]) {
            plan->bucket_ids.push_back(b);
            plan->bucket_variant.push_back(variant_of_bucket[b]);
        }

    *out = plan;
    return KAMI_OK;
}

kami_status kami_batched_execute(kami_batched_plan* plan, void* stream) {
    if (!plan) return KAMI_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    const BatchArgs a{plan->queue.items(), plan->queue.units(), plan->queue.n_units, plan->alpha, plan->beta,
                      plan->queue.cap};
    const hipError_t e = launch_batched(plan->prec, a, plan->b_kn, s);
    if (e != hipSuccess) return hip_fail(e);
    return KAMI_OK;
}

kami_status kami_batched_plan_info(const kami_batched_plan* plan, kami_plan_info* out) {
    if (!plan || !out) return KAMI_EINVAL;
    std::memset(out, 0, sizeof(*out));
    out->problems = plan->problems;
    out->work_items = plan->n_items;
    out->buckets = (int32_t)plan->bucket_ids.size();
    out->workgroups = (int32_t)std::min<int64_t>(batched_groups(plan->queue.n_units), INT32_MAX);
    out->flops = plan->flops;
    for (size_t i = 0; i < plan->bucket_variant.size() && i < 16; ++i)
        out->variant_of_bucket[i] = plan->bucket_variant[i];
    return KAMI_OK;
}

kami_status kami_batched_plan_destroy(kami_batched_plan* plan) {
    free_plan(plan);
    return KAMI_OK;
}

kami_status kami_batched_gemm_static(const kami_problem* probs, int64_t count, int32_t precision,
                                     const kami_batched_opts* opts, void* stream) {
    if (!probs || count <= 0) return KAMI_EINVAL;
    if (precision != KAMI_PREC_F64 && precision != KAMI_PREC_F16_F32 &&
        precision != KAMI_PREC_BF16_F32)
        return KAMI_ENOTSUP;
    kami_batched_opts o;
    std::memset(&o, 0, sizeof(o));
    o.alpha = 1.0;
    if (opts) o = *opts;
    if (o.b_layout != KAMI_B_NK && o.b_layout != KAMI_B_KN) return KAMI_EINVAL;
    if (o.autotune || o.use_graph) return KAMI_EINVAL;  // both need memory of their own
    if (count > kStaticItems) return KAMI_ENOSPC;
    const int ei = elt_in(precision), eo = elt_out(precision);
    const bool b_kn = o.b_layout == KAMI_B_KN;

    std::lock_guard<std::mutex> lock(g_static.mu);
    int variant_of_bucket[125];
    untimed_variants(precision, variant_of_bucket);
    for (int64_t i = 0; i < count; ++i) {
        kami_problem& p = g_static.probs[i];
        p = probs[i];
        const kami_status pst = check_problem(p, o.b_layout, ei, eo);
        if (pst != KAMI_OK) return pst;
        g_static.bucket[i] = bucket_of(p);
    }
    const int64_t n_items = count_items(g_static.probs, count, g_static.bucket, variant_of_bucket);
    if (n_items > kStaticItems) return KAMI_ENOSPC;
    kami_status st = device_check();
    if (st != KAMI_OK) return st;
    unsigned char* base = nullptr;
    st = static_scratch(&base);
    if (st != KAMI_OK) return st;
    WorkItem* const items = reinterpret_cast<WorkItem*>(g_static.queue);
    WaveUnit* const units = reinterpret_cast<WaveUnit*>(items + n_items);
    build_items(g_static.probs, count, g_static.bucket, variant_of_bucket, ei, eo, b_kn,
                g_static.order, items);
    int64_t n_units = 0;
    const int cap = wave_cap(items, n_items, ei, b_kn, &n_units);
    build_units(items, n_items, cap, n_units, units);
    hipStream_t s = (hipStream_t)stream;
    // From pageable memory the copy has consumed the staging array when the call returns,
    // so the next call may refill it.
    hipError_t e = hipMemcpyAsync(base, g_static.queue,
                                  (size_t)n_items * sizeof(WorkItem) + (size_t)n_units * sizeof(WaveUnit),
                                  hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return hip_fail(e);
    const WorkItem* d_items = reinterpret_cast<const WorkItem*>(base);
    BatchArgs a{d_items, reinterpret_cast<const WaveUnit*>(d_items + n_items), n_units, o.alpha, o.beta, cap};
    e = launch_batched(precision, a, b_kn, s);
    if (e != hipSuccess) return hip_fail(e);
    return KAMI_OK;
}

}  // extern "C"
