// Block SpMM: C (M x N) = alpha * A * op(B) + beta * C with A in BSR and B dense.
//
// The reference computes one such product per CTA with A re-tiled per warp rank
// (src/sparse/spmm/2d/block_spmm_2d_half_mma.cu:72-235, bsr2tilebsr :264-291) and B stored
// N x K, so C(i, j) = sum_k A(i, k) B[j * K + k] (check loop :378-403).  Here A stays in
// plain BSR (the same format the SpGEMM entry points take) and the product is spread
// over workgroups:
//   * one workgroup per (block row i, column tile of C).  The row's blocks are cut into
//     stages of one line of K (up to 128 bytes) per row of A and column of B; the stages
//     are shared out over the workgroup's K groups of waves, which sum their partial tiles
//     through LDS in a fixed order;
//   * a wave stages lines through LDS of its own (no barrier in its loop): loading MFMA
//     fragments straight from memory puts 16 lines under 16 consecutive lanes, which the
//     address unit takes four lanes a clock, four times as long as whole lines;
//   * the next stage's lines are loaded while the current one is multiplied; column
//     indices come through scalar loads, two stages ahead;
//   * workgroups are numbered so that each XCD (workgroup L runs on XCD L mod 8) takes a
//     contiguous run of (column tile, block row) pairs: its L2 sees the B columns of few
//     tiles;
//   * FP16 / BF16 inputs accumulate in FP32, FP64 in FP64; block rows without stored
//     blocks still write beta * C.
#include <algorithm>

#include "kami_internal.hpp"

namespace kami {

struct SpmmArgs {
    int32_t mb, nb, n, b_kn;
    int64_t nnzb, ldb, ldc;
    const int32_t* rowptr;
    const int32_t* colidx;
    const void* vals;
    const void* B;
    void* C;
    double alpha, beta;
    uint32_t first;  // tile of the dispatch's first workgroup
};

// One workgroup per (block row i, tile of WN x 16 CT columns of C): wave (wk, wn) multiplies
// the row's stages wk, wk + WK, ... with its 16 CT columns, so the longest row's chain of
// load-multiply steps is 1 / WK as long.  The partial tiles are summed through LDS in the
// order of wk (the same order every run), then C = alpha sum + beta C.
// What bounds it: 8192^2, 2 % of 32 x 32 blocks, n = 256.  FP64 23.5 us (the earlier kernel,
// fragments of B straight from memory and a barrier per block: 30.4): 89 MB of A and B
// reach the XCDs' L2s and MFMA pipes are 44 % busy; the longest rows (13 blocks against a
// mean of 5) end last.  FP16 6.4 us replayed from a graph (8.3): the chain row pointers ->
// column indices -> lines -> LDS -> sum -> store, once.
template <int BS, class AT, bool KN, int WK_, int WN_, int CT>
struct SpmmGeom {
    using in_t = typename AT::in_t;
    using acc_t = typename AT::acc_t;
    static constexpr int WK = WK_, WN = WN_, WAVES = WK * WN, NT = 64 * WAVES, IM = BS / 16;
    static constexpr int WTN = 16 * CT, TN = WTN * WN;  // columns of a wave, of the workgroup
    static constexpr int ELT = (int)sizeof(in_t), VE = 16 / ELT;
    static constexpr bool F64 = ELT == 8;
    static constexpr int RB = BS * ELT < 128 ? BS * ELT : 128;
    static constexpr int HS = BS * ELT / RB;     // stages per block
    static constexpr int KS = RB / ELT;          // K of a stage
    static constexpr int NF = KS / AT::KSTEP;    // fragments per stage
    static constexpr int PPR = RB / 16;          // 16-byte pieces of a line
    static constexpr int RPI = 64 / PPR;         // lines of one load instruction
    static constexpr int NA = (BS + RPI - 1) / RPI;
    // K x N operands: FP64 fragments straight from memory (16 lanes read 16 consecutive
    // columns), rows of 2-byte values turned by transposing LDS reads
    static constexpr bool TURN = KN && !F64;
    static constexpr int TROW = CT * 32 + 16;    // bytes of a turned K row in LDS
    static constexpr int TPR = CT * 2;           // its 16-byte pieces
    static constexpr int NB = !KN ? (WTN + RPI - 1) / RPI : TURN ? (KS * TPR + 63) / 64 : CT * NF;
    static constexpr int A_LDS = BS * RB;
    static constexpr int B_LDS = !KN ? WTN * RB : TURN ? KS * TROW : 0;
    // a wave's partial tile: FP64 as the accumulators lie; FP32 in rows, padded so that the
    // four rows of one store fall on different banks
    static constexpr int CROW = WTN * 4 + 16;
    static constexpr int PART = F64 ? IM * CT * 4 * 64 * 8 : BS * CROW;
    static constexpr int WAVE_LDS = A_LDS + B_LDS > PART ? A_LDS + B_LDS : PART;
    static_assert(BS % AT::KSTEP == 0 && BS % 16 == 0 && KS % AT::KSTEP == 0, "block size");
    static_assert(WAVES * WAVE_LDS <= 160 * 1024 && NT <= 1024, "workgroup");
};

template <int BS, class AT, bool KN, int WK_, int WN_, int CT>
__global__ void __launch_bounds__(64 * WK_ * WN_) __attribute__((amdgpu_waves_per_eu(4)))
spmm_kernel(SpmmArgs a) {
    using G = SpmmGeom<BS, AT, KN, WK_, WN_, CT>;
    using in_t = typename AT::in_t;
    using acc_t = typename AT::acc_t;
    using out_t = typename AT::out_t;
    using frag_t = typename AT::frag_t;
    using accv_t = typename AT::accv_t;
    constexpr int FB = AT::FRAG_BYTES, NF = G::NF, IM = G::IM;
    __shared__ __attribute__((aligned(16))) unsigned char smem[G::WAVES * G::WAVE_LDS];

    const int tid = threadIdx.x, lane = tid & 63, grp = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned char* const lds = smem + wave * G::WAVE_LDS;
    // XCD x = L mod 8 takes the contiguous run [x q + min(x, r), ...) of the tile-major
    // order, q = total / 8, r = total mod 8 (a bijection of [0, total)).
    const uint32_t L = blockIdx.x, total = gridDim.x;
    const uint32_t x = L % 8, q8 = total / 8, r8 = total % 8;
    const uint32_t P = a.first + x * q8 + (x < r8 ? x : r8) + L / 8;
    const int i = (int)(P % (uint32_t)a.mb);             // block row of A and C
    const int nt = (int)(P / (uint32_t)a.mb) * G::TN;    // first column of the C tile
    const int wk = wave / G::WN, wn = wave % G::WN;
    const int n0 = nt + wn * G::WTN;                     // first column of the wave
    const in_t* __restrict__ vals = reinterpret_cast<const in_t*>(a.vals);
    const in_t* __restrict__ B = reinterpret_cast<const in_t*>(a.B);
    // stored blocks of row i (clamped to the arrays the caller described)
    const int64_t rb = load_uniform(a.rowptr + i), re = load_uniform(a.rowptr + i + 1);
    const int64_t beg = rb < 0 ? 0 : rb;
    const int64_t end = re > a.nnzb ? a.nnzb : re;

    const int64_t n_st = (end > beg ? end - beg : 0) * G::HS;
    // block column of stage st (of the row's last block past the end)
    auto block_col = [&](int64_t st) {
        return load_uniform(a.colidx + (st < n_st ? beg + st / G::HS : end - 1));
    };

    // Lines of A and of B (N x K) are loaded by PPR lanes each (a load of fragments would
    // put 16 lines under 16 consecutive lanes, four times the address unit's clocks) and
    // turned into fragments through the wave's own LDS.  Columns past n repeat the last.
    const int lrow = lane / G::PPR, lpiece = lane % G::PPR;
    const in_t* const pa = vals + (lrow % BS) * BS + lpiece * G::VE;
    const in_t* pb[G::NB];
#pragma unroll
    for (int j = 0; j < G::NB; ++j) {
        if constexpr (!KN) {
            const int col = min(n0 + (lrow % G::WTN) + j * G::RPI, a.n - 1);
            pb[j] = B + (int64_t)col * a.ldb + lpiece * G::VE;
        } else if constexpr (G::TURN) {
            const int p = (lane + 64 * j) % (G::KS * G::TPR);
            const int col = min(n0 + (p % G::TPR) * 8, a.n - 8);
            pb[j] = B + (int64_t)(p / G::TPR) * a.ldb + col;
        } else {
            const int col = min(n0 + (j / NF) * 16 + (lane & 15), a.n - 1);
            pb[j] = B + (int64_t)((j % NF) * AT::KSTEP + 2 * grp) * a.ldb + col;
        }
    }
    struct Stage {
        u4_t a[G::NA], b[G::NB];
    };
    // stage st of the row: block beg + st / HS, columns h KS .. of it, h = st mod HS
    auto load_a = [&](int64_t st, Stage& s) {
        const int64_t ao = (beg + st / G::HS) * BS * BS + st % G::HS * G::KS;
#pragma unroll
        for (int t = 0; t < G::NA; ++t) s.a[t] = load_raw<16>(pa + ao + t * G::RPI * BS);
    };
    auto valid = [&](int kb) { return kb >= 0 && kb < a.nb; };  // wave-uniform
    auto load_b = [&](int64_t st, int kb, Stage& s) {
        const int64_t k0 = (int64_t)(valid(kb) ? kb : 0) * BS + st % G::HS * G::KS;
        const int64_t bo = KN ? k0 * a.ldb : k0;
#pragma unroll
        for (int j = 0; j < G::NB; ++j) {
            if constexpr (KN && G::F64) {
                const in_t* p = pb[j] + bo;
                const d2_t v = {p[0], p[a.ldb]};
                s.b[j] = bitcast<u4_t>(v);
            } else {
                s.b[j] = load_raw<16>(pb[j] + bo);
            }
        }
    };
    auto write = [&](const Stage& s) {
#pragma unroll
        for (int t = 0; t < G::NA; ++t) {
            const int r = lrow % BS + t * G::RPI;
            store_raw<16>(lds + r * G::RB + (line_slot<G::RB>(r, lpiece) << 4), s.a[t]);
        }
#pragma unroll
        for (int j = 0; j < G::NB; ++j) {
            if constexpr (!KN) {
                const int r = lrow % G::WTN + j * G::RPI;
                store_raw<16>(lds + G::A_LDS + r * G::RB + (line_slot<G::RB>(r, lpiece) << 4), s.b[j]);
            } else if constexpr (G::TURN) {
                const int p = (lane + 64 * j) % (G::KS * G::TPR);
                store_raw<16>(lds + G::A_LDS + (p / G::TPR) * G::TROW + (p % G::TPR) * 16, s.b[j]);
            }
        }
    };
    struct Frags {
        frag_t a[IM][NF], b[CT][NF];
    };
    auto read = [&](const Stage& s, Frags& f) {
        const int r = lane & 15;
        auto line_frag = [&](const unsigned char* base, int t) {
            if constexpr (FB == 16)
                return bitcast<frag_t>(load_raw<FB>(base + r * G::RB + (line_slot<G::RB>(r, 4 * t + grp) << 4)));
            else
                return bitcast<frag_t>(load_raw<FB>(base + r * G::RB + grp * FB));
        };
#pragma unroll
        for (int t = 0; t < NF; ++t) {
#pragma unroll
            for (int im = 0; im < IM; ++im) f.a[im][t] = line_frag(lds + im * 16 * G::RB, t);
#pragma unroll
            for (int jn = 0; jn < CT; ++jn) {
                if constexpr (!KN) {
                    f.b[jn][t] = line_frag(lds + G::A_LDS + jn * 16 * G::RB, t);
                } else if constexpr (G::TURN) {
                    const unsigned char* p = lds + G::A_LDS + (t * AT::KSTEP + AT::KV * grp + (r >> 2)) * G::TROW +
                                             jn * 32 + 8 * (lane & 3);
                    if constexpr (FB == 16) {
                        const u2_t lo = lds_read_turned(p), hi = lds_read_turned(p + 4 * G::TROW);
                        f.b[jn][t] = bitcast<frag_t>(u4_t{lo[0], lo[1], hi[0], hi[1]});
                    } else {
                        f.b[jn][t] = bitcast<frag_t>(lds_read_turned(p));
                    }
                } else {
                    f.b[jn][t] = bitcast<frag_t>(s.b[jn * NF + t]);
                }
            }
        }
    };

    accv_t acc[IM][CT];
#pragma unroll
    for (int im = 0; im < IM; ++im)
#pragma unroll
        for (int jn = 0; jn < CT; ++jn) acc[im][jn] = accv_t{0, 0, 0, 0};

    // stage in LDS, the next one in registers or on its way
    if (wk < n_st && n0 < a.n) {  // wave-uniform
        Stage s;
        Frags f;
        int kb = block_col(wk), kb_next = block_col(wk + G::WK);
        load_a(wk, s);
        load_b(wk, kb, s);
        for (int64_t st = wk; st < n_st; st += G::WK) {
            const bool ok = valid(kb);
            write(s);
            wave_lds_order();
            read(s, f);
            wave_lds_order();
            if (st + G::WK < n_st) {
                kb = kb_next;
                load_a(st + G::WK, s);
                load_b(st + G::WK, kb, s);
                kb_next = block_col(st + 2 * G::WK);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (ok) {
#pragma unroll
                for (int t = 0; t < NF; ++t)
#pragma unroll
                    for (int e = 0; e < AT::NSUB; ++e)
#pragma unroll
                        for (int jn = 0; jn < CT; ++jn)
#pragma unroll
                            for (int im = 0; im < IM; ++im) AT::mma_sub(acc[im][jn], f.a[im][t], f.b[jn][t], e);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // the wave's partial tile over its own stages, which it has left
    out_t* __restrict__ C = reinterpret_cast<out_t*>(a.C);
    const acc_t alpha = (acc_t)a.alpha, beta = (acc_t)a.beta;
#pragma unroll
    for (int im = 0; im < IM; ++im)
#pragma unroll
        for (int jn = 0; jn < CT; ++jn)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int at = G::F64 ? (((im * CT + jn) * 4 + v) * 64 + lane) * 8
                                      : (im * 16 + AT::out_row(lane, v)) * G::CROW + (jn * 16 + (lane & 15)) * 4;
                *reinterpret_cast<acc_t*>(lds + at) = acc[im][jn][v];
            }
    __syncthreads();
    // wave (wk, wn)'s partial tile lies in region wk WN + wn
    if constexpr (G::F64) {
        constexpr int NE = IM * CT * 4 * 64;  // values of a wave tile
#pragma unroll
        for (int s = 0; s < (G::WN * NE + G::NT - 1) / G::NT; ++s) {
            const int g = tid + G::NT * s, e = g % NE, cn = g / NE;
            if (G::WN * NE % G::NT != 0 && cn >= G::WN) break;
            const unsigned char* at = smem + cn * G::WAVE_LDS + e * 8;
            acc_t sum = *reinterpret_cast<const acc_t*>(at);
#pragma unroll
            for (int w = 1; w < G::WK; ++w)
                sum += *reinterpret_cast<const acc_t*>(at + w * G::WN * G::WAVE_LDS);
            const int iv = e >> 6, l = e & 63;  // (im, jn, v) and lane
            const int im = iv / (CT * 4), jn = (iv / 4) % CT, v = iv % 4;
            const int col = nt + cn * G::WTN + jn * 16 + (l & 15);
            if (col >= a.n) continue;
            out_t* dst = C + ((int64_t)i * BS + im * 16 + AT::out_row(l, v)) * a.ldc + col;
            acc_t val = alpha * sum;
            if (beta != (acc_t)0) val += beta * (acc_t)(*dst);
            *dst = (out_t)val;
        }
    } else {
        typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));  // C: 4-byte aligned
        constexpr int QR = G::TN / 4;  // 16-byte pieces of a C row
#pragma unroll
        for (int s = 0; s < (BS * QR + G::NT - 1) / G::NT; ++s) {
            const int e = tid + G::NT * s, row = e / QR, c4 = (e % QR) * 4;
            if (BS * QR % G::NT != 0 && row >= BS) break;
            const unsigned char* at = smem + c4 / G::WTN * G::WAVE_LDS + row * G::CROW + c4 % G::WTN * 4;
            f4_t sum = *reinterpret_cast<const f4_t*>(at);
#pragma unroll
            for (int w = 1; w < G::WK; ++w)
                sum += *reinterpret_cast<const f4_t*>(at + w * G::WN * G::WAVE_LDS);
            if (nt + c4 >= a.n) continue;
            f4u_t* dst = reinterpret_cast<f4u_t*>(C + ((int64_t)i * BS + row) * a.ldc + nt + c4);
            f4u_t val = alpha * sum;
            if (beta != (acc_t)0) val += beta * *dst;
            *dst = val;
        }
    }
}

// A dispatch holds fewer than 2^32 work-items; more tiles take several.
template <int BS, class AT, int WK, int WN, int CT>
static hipError_t launch_form(SpmmArgs a, hipStream_t s) {
    using G = SpmmGeom<BS, AT, false, WK, WN, CT>;
    constexpr int64_t kMost = ((int64_t)1 << 31) / G::NT;
    const int64_t total = (int64_t)a.mb * (((int64_t)a.n + G::TN - 1) / G::TN);
    hipError_t e = hipSuccess;
    for (int64_t first = 0; first < total && e == hipSuccess; first += kMost) {
        const dim3 grid((unsigned)std::min(total - first, kMost)), block(G::NT);
        a.first = (uint32_t)first;
        if (a.b_kn)
            hipLaunchKernelGGL((spmm_kernel<BS, AT, true, WK, WN, CT>), grid, block, 0, s, a);
        else
            hipLaunchKernelGGL((spmm_kernel<BS, AT, false, WK, WN, CT>), grid, block, 0, s, a);
        e = hipGetLastError();
    }
    return e;
}

// Which form.  Four K groups of waves share a row's stages; FP64 blocks of 32 two K groups x two
// column groups (a row's two stages per block go to one wave each, and the column groups read
// A's lines together: 23.5 us against 26.2 for four K groups at 8192^2, 2 % of 32 x 32
// blocks, n = 256).  Where the tiles leave the chip idle and the rows are long, one row's stages
// go to 16 or 8 waves: 20 block rows of 80 blocks of 32, n = 48: FP64 28.6 us against 43.5 with
// four, FP16 11.2 against 13.6; 100 rows of 20, n = 64: FP64 15.1 against 17.0.
// 16 columns are one atom (4096 rows of 2 blocks of 16: FP64 10.4 us with the tiles of
// more columns, 6.1; FP16 5.9 and 4.0).
// FP64 with tiles enough to fill the chip shares a row's A among four column groups, so that no
// partial tiles are summed: blocks of 16, 4096 rows of 1, n = 1024 291 us with four K groups, 194;
// rows of 16, n = 256 407 and 323; but with few tiles for the rows' length four K groups: 256
// rows of 51, n = 1024 142 and 154, 4800^2, 20 %, n = 128 31.7 and 36.3.  Columns of one atom a wave
// (64 a workgroup) where there are no more, or rows and tiles are few (1000 rows of 1, n = 256 16.9
// us, 11.8; with 128 a workgroup 12.7).  Blocks of 32 split K of their own block two ways already, and
// uneven rows want that (512 rows of 3.2, n = 256 27 us, 30 with column groups); rows of 1 (4096, n
// = 256 112 and 104) and long ones (16, n = 256 941 and 820) do not.
// 2-byte blocks of 16 whose B, stored N x K, has more than an XCD's L2 (4 MiB) under 64 columns take 32 (4096
// rows of 4, n = 256 57 us, 41; rows of 1 27 and 29; K x N 28 and 47).
template <int BS, class AT, int CT>
static hipError_t launch_spmm(const SpmmArgs& a, hipStream_t s) {
    using G = SpmmGeom<BS, AT, false, 4, 1, CT>;
    const int64_t tiles = (int64_t)a.mb * ((a.n + G::WTN - 1) / G::WTN);
    const int64_t stages = a.nnzb * G::HS / a.mb;  // of an average row
    if (tiles <= 256 && stages >= 32) return launch_form<BS, AT, 16, 1, CT>(a, s);
    if (tiles <= 512 && stages >= 16) return launch_form<BS, AT, 8, 1, CT>(a, s);
    if (a.n <= 16) return tiles <= 512 ? launch_form<BS, AT, 4, 1, 1>(a, s) : launch_form<BS, AT, 2, 1, 1>(a, s);
    const bool many = tiles > std::max<int64_t>(1024, 400 * stages);
    if constexpr (G::F64 && BS == 32) {
        if (many && stages <= 2 && a.n > 32 && a.n <= 64) return launch_form<BS, AT, 1, 4, 1>(a, s);
        if (many && (stages <= 2 || stages >= 24) && a.n >= 128) return launch_form<BS, AT, 1, 4, 2>(a, s);
        return launch_form<BS, AT, 2, 2, CT>(a, s);
    } else if constexpr (G::F64) {
        if (a.n <= 32 && stages <= 2) return launch_form<BS, AT, 1, 2, 1>(a, s);
        if (many && a.n > 32) {
            if (a.n < 128 || (stages <= 6 && tiles < 8192)) return launch_form<BS, AT, 1, 4, 1>(a, s);
            return launch_form<BS, AT, 1, 4, 2>(a, s);
        }
    } else if constexpr (BS == 16) {
        if (!a.b_kn && stages >= 3 && (int64_t)a.nb * BS * 64 * G::ELT > (4 << 20)) return launch_form<BS, AT, 4, 1, 2>(a, s);
    }
    return launch_form<BS, AT, 4, 1, CT>(a, s);
}

}  // namespace kami

using namespace kami;

extern "C" {

kami_status kami_bsr_spmm(const kami_bsr* A, const void* B, int32_t n, int64_t ldb,
                          int32_t b_layout, void* C, int64_t ldc, int32_t precision,
                          double alpha, double beta, void* stream) {
    if (!A || A->mb <= 0 || A->nb <= 0 || A->nnzb < 0 || !A->rowptr) return KAMI_EINVAL;
    if (A->nnzb > 0 && (!A->colidx || !A->vals)) return KAMI_EINVAL;
    if (b_layout != KAMI_B_NK && b_layout != KAMI_B_KN) return KAMI_EINVAL;
    if (n <= 0 || n % 16 || !B || !C) return KAMI_EINVAL;
    if (A->bs != 16 && A->bs != 32) return KAMI_ENOTSUP;
    int ei, eo;
    if (precision == KAMI_PREC_F16_F32 || precision == KAMI_PREC_BF16_F32) {
        ei = 2;
        eo = 4;
    } else if (precision == KAMI_PREC_F64) {
        ei = 8;
        eo = 8;
    } else {
        return KAMI_ENOTSUP;
    }
    const int64_t K = (int64_t)A->nb * A->bs;
    if (ldb == 0) ldb = b_layout == KAMI_B_NK ? K : n;
    if (ldc == 0) ldc = n;
    if ((b_layout == KAMI_B_NK && ldb < K) || (b_layout == KAMI_B_KN && ldb < n) || ldc < n)
        return KAMI_EINVAL;
    if (!span_fits(b_layout == KAMI_B_NK ? n : K, ldb, ei) ||
        !span_fits((int64_t)A->mb * A->bs, ldc, eo))
        return KAMI_EINVAL;
    if ((ldb * ei) % 16 || ((uintptr_t)B % 16) || ((uintptr_t)C % eo)) return KAMI_EINVAL;
    if (A->nnzb > 0 && ((uintptr_t)A->vals % 16)) return KAMI_EINVAL;
    // (fewer than 2^26 tiles of any form)
    if ((int64_t)A->mb * (((int64_t)n + 63) / 64) >= ((int64_t)1 << 24)) return KAMI_ENOTSUP;
    kami_status st = device_check();
    if (st != KAMI_OK) return st;
    SpmmArgs a;
    a.mb = A->mb;
    a.nb = A->nb;
    a.n = n;
    a.b_kn = b_layout == KAMI_B_KN;
    a.nnzb = A->nnzb;
    a.ldb = ldb;
    a.ldc = ldc;
    a.rowptr = A->rowptr;
    a.colidx = A->colidx;
    a.vals = A->vals;
    a.B = B;
    a.C = C;
    a.alpha = alpha;
    a.beta = beta;
    hipStream_t s = (hipStream_t)stream;
    hipError_t e;
    if (precision == KAMI_PREC_F16_F32)
        e = A->bs == 16 ? launch_spmm<16, AtomF16x16, 4>(a, s) : launch_spmm<32, AtomF16x32, 4>(a, s);
    else if (precision == KAMI_PREC_BF16_F32)
        e = A->bs == 16 ? launch_spmm<16, AtomBF16x16, 4>(a, s) : launch_spmm<32, AtomBF16x32, 4>(a, s);
    else
        e = A->bs == 16 ? launch_spmm<16, AtomF64, 2>(a, s) : launch_spmm<32, AtomF64, 2>(a, s);
    if (e != hipSuccess) return hip_fail(e);
    return KAMI_OK;
}

}  // extern "C"
