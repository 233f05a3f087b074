// C ABI: status handling, descriptor validation, instance selection, block-GEMM launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/kami.h"
#include "block_gemm_registry.hpp"
#include "kami_internal.hpp"

namespace kami {

thread_local int32_t g_last_hip = 0;

kami_status hip_fail(hipError_t e) {
    g_last_hip = (int32_t)e;
    return KAMI_EHIP;
}

static std::once_flag g_reg_once;
static std::vector<BlockInstance>* g_reg = nullptr;

const std::vector<BlockInstance>& registry() {
    std::call_once(g_reg_once, [] {
        auto* v = new std::vector<BlockInstance>();
        register_f64_instances(*v);
        register_f16_instances(*v);
        register_bf16_instances(*v);
        g_reg = v;
    });
    return *g_reg;
}

int elt_in(int prec) {
    switch (prec) {
        case KAMI_PREC_F16_F32:
        case KAMI_PREC_BF16_F32: return 2;
        default: return 8;
    }
}
int elt_out(int prec) {
    switch (prec) {
        case KAMI_PREC_F16_F32:
        case KAMI_PREC_BF16_F32: return 4;
        default: return 8;
    }
}

// Per-device gfx950 check, cached.
kami_status device_check() {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        g_last_hip = (int32_t)e;
        return KAMI_ENODEV;
    }
    static std::atomic<int> cache[64];  // 0 unknown, 1 ok, 2 not gfx950
    if (dev >= 0 && dev < 64) {
        int c = cache[dev].load(std::memory_order_relaxed);
        if (c == 1) return KAMI_OK;
        if (c == 2) return KAMI_ENODEV;
    }
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, dev);
    if (e != hipSuccess) {
        g_last_hip = (int32_t)e;
        return KAMI_ENODEV;
    }
    const bool ok = std::strncmp(prop.gcnArchName, "gfx950", 6) == 0;
    if (dev >= 0 && dev < 64) cache[dev].store(ok ? 1 : 2, std::memory_order_relaxed);
    return ok ? KAMI_OK : KAMI_ENODEV;
}

// Default wave-grid edge when the caller leaves ranks = 0, per partition.  These are
// the reference's sweep tables (scripts/fp64_block_square_GH200.sh:11-25,
// scripts/fp16_block_square_GH200.sh:11-25) mapped to wave64: 1D keeps M/16 waves of
// 16 rows for FP64; FP16 uses the fewest waves whose accumulators fit.
static int default_ranks(int prec, int part, int m, int n, int k) {
    (void)k;
    const bool f64 = prec == KAMI_PREC_F64 || is_split(prec);
    const int mn = std::max(m, n);
    if (part == KAMI_PART_1D) {
        if (f64) return std::max(1, m / 16);
        if (mn <= 64) return 1;
        if (mn <= 128) return 4;
        return 8;
    }
    if (part == KAMI_PART_2D) {
        if (mn <= 32) return 1;
        if (mn <= 128) return 2;
        return 4;
    }
    // 3D
    if (mn <= 16) return 1;
    return 2;
}

// Choices recorded by kami_block_gemm_autotune per (precision, M, N, K); AUTO uses them
// ahead of the measured priors.
static std::mutex g_tune_mu;
struct TuneKey {
    int prec, m, n, k;
    bool operator==(const TuneKey& o) const {
        return prec == o.prec && m == o.m && n == o.n && k == o.k;
    }
};
struct TuneVal {
    int part, ranks, pipe;
};
static std::vector<std::pair<TuneKey, TuneVal>> g_tuned;

void set_tuned_choice(int prec, int m, int n, int k, int part, int ranks, int pipe) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    for (auto& kv : g_tuned)
        if (kv.first == TuneKey{prec, m, n, k}) {
            kv.second = TuneVal{part, ranks, pipe};
            return;
        }
    g_tuned.push_back({TuneKey{prec, m, n, k}, TuneVal{part, ranks, pipe}});
}

std::vector<TunedBlock> tuned_block_choices() {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    std::vector<TunedBlock> v;
    for (auto& kv : g_tuned)
        v.push_back(TunedBlock{kv.first.prec, kv.first.m, kv.first.n, kv.first.k, kv.second.part,
                               kv.second.ranks, kv.second.pipe});
    return v;
}

void clear_tuned_block_choices() {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned.clear();
}

static bool get_tuned_choice(int prec, int m, int n, int k, TuneVal* out) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    for (auto& kv : g_tuned)
        if (kv.first == TuneKey{prec, m, n, k}) {
            *out = kv.second;
            return true;
        }
    return false;
}

kami_status validate_desc(const kami_gemm_desc* d) {
    if (!d) return KAMI_EINVAL;
    if (d->m <= 0 || d->n <= 0 || d->k <= 0) return KAMI_EINVAL;
    if (d->precision < KAMI_PREC_F64 || d->precision > KAMI_PREC_F64_SPLIT_I8) return KAMI_EINVAL;
    if (d->partition < KAMI_PART_AUTO || d->partition > KAMI_PART_3D) return KAMI_EINVAL;
    if (d->ranks < 0 || d->iters < 1) return KAMI_EINVAL;
    if (d->b_layout != KAMI_B_NK && d->b_layout != KAMI_B_KN) return KAMI_EINVAL;
    if (d->lda < 0 || d->ldb < 0 || d->ldc < 0 || d->slices < 0) return KAMI_EINVAL;
    if (d->pipeline < 0 || d->pipeline > 2) return KAMI_EINVAL;
    const int64_t lda = d->lda ? d->lda : d->k;
    const int64_t ldb = d->ldb ? d->ldb : (d->b_layout == KAMI_B_NK ? d->k : d->n);
    const int64_t ldc = d->ldc ? d->ldc : d->n;
    if (lda < d->k) return KAMI_EINVAL;
    if (ldb < (d->b_layout == KAMI_B_NK ? d->k : d->n)) return KAMI_EINVAL;
    if (ldc < d->n) return KAMI_EINVAL;
    const int e = elt_in(d->precision);
    if (!span_fits(d->m, lda, e) || !span_fits(d->b_layout == KAMI_B_NK ? d->n : d->k, ldb, e) ||
        !span_fits(d->m, ldc, elt_out(d->precision)))
        return KAMI_EINVAL;
    // operands are staged with 16-byte loads
    if ((lda * e) % 16 != 0 || (ldb * e) % 16 != 0) return KAMI_EINVAL;
    return KAMI_OK;
}

// Streaming-mode winners of the instance sweep on MI355X, 64 to 8192 problems.  FP64: the
// persistent 2D form, pipe = 2, from 64^3 up for 512 problems and more (64^3 x 1024 21.5 us
// against 23.5; with 64 problems 5.1 against 4.6), at 32^3 the plain one (x 512 3.7 us against
// 4.2, x 4096 18.2, 19.0); 128 x 128 x 512 2D 4 x 4 317 us x 1024 against 345 for 1D.  BF16 64^3
// 1D like FP16 (x 4096 25.7 us against 29.0 for 2D 4 x 4).  Low rank: more, thinner waves hide
// a small batch's loads (256 x 256 x 32 x 512 1D 8 waves 28.2 us, 16 33.0; 192 x 192 x 32 x 64
// 12 waves 4.8, 4 6.2, x 1024 34.4 and 33.6; 128 x 128 x 32 x 4096 8 waves 63.2, 4 67.9).
// Used for KAMI_PART_AUTO until kami_block_gemm_autotune has measured the shape
// in this process (or a tuning file has been loaded).
struct Prior {
    int prec, m, n, k, part, ranks, pipe = 1;
};
static const Prior kPriors[] = {
    {KAMI_PREC_F64, 16, 16, 16, KAMI_PART_2D, 1},
    {KAMI_PREC_F64, 32, 32, 32, KAMI_PART_2D, 2},
    {KAMI_PREC_F64, 64, 64, 64, KAMI_PART_2D, 4, 2},
    {KAMI_PREC_F64, 128, 128, 128, KAMI_PART_2D, 4, 2},
    {KAMI_PREC_F64, 128, 128, 512, KAMI_PART_2D, 4},
    {KAMI_PREC_F16_F32, 32, 32, 32, KAMI_PART_2D, 1}, {KAMI_PREC_F16_F32, 64, 64, 64, KAMI_PART_1D, 4},
    {KAMI_PREC_F16_F32, 128, 128, 128, KAMI_PART_1D, 4},
    {KAMI_PREC_F16_F32, 256, 256, 256, KAMI_PART_1D, 16},
    {KAMI_PREC_F16_F32, 128, 128, 32, KAMI_PART_1D, 8},
    {KAMI_PREC_F16_F32, 192, 192, 16, KAMI_PART_1D, 12},
    {KAMI_PREC_F16_F32, 256, 256, 16, KAMI_PART_1D, 16}, {KAMI_PREC_F16_F32, 256, 256, 32, KAMI_PART_1D, 8},
    {KAMI_PREC_BF16_F32, 32, 32, 32, KAMI_PART_2D, 1}, {KAMI_PREC_BF16_F32, 64, 64, 64, KAMI_PART_1D, 4},
    {KAMI_PREC_BF16_F32, 128, 128, 128, KAMI_PART_1D, 4},
    {KAMI_PREC_BF16_F32, 256, 256, 256, KAMI_PART_1D, 16},
    {KAMI_PREC_BF16_F32, 128, 128, 32, KAMI_PART_1D, 8},
    {KAMI_PREC_BF16_F32, 192, 192, 16, KAMI_PART_1D, 12},
    {KAMI_PREC_BF16_F32, 256, 256, 16, KAMI_PART_1D, 16}, {KAMI_PREC_BF16_F32, 256, 256, 32, KAMI_PART_1D, 8},
};

// Forms for batches of a few problems, where AUTO would take one of the priors.  Up to as many
// problems as CUs every one has a CU to itself, and more waves on it hide its loads better, while
// there is no next problem to load ahead (us, this form against the prior: FP64 64^3 x 64 4.5,
// 5.1; x 256 7.2, 7.6; x 768 18.0, 15.9.  BF16 128^3 x 64 3.8, 4.6; x 512 12.5, 11.1.  FP16
// 256^3 x 64 13.1, 15.6; x 256 28.1, 28.4; x 512 59.3, 58.0).  128 x 128 x 32 between two
// workgroups of eight waves a CU and the size that caps them wants four waves (x 512 9.6, 9.1;
// x 1024 16.4, 20.2; x 2048 34.9, 33.6), 192 x 192 x 32 twelve only while there is one workgroup
// or two a CU (x 64 4.8, 6.2; x 512 17.4, 17.4; x 8192, 32 times, 392, 384).  The same products in
// the same order, so the bits do not depend on it; the query reports the prior.
struct BatchPrior {
    int64_t first, last;  // problems
    Prior form;
};
static const BatchPrior kBatchPriors[] = {
    {1, 256, {KAMI_PREC_F64, 64, 64, 64, KAMI_PART_2D, 4}},
    {1, 256, {KAMI_PREC_F16_F32, 128, 128, 128, KAMI_PART_2D, 4}},
    {1, 256, {KAMI_PREC_F16_F32, 256, 256, 256, KAMI_PART_2D, 4}},
    {1, 256, {KAMI_PREC_BF16_F32, 128, 128, 128, KAMI_PART_2D, 4}},
    {1, 256, {KAMI_PREC_BF16_F32, 256, 256, 256, KAMI_PART_2D, 4}},
    {513, 1228, {KAMI_PREC_F16_F32, 128, 128, 32, KAMI_PART_1D, 4}},
    {513, 1228, {KAMI_PREC_BF16_F32, 128, 128, 32, KAMI_PART_1D, 4}},
    {1, 512, {KAMI_PREC_F16_F32, 192, 192, 32, KAMI_PART_1D, 12}},
    {1, 512, {KAMI_PREC_BF16_F32, 192, 192, 32, KAMI_PART_1D, 12}},
};
static const Prior* batch_prior(const kami_gemm_desc* d, int64_t count) {
    TuneVal tv;
    if (d->partition != KAMI_PART_AUTO || d->pipeline != 0) return nullptr;
    for (const BatchPrior& b : kBatchPriors) {
        const Prior& p = b.form;
        if (p.prec != d->precision || p.m != d->m || p.n != d->n || p.k != d->k) continue;
        if (count < b.first || count > b.last) continue;
        if (d->iters > 1)  // a resident form is the better one for those
            for (const auto& in : registry())
                if (in.resident && in.prec == p.prec && in.m == p.m && in.n == p.n && in.k == p.k) return nullptr;
        return get_tuned_choice(p.prec, p.m, p.n, p.k, &tv) ? nullptr : &p;
    }
    return nullptr;
}

// The persistent form can be asked for with the 2D partition, B stored N x K and iters = 1.
static bool pipe_allowed(const kami_gemm_desc* d) {
    return d->b_layout == KAMI_B_NK && d->iters == 1;
}

// FP64 has it for B stored K x N too, where no form is asked for.
static bool pipe_chosen_kn(const kami_gemm_desc* d) {
    return d->b_layout == KAMI_B_KN && d->precision == KAMI_PREC_F64 && d->iters == 1 && d->pipeline == 0;
}

// FP64 with B stored K x N and neither a form asked for nor one measured: the persistent form of
// 4 x 4 waves, where one is compiled and the problem is not small (128^3 x 4096 346 us against
// 380, 64^3 x 1024 20.6 against 27.0; but 32^3 x 4096 19.3 against 18.1, x 64 4.4 against 3.9, and 2 x 2
// waves 64^3 x 8192 152 against 138, x 64 6.7 against 5.2).
static const BlockInstance* untuned_form(const kami_gemm_desc* d, bool tuned, const BlockInstance& in) {
    if (tuned || !pipe_chosen_kn(d) || in.m < 64 || in.ranks < 4) return &in;
    for (const auto& o : registry())
        if (o.pipe == 2 && o.prec == in.prec && o.m == in.m && o.n == in.n && o.k == in.k &&
            o.part == in.part && o.ranks == in.ranks)
            return &o;
    return &in;
}

const BlockInstance* resolve_block(const kami_gemm_desc* d, kami_status* st) {
    int part = d->partition, ranks = d->ranks, pipe = d->pipeline;
    bool tuned = false;
    if (pipe < 0 || pipe > 2) {
        *st = KAMI_EINVAL;
        return nullptr;
    }
    if (part == KAMI_PART_AUTO) {
        TuneVal tv;
        part = KAMI_PART_1D;
        ranks = 0;
        int ppipe = 1;
        if (get_tuned_choice(d->precision, d->m, d->n, d->k, &tv)) {
            tuned = true;
            part = tv.part;
            ranks = tv.ranks;
            ppipe = tv.pipe;
        } else {
            for (const Prior& p : kPriors)
                if (p.prec == d->precision && p.m == d->m && p.n == d->n && p.k == d->k) {
                    part = p.part;
                    ranks = p.ranks;
                    ppipe = p.pipe;
                }
        }
        if (pipe == 0) pipe = ppipe;
    }
    if (pipe == 2 && !pipe_allowed(d)) {
        if (d->pipeline == 2) {
            *st = KAMI_ENOTSUP;
            return nullptr;
        }
        if (!(tuned && pipe_chosen_kn(d))) pipe = 1;
    }
    const bool ranks_defaulted = ranks == 0;
    if (ranks_defaulted) ranks = default_ranks(d->precision, part, d->m, d->n, d->k);
    // repeated products (iters > 1) use a key's resident form (all of K in one LDS stage)
    // where one is compiled; a single product uses the streaming form.  The resident forms turn
    // K x N rows of 2-byte values as they write them, all of K before the first product, which
    // two repetitions do not pay for (256^3 x 512 twice 115 us, streamed 83).
    const int resident_from = d->b_layout == KAMI_B_KN && d->precision != KAMI_PREC_F64 ? 3 : 2;
    auto same_key = [&](const BlockInstance& in, int want_pipe) {
        return in.prec == d->precision && in.m == d->m && in.n == d->n && in.k == d->k &&
               in.part == part && in.ranks == ranks && in.pipe == want_pipe;
    };
    if (d->iters >= resident_from && (pipe == 0 || pipe == 1))
        for (const auto& in : registry())
            if (in.resident && same_key(in, 1)) {
                *st = KAMI_OK;
                return &in;
            }
    if (pipe == 0) {
        // a partition (and wave count) given without a form: for FP64 the persistent form
        // where one is compiled for it (measured faster at every such shape: 64^3 x 1024
        // 2D P=2 20.3 us vs 24.6 us, 32^3 x 4096 15.4 vs 17.0 us, 128^3 x 4096 48 vs 37
        // TFLOPS); FP16 / BF16 stream at the HBM rate either way and one workgroup per
        // problem is as fast or faster (128^3 x 8192: 194-199 us vs 206-214 us)
        pipe = 1;
        if (pipe_allowed(d) && d->precision == KAMI_PREC_F64)
            for (const auto& in : registry())
                if (same_key(in, 2)) pipe = 2;
    }
    for (const auto& in : registry()) {
        if (!in.resident && same_key(in, pipe)) {
            *st = KAMI_OK;
            return untuned_form(d, tuned, in);
        }
    }
    // a defaulted wave count that has no compiled instance of this shape: the first
    // compiled instance of the requested partition
    if (ranks_defaulted) {
        for (const auto& in : registry())
            if (!in.resident && in.prec == d->precision && in.m == d->m && in.n == d->n &&
                in.k == d->k && in.part == part && in.pipe == pipe) {
                *st = KAMI_OK;
                return untuned_form(d, tuned, in);
            }
    }
    // AUTO falls back to any compiled per-problem instance of the shape
    if (d->partition == KAMI_PART_AUTO) {
        for (const auto& in : registry())
            if (!in.resident && in.prec == d->precision && in.m == d->m && in.n == d->n &&
                in.k == d->k && in.pipe == 1) {
                *st = KAMI_OK;
                return untuned_form(d, tuned, in);
            }
    }
    *st = KAMI_ENOTSUP;
    return nullptr;
}

}  // namespace kami

using namespace kami;

extern "C" {

const char* kami_status_string(kami_status s) {
    // A C caller may pass any int; read the bits as one rather than as the C++ enum,
    // whose value range ends at 7.
    static_assert(sizeof(kami_status) == sizeof(int32_t), "kami_status is an int");
    int32_t v;
    std::memcpy(&v, &s, sizeof v);
    switch (v) {
        case KAMI_OK: return "KAMI_OK: success";
        case KAMI_EINVAL: return "KAMI_EINVAL: invalid argument";
        case KAMI_ENOTSUP: return "KAMI_ENOTSUP: no compiled instance for this request";
        case KAMI_ENOMEM: return "KAMI_ENOMEM: allocation failed";
        case KAMI_EHIP: return "KAMI_EHIP: HIP runtime error";
        case KAMI_ENOSPC: return "KAMI_ENOSPC: workspace too small";
        case KAMI_ENODEV: return "KAMI_ENODEV: no gfx950 device";
    }
    return "KAMI: unknown status";
}

int32_t kami_last_hip_error(void) { return g_last_hip; }

const char* kami_version(void) { return "kami-mi355x 0.1 (gfx950)"; }

kami_status kami_device_check(void) { return device_check(); }

kami_status kami_gemm_desc_init(kami_gemm_desc* d, int32_t m, int32_t n, int32_t k,
                                int32_t precision) {
    if (!d) return KAMI_EINVAL;
    std::memset(d, 0, sizeof(*d));
    d->m = m;
    d->n = n;
    d->k = k;
    d->precision = precision;
    d->partition = KAMI_PART_AUTO;
    d->ranks = 0;
    d->b_layout = KAMI_B_NK;
    d->iters = 1;
    d->alpha = 1.0;
    d->beta = 0.0;
    return KAMI_OK;
}

kami_status kami_block_gemm_query(const kami_gemm_desc* d, kami_gemm_config* out) {
    kami_status st = validate_desc(d);
    if (st != KAMI_OK) return st;
    if (!out) return KAMI_EINVAL;
    if (is_split(d->precision)) return split_query(d, out);
    const BlockInstance* in = resolve_block(d, &st);
    if (!in) return st;
    out->partition = in->part;
    out->ranks = in->ranks;
    out->waves_m = in->pm;
    out->waves_n = in->pn;
    out->waves_k = in->pk;
    out->threads = in->threads;
    out->k_stage = in->ks;
    out->lds_bytes = in->lds;
    out->slices = 0;
    out->instance = (int32_t)(in - registry().data());
    out->pipeline = in->pipe;
    out->prefetch = in->prefetch;
    return KAMI_OK;
}

// Operand pointers, leading dimensions and problem strides of a kami_block_gemm-style
// call (strides of 0 mean packed problems).
static kami_status prepare_args(const kami_gemm_desc* d, const void* A, const void* B, void* C,
                                int64_t count, int64_t stride_a, int64_t stride_b,
                                int64_t stride_c, BlockArgs& args) {
    kami_status st = validate_desc(d);
    if (st != KAMI_OK) return st;
    if (count < 0 || count > 0x7fffffffLL) return KAMI_EINVAL;
    if (stride_a < 0 || stride_b < 0 || stride_c < 0) return KAMI_EINVAL;
    if (count == 0) return KAMI_OK;
    if (!A || !B || !C) return KAMI_EINVAL;
    const int ei = elt_in(d->precision), eo = elt_out(d->precision);
    if (((uintptr_t)A % 16) || ((uintptr_t)B % 16) || ((uintptr_t)C % eo)) return KAMI_EINVAL;
    args.A = A;
    args.B = B;
    args.C = C;
    args.lda = d->lda ? d->lda : d->k;
    args.ldb = d->ldb ? d->ldb : (d->b_layout == KAMI_B_NK ? d->k : d->n);
    args.ldc = d->ldc ? d->ldc : d->n;
    const int64_t a_span = (int64_t)(d->m - 1) * args.lda + d->k;
    const int64_t b_span = d->b_layout == KAMI_B_NK ? (int64_t)(d->n - 1) * args.ldb + d->k
                                                    : (int64_t)(d->k - 1) * args.ldb + d->n;
    const int64_t c_span = (int64_t)(d->m - 1) * args.ldc + d->n;
    args.sa = stride_a ? stride_a : (d->lda ? a_span : (int64_t)d->m * d->k);
    args.sb = stride_b ? stride_b : (d->ldb ? b_span : (int64_t)d->n * d->k);
    args.sc = stride_c ? stride_c : (d->ldc ? c_span : (int64_t)d->m * d->n);
    // the whole batch within the span limit (each operand already is)
    if (!span_fits(count, args.sa, ei) || !span_fits(count, args.sb, ei) ||
        !span_fits(count, args.sc, eo))
        return KAMI_EINVAL;
    if (count > 1 && ((args.sa * ei) % 16 || (args.sb * ei) % 16)) return KAMI_EINVAL;
    // problems whose C regions overlap would race on the shared elements
    if (count > 1 && args.sc < c_span) return KAMI_EINVAL;
    args.alpha = d->alpha;
    args.beta = d->beta;
    args.iters = d->iters;
    args.b_kn = d->b_layout == KAMI_B_KN;
    return KAMI_OK;
}

kami_status kami_block_gemm(const kami_gemm_desc* d, const void* A, const void* B, void* C,
                            int64_t count, int64_t stride_a, int64_t stride_b, int64_t stride_c,
                            void* stream) {
    BlockArgs args;
    kami_status st = prepare_args(d, A, B, C, count, stride_a, stride_b, stride_c, args);
    if (st != KAMI_OK || count == 0) return st;
    if (is_split(d->precision)) return split_launch(d, args, count, (hipStream_t)stream);
    kami_gemm_desc small = *d;
    if (const Prior* p = batch_prior(d, count)) {
        small.partition = p->part;
        small.ranks = p->ranks;
        small.pipeline = p->pipe;
        d = &small;
    }
    const BlockInstance* in = resolve_block(d, &st);
    if (!in) return st;
    // one workgroup per problem: the grid's work-items must stay below 2^32
    if (in->pipe != 2 && (uint64_t)count * (uint64_t)in->threads >= (1ull << 32))
        return KAMI_ENOTSUP;
    st = device_check();
    if (st != KAMI_OK) return st;
    hipError_t e = in->launch(args, count, (hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    return KAMI_OK;
}

kami_status kami_split_gemm(const kami_gemm_desc* d, const void* A, const void* B, void* C,
                            int64_t count, int64_t stride_a, int64_t stride_b, int64_t stride_c,
                            void* stream) {
    BlockArgs args;
    kami_status st = prepare_args(d, A, B, C, count, stride_a, stride_b, stride_c, args);
    if (st != KAMI_OK || count == 0) return st;
    return split_gemm_tiled(d, args, count, (hipStream_t)stream);
}

kami_status kami_block_gemm_autotune(const kami_gemm_desc* d, const void* A, const void* B,
                                     void* C, int64_t count, void* stream,
                                     kami_gemm_config* chosen) {
    kami_status st = validate_desc(d);
    if (st != KAMI_OK) return st;
    if (is_split(d->precision)) return KAMI_ENOTSUP;
    if (count <= 0 || count > 0x7fffffffLL || !A || !B || !C) return KAMI_EINVAL;
    st = device_check();
    if (st != KAMI_OK) return st;
    hipStream_t s = (hipStream_t)stream;
    hipEvent_t e0, e1;
    hipError_t he = hipEventCreate(&e0);
    if (he != hipSuccess) return hip_fail(he);
    he = hipEventCreate(&e1);
    if (he != hipSuccess) {
        (void)hipEventDestroy(e0);
        return hip_fail(he);
    }
    float best_ms = 1e30f;
    int best_part = 0, best_ranks = 0, best_pipe = 1;
    kami_gemm_desc untold = *d;
    untold.pipeline = 0;  // every form is timed, whichever the caller asks for
    st = KAMI_ENOTSUP;
    for (const auto& in : registry()) {
        if (in.prec != d->precision || in.m != d->m || in.n != d->n || in.k != d->k) continue;
        const bool kn_form = in.pipe == 2 && pipe_chosen_kn(&untold);  // not to be had by asking
        if (in.pipe == 2 && !pipe_allowed(d) && !kn_form) continue;
        if (in.resident) continue;  // dispatched by iters under its streaming form's key
        kami_gemm_desc t = *d;
        t.partition = in.part;
        t.ranks = in.ranks;
        t.pipeline = in.pipe;
        t.beta = 0.0;  // repeated runs must not feed back into C
        BlockArgs args;
        auto run = [&]() -> kami_status {
            if (!kn_form) return kami_block_gemm(&t, A, B, C, count, 0, 0, 0, stream);
            const kami_status r = prepare_args(&t, A, B, C, count, 0, 0, 0, args);
            if (r != KAMI_OK) return r;
            const hipError_t e = in.launch(args, count, s);
            return e == hipSuccess ? KAMI_OK : hip_fail(e);
        };
        kami_status r = run();  // warm-up
        if (r != KAMI_OK) { st = r; break; }
        (void)hipEventRecord(e0, s);
        for (int rep = 0; rep < 3; ++rep) (void)run();
        (void)hipEventRecord(e1, s);
        he = hipEventSynchronize(e1);
        if (he != hipSuccess) { st = hip_fail(he); break; }
        float ms = 0;
        (void)hipEventElapsedTime(&ms, e0, e1);
        if (ms < best_ms) {
            best_ms = ms;
            best_part = in.part;
            best_ranks = in.ranks;
            best_pipe = in.pipe;
        }
        st = KAMI_OK;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (st != KAMI_OK) return st;
    set_tuned_choice(d->precision, d->m, d->n, d->k, best_part, best_ranks, best_pipe);
    if (chosen) {
        kami_gemm_desc t = *d;
        t.partition = KAMI_PART_AUTO;
        t.ranks = 0;
        t.pipeline = 0;
        return kami_block_gemm_query(&t, chosen);
    }
    return KAMI_OK;
}

}  // extern "C"
