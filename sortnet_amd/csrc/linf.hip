// l-inf distance, masked order-statistic neuron and interval-bound forward entry points.
#include "fwd_tile.h"
#include "fwd_args.h"
#include "fwd_cols.h"
#include "bound_cols.h"
#include "sort_cols.h"
#include "row_cands.h"
#include "row_stream.h"
#include <atomic>
#include <mutex>
#include <type_traits>

using namespace sd;

// largest share of marked (tile, weight row, input) triples at which the candidate-table kernel of the interval
// forward runs instead of the kernel that evaluates every term (sd_set_bound_candidate_density); negative: built-in
static std::atomic<float> g_bound_density{-1.f};
// measured at B = 512, M = N = 5120: the table kernel takes 0.09 + 2.6 x share ms (about 60 SIMD cycles per marked
// (tile, weight row, input)) after 0.10 ms for the tables, against 1.00 ms for every term.  The tables are paid for by the time
// the choice is made, so the limit sits a little below where the two would meet.  Per batch row (us, every term / tables):
// 1004 / 379 (9.2 % marked), with positions 1246 / 466; 981 / 538 (37 %), with positions 1268 / 888; 128 x 5120 x
// 5120 293 / 178 and 350 / 256 (19 %), 289 / 234 and 355 / 352 (37 %).
constexpr float kBoundColsCap = 0.30f, kBoundRowsCap = 0.40f;
// With the built-in limits, layers below this many terms go without tables: building them and starting the table
// kernel takes about 0.19 ms, which is what the every-term kernel needs for 2.4 G terms (512 x 10 x 5120: 0.06 ms
// for every term against 0.10 ms from tables).
constexpr long long kBoundColsMinTerms = 1ll << 31;
// The forward that also returns positions: its table kernel spends about twice as long per mark (a compare and two
// selects per output instead of a three-operand minimum or maximum) and the every-term kernel 1.5 times as long per
// term, so the limit is lower per weight row.
constexpr float kBoundPosColsCap = 0.15f;
// Layers between kBoundRowsMinTerms + kBoundRowsMinOutputs x inputs and kBoundColsMinTerms terms are given the tables per batch
// row alone: a wavefront walks a row, so the time follows the length of the rows (about 14 us + 17 us per 1024 inputs) and not
// the outputs, which is what the every-term kernel's time follows.  Every term / tables, us, images against weights of scale
// 0.02 (9.4 % marked), without and with positions: 512 x 1024 x 1024 57 / 41, 95 / 56; 250 x 3072 x 1021 84 / 70, 110 / 87; 400 x
// 5120 x 640 139 / 95, 218 / 114; below the line 128 x 1024 x 1024 21 / 34, 39 / 42 and 100 x 3072 x 1024 44 / 65, 62 / 80.  At 22.5 %
// marked 256 x 2048 x 1200 takes 67 / 73, 99 / 109 (512 x 1024 x 1024 57 / 51), which is where their limit comes from.  Weights
// that decide mark everything: about 25 us for the tables, until the hints say not to build them; a graph, whose replays the
// hints do not reach, holds them only where they served the layer's last calls.
constexpr long long kBoundRowsMinTerms = 1ll << 27, kBoundRowsMinOutputs = 3ll << 16;
constexpr float kBoundSmallRowsCap = 0.18f;
constexpr int kHintSiteBound = 1, kHintSiteBoundSparse = 8, kHintSiteBoundPos = 9;
constexpr float kBoundSparseCap = 0.03f;   // marked share up to which the kernel without LDS staging runs
static std::atomic<int> g_bound_form{0};            // 0: chosen per layer, 1: staged tiles, 2: transposed-row walk

// The l-inf forward (plain, and under the factored mask) on dense single-group layers queues a kernel that works from
// per-weight-row candidate tables in front of the kernels that evaluate every term; a count taken on the device
// decides which runs.  Negative g_linf_density: built-in limit, layers of at least kMaxColsMinTerms terms, and not
// where the tables have not paid lately (hint_build_tables); 0 never; up to 1: that share, at any size.
static std::atomic<float> g_linf_density{-1.f};
static std::atomic<int> g_linf_depth{0};   // under the mask: inputs the bound of a weight row rests on (0 = from the keep probability)
constexpr float kMaxColsCap = 0.10f;
constexpr long long kMaxColsMinTerms = 1ll << 31;   // below, the tables cost more than evaluating every term
constexpr int kHintSiteLinf = 4, kHintSiteMasked = 5;

// Depth of the tables' bound for this shape and mask (0 = the call is not served from tables), by shape and size
// alone: the workspace is sized by this, so that a call under graph capture (which always builds tables) never needs
// more than the eager call before it did.
static int max_cols_eligible(const FwdArgs& a, float keep_x, int B, int CO, int CI, int G, int HW) {
    const float density = g_linf_density.load(std::memory_order_relaxed);
    const int depth = g_linf_depth.load(std::memory_order_relaxed);
    if (density == 0.f || G != 1 || HW != 1 || CI % kSortColsChunk != 0 || CI > 65536 || !a.fast_x || !a.fast_w ||
        a.ci_idx || a.co_idx) return 0;
    int K = max_cols_depth(keep_x);
    if (depth > 0 && keep_x < 1.f) K = depth;
    if (K == 0 || density > 0.f) return K;
    return (long long)B * CO * CI >= kMaxColsMinTerms ? K : 0;
}
// eligible depth `K`, or 0 when (with the built-in limit) the layer's tables have not paid lately
static int max_cols_wanted(const FwdArgs& a, int K, int site, int B, int CO, int CI, hipStream_t st) {
    if (K == 0 || g_linf_density.load(std::memory_order_relaxed) > 0.f) return K;
    return hint_build_tables(site, a.w, B, CO, CI, st) ? K : 0;
}

// Largest share of marked (tile of 128 weight rows, batch row, input) triples at which the l-inf kernel of the tables
// per batch row runs, and the smallest layer (in terms) given such tables under the built-in limit.  Every term / tables, us,
// 512 x 5120 x 5120, inputs in [0, 1] against weights of growing scale: without positions 384 / 263 (6.5 % marked), 383 / 303
// (13 %), 387 / 373 (25 %); with them 516 / 281, 504 / 326, 507 / 422; factored mask with positions 554 / 326 (4 %), 552 / 352
// (7 %), 549 / 409 (14 %).  Smaller layers lose: 128 x 5120 x 5120 110 / 139, with positions 168 / 146.  With the
// 512 x 3072 x 5120 layer served from tables the benchmark step gained 0.1 ms on one stream and lost 0.05 ms on three
// (presumably the table passes and the transposed copy, which stream the operands through memory, meet the traffic of the
// optimizer and the backward on the other streams), so the size limit sits above that layer.
constexpr float kMaxRowsCap = 0.20f;
constexpr long long kMaxRowsMinTerms = 1ll << 33;

// bytes of both tables' workspace for one call: per weight row first, per batch row behind it
static size_t max_tables_bytes(int B, int CO, int CI, int K) {
    const size_t cols = (sort_cols_workspace(B, CO, CI) + 255) / 256 * 256;
    return cols + (row_cands_supported(kRowsMax, K) ? (row_cands_workspace(kRowsMax, B, CO, CI) + 255) / 256 * 256 : 0);
}

// `ws`: max_tables_bytes() bytes.  Afterwards a.gate[0] is non-zero when the every-term kernels are to run.
static int queue_max_cols(FwdArgs& a, int K, int B, int CO, int CI, void* ws, hipStream_t st) {
    const float density = g_linf_density.load(std::memory_order_relaxed);
    const float cap = density > 0.f ? density : kMaxColsCap;
    // depth 1: the mask keeps everything
    const uint32_t* xkeep = K == 1 ? nullptr : a.xmask;
    const uint32_t* wkeep = K == 1 ? nullptr : a.wmask;
    int rc = max_cols_forward(a.x0, a.w, xkeep, wkeep, B, CO, CI, K, a.y0, a.p0, ws, cap, &a.gate, &a.gate_limit, st);
    a.gate_above = 1;
    const bool rows = row_cands_supported(kRowsMax, K) && (density > 0.f || (long long)B * CO * CI >= kMaxRowsMinTerms);
    if (rc || !rows) {
        if (!rc) { a.gate = a.gate + 1; a.gate_limit = 0ull; }   // the flag behind the counter, as with both tables
        return rc;
    }
    const unsigned long long* col_count = a.gate;
    char* rows_ws = static_cast<char*>(ws) + (sort_cols_workspace(B, CO, CI) + 255) / 256 * 256;
    const unsigned long long* every = nullptr;
    rc = row_cands_forward(kRowsMax, a.x0, nullptr, a.w, xkeep, wkeep, B, CO, CI, 0.f, K, nullptr, a.y0, a.p0, rows_ws,
                           density > 0.f ? density : kMaxRowsCap, density > 0.f, sort_cols_probe_sums(col_count), col_count, &every, st);
    if (rc) return rc;
    a.gate = every;
    a.gate_limit = 0ull;
    note_term_counts(every - 1, 3, (double)((CO + 127) / 128) * B * CI, (double)((B + 127) / 128) * CO * CI);
    return SD_OK;
}

// before the every-term kernel is queued behind the table kernels: where it reports
static void max_cols_expect(FwdArgs& a, const float* weight, int site, int B, int CO, int CI, hipStream_t st) {
    if (g_linf_density.load(std::memory_order_relaxed) < 0.f && a.gate) a.told = hint_expect(site, weight, B, CO, CI, st);
}

extern "C" int sd_set_linf_candidate_density(float density) {
    SD_REQUIRE(density <= 1.f, "set_linf_candidate_density: %g is above 1", (double)density);
    g_linf_density = density;
    return SD_OK;
}

extern "C" int sd_set_linf_candidate_depth(int depth) {
    SD_REQUIRE(depth == 0 || depth == 8 || depth == 12 || depth == 16 || depth == 20 || depth == 24,
               "set_linf_candidate_depth: %d is not one of 0, 8, 12, 16, 20, 24", depth);
    g_linf_depth = depth;
    return SD_OK;
}

// One work-item per (row, chunk): the 32 keep bits of the factored mask for inputs
// chunk*32 .. chunk*32+31 of an x row (stream 1) or, behind the xrows x rows, of a w row (stream 2).
static __global__ void __launch_bounds__(256) build_masks_kernel(uint32_t* __restrict__ out, long long xrows, long long rows, int nchunks,
                                                          int CIg, uint32_t seed, uint32_t t16) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * nchunks) return;
    const long long r = i / nchunks;
    const int chunk = (int)(i - r * nchunks);
    const uint32_t key = r < xrows ? rng_row_key(seed, 1u, (uint32_t)r) : rng_row_key(seed, 2u, (uint32_t)(r - xrows));
    uint32_t bits = 0;
    #pragma unroll 8
    for (int k = 0; k < KT; k++) {
        int n = chunk * KT + k;
        if (n < CIg && (rng_word(key, (uint32_t)n) >> 16) < t16) bits |= 1u << k;
    }
    out[i] = bits;
}

// forward with positions: chunk-tracking kernel (split-N through the packed workspace when the
// grid would otherwise be too small) followed by the position resolve pass
// merge_buf / merge_cap: caller-supplied memory for the split-N merge instead of the library workspace (the entry
// point that allocates nothing); a problem that needs more than merge_cap bytes is rejected
template <class P>
static int run_chunk_pos(FwdArgs& a, bool index_lists, hipStream_t st, void* merge_buf = nullptr, size_t merge_cap = 0) {
    // with index lists a batch tile must stay inside one 32-sample sub-batch
    static const int kTb42[] = {4, 2};
    const bool narrow = narrow_tiles(a);
    // served by the scalar-load kernel, which the layers with several positions and rows that are no multiple of 16
    // bytes take as well as the index lists (512 rows of 4 positions x 5120 x 2560: 490 -> 393 us against fwd_kernel,
    // which loads a chunk only when the one before it is done)
    const bool gather = P::LISTS && (index_lists || a.mask_mode < 0) && !(a.fast_x && a.fast_w);
    const int TB = index_lists || narrow || gather ? 2 : pick_tb(a, kTb42, 2, 16 * P::WIDE_TM);
    auto slices = [&] {
        if (narrow) return pick_nsplit(a, 32, 32);
        return TB == 2 ? pick_nsplit(a, 32, gather ? 128 : 16 * P::WIDE_TM, gather && index_lists ? 1 : 8) : pick_nsplit(a, 16 * P::WIDE_TB, 16 * P::WIDE_TM);
    };
    a.nsplit = slices();
    // (what went in one slice needs no scratch, so a stream under capture must not ask for it)
    if (a.nsplit > 1 && !merge_buf && !a.xmask && !workspace_ready((size_t)a.R * a.G * a.COg * 8, st)) { a.coarse = 1; a.nsplit = slices(); }
    // dense exact tiles of the l-inf policy: LDS-direct kernel with 4 x 8 outputs per work-item and the chunk numbers
    // packed four to a register (same (value, chunk) results, so the same resolve pass follows)
    bool packed_direct = false;
    if constexpr (std::is_same<P, LinfChunk>::value) {
        if (TB == 4 && direct_ok<4, 8>(a)) {
            const int ns = pick_nsplit(a, 64, 128);
            if ((a.CIg / KT + ns - 1) / ns <= LinfChunkPacked::MAX_CHUNKS) { packed_direct = true; a.nsplit = ns; }
        }
    }
    int rc;
    if (a.nsplit > 1) {
        // the merge buffer sits at the start of the workspace; a factored-mask call has already sized
        // the workspace for it and placed its bit masks behind it
        size_t n = (size_t)a.R * a.G * a.COg;
        if (merge_buf) {
            SD_REQUIRE(n * 8 <= merge_cap, "inf_dist_forward_noalloc: %zu outputs need %zu bytes of merge scratch, the "
                       "built-in buffer holds %zu (at most %zu outputs)", n, n * 8, merge_cap, merge_cap / 8);
            a.packed0 = static_cast<unsigned long long*>(merge_buf);
        } else a.packed0 = static_cast<unsigned long long*>(a.xmask ? workspace(0, st) : workspace(n * 8, st));
        if (!a.packed0) return SD_ERR_HIP;
        if ((rc = fill_zero(a.packed0, n * 2, st))) return rc;
    }
    if (packed_direct) {
        forward_kernel_timer(st, false);
        rc = launch_fwd_direct<LinfChunkPacked, 4, 8>(a, st);
        forward_kernel_timer(st, true);
    }
    else if (narrow) rc = launch_fwd<P, 2, 2>(a, st);
    else if (TB == 2) rc = gather ? launch_fwd<P, 2, 8>(a, st) : launch_fwd<P, 2, P::WIDE_TM>(a, st);
    else rc = launch_fwd<P, P::WIDE_TB, P::WIDE_TM>(a, st);
    if (rc) return rc;
    return launch_resolve(a, st);
}

// shift: see FwdArgs.  Only the kernels that stream the weights add it to what they store; the others' slices meet in the output (by atomic
// maxima, or by either of two kernels, as the device decides), so there it is added behind them, by the caller: *shifted tells which.
static int linf_values(const float* input, const float* weight, int B, int CO, int CI, int G, int HW, float* output, const float* shift,
                       float sign, bool* shifted, sd_stream_t stream) {
    FwdArgs a;
    *shifted = false;
    int rc = make_fwd_args(a, "inf_dist_forward_nograd", input, nullptr, weight, B, CO, CI, G, HW, nullptr, nullptr, 0, 0);
    if (rc) return rc;
    SD_REQUIRE(output, "inf_dist_forward_nograd: null output");
    a.y0 = output;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool streamed = g_linf_density.load(std::memory_order_relaxed) <= 0.f;   // not where tables are forced
    if (streamed && row_stream_ok(a, kStreamMaxTerms)) {
        a.shift = shift; a.shift_sign = sign;
        *shifted = true;
        return row_stream_linf(a, st);
    }
    if (cols_ok(a, kColsHW, kColsTerms) && workspace_ready(cols_workspace(a), st)) {
        void* ws = workspace(cols_workspace(a), st);
        if (!ws) return SD_ERR_HIP;
        a.nsplit = cols_nsplit(a);
        if (a.nsplit > 1 && (rc = fill_zero(output, (size_t)B * CO * HW, st))) return rc;
        return cols_linf(a, ws, st);
    }
    static const int kTb42[] = {4, 2};   // 8 rows per work-item measured slower (168 registers, three waves per SIMD)
    const bool narrow = narrow_tiles(a);
    const int TB = narrow ? 2 : pick_tb(a, kTb42, 2, 128);
    a.nsplit = pick_nsplit(a, 16 * TB, narrow ? 32 : 128);
    if (a.nsplit > 1 && (rc = fill_zero(output, (size_t)B * CO * HW, st))) return rc;
    const int KE = max_cols_eligible(a, 1.f, B, CO, CI, G, HW);
    const int K = max_cols_wanted(a, KE, kHintSiteLinf, B, CO, CI, st);
    if (KE) {
        void* ws = workspace(max_tables_bytes(B, CO, CI, KE), st);   // the only request of this call
        if (!ws) return SD_ERR_HIP;
        if (K && (rc = queue_max_cols(a, K, B, CO, CI, ws, st))) return rc;
    }
    if (K) max_cols_expect(a, weight, kHintSiteLinf, B, CO, CI, st);
    rc = narrow ? launch_fwd<LinfNograd, 2, 2>(a, st) : TB == 2 ? launch_fwd<LinfNograd, 2, 8>(a, st) : launch_fwd<LinfNograd, 4, 8>(a, st);
    if (rc) hint_forget(a.told);
    return rc;
}

extern "C" int sd_inf_dist_forward_nograd(const float* input, const float* weight,
                                          int B, int CO, int CI, int G, int HW, float* output, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    bool shifted;
    return linf_values(input, weight, B, CO, CI, G, HW, output, nullptr, 0.f, &shifted, stream);
}

extern "C" int sd_inf_dist_forward_shifted(const float* input, const float* weight, int B, int CO, int CI, int G, int HW, float* output,
                                           const float* shift, float sign, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    SD_REQUIRE(shift && (sign == 1.f || sign == -1.f), "inf_dist_forward_shifted: null shift, or a sign (%g) other than 1 and -1", (double)sign);
    SD_REQUIRE(aligned16(shift) && aligned16(output), "inf_dist_forward_shifted: shift and output must be 16-byte aligned");
    bool shifted;
    const int rc = linf_values(input, weight, B, CO, CI, G, HW, output, shift, sign, &shifted, stream);
    return rc || shifted ? rc : channel_shift(output, shift, B, CO, HW, sign, output, static_cast<hipStream_t>(stream));
}

extern "C" int sd_inf_dist_forward(const float* input, const float* weight,
                                   int B, int CO, int CI, int G, int HW, float* output, int* pos,
                                   const int* w_index_ci, const int* w_index_co, int W_CO, int W_CI,
                                   sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    FwdArgs a;
    int rc = make_fwd_args(a, "inf_dist_forward", input, nullptr, weight, B, CO, CI, G, HW,
                           w_index_ci, w_index_co, W_CO, W_CI);
    if (rc) return rc;
    SD_REQUIRE(output && pos, "inf_dist_forward: null output or pos");
    a.y0 = output; a.p0 = pos;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (g_linf_density.load(std::memory_order_relaxed) <= 0.f && row_stream_ok(a, kStreamPosTerms)) return row_stream_linf(a, st);
    if (cols_ok(a, kColsPosHW, kColsPosTerms)) {
        a.nsplit = cols_nsplit(a);
        const size_t weights = (cols_workspace(a) + 255) / 256 * 256, merge = a.nsplit > 1 ? (size_t)a.R * CO * 8 : 0;
        if (workspace_ready(weights + merge, st)) {
            char* ws = static_cast<char*>(workspace(weights + merge, st));
            if (!ws) return SD_ERR_HIP;
            a.packed0 = reinterpret_cast<unsigned long long*>(ws + weights);
            if (merge && (rc = fill_zero(a.packed0, merge / 4, st))) return rc;
            return cols_linf(a, ws, st);
        }
    }
    const int KE = max_cols_eligible(a, 1.f, B, CO, CI, G, HW);
    if (!KE) return run_chunk_pos<LinfChunk>(a, w_index_ci || w_index_co, st);
    const int K = max_cols_wanted(a, KE, kHintSiteLinf, B, CO, CI, st);
    // one workspace request for both users: the split-N merge buffer first, the tables (with the counter the gates
    // read) behind it
    const size_t merge = (((size_t)B * CO * 8) + 255) / 256 * 256;
    char* base = static_cast<char*>(workspace(merge + max_tables_bytes(B, CO, CI, KE), st));
    if (!base) return SD_ERR_HIP;
    if (K && (rc = queue_max_cols(a, K, B, CO, CI, base + merge, st))) return rc;
    if (K) max_cols_expect(a, weight, kHintSiteLinf, B, CO, CI, st);
    rc = run_chunk_pos<LinfChunk>(a, false, st, base, merge);
    if (rc) hint_forget(a.told);
    return rc;
}

// ---- the entry point that allocates nothing ---------------------------------------------------
// Same operation as sd_inf_dist_forward for callers that cannot call hipMalloc (code under graph capture,
// serving loops, harnesses that forbid allocation).  The split-N merge buffer, which sd_inf_dist_forward takes
// from the grow-only library workspace, lives in a file-scope device array instead.  Every GPU holds its own
// copy of the array at its own address: the address is looked up once per device with hipGetSymbolAddress and
// only that pointer is ever handed to kernels.  All calls on one GPU share the array, so calls that overlap on
// one GPU (different streams or threads) race; the part a call uses is cleared by a fill kernel first.
constexpr size_t kScratchBytes = (size_t)32 << 20;   // 4 Mi outputs of 8 bytes: covers 512 x 5120 outputs
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

static int scratch_address(void** out) {
    static std::mutex mu;
    static void* ptrs[64] = {nullptr};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
        (void)hipGetLastError();
        set_error("inf_dist_forward_noalloc: no current device");
        return SD_ERR_HIP;
    }
    std::lock_guard<std::mutex> lock(mu);
    if (!ptrs[dev]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            (void)hipGetLastError();
            set_error("inf_dist_forward_noalloc: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
            return SD_ERR_HIP;
        }
        ptrs[dev] = p;
    }
    *out = ptrs[dev];
    return SD_OK;
}

extern "C" int sd_inf_dist_forward_noalloc(const float* input, const float* weight,
                                           int B, int CO, int CI, int G, int HW, float* output, int* pos,
                                           const int* w_index_ci, const int* w_index_co, int W_CO, int W_CI,
                                           sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    FwdArgs a;
    int rc = make_fwd_args(a, "inf_dist_forward_noalloc", input, nullptr, weight, B, CO, CI, G, HW,
                           w_index_ci, w_index_co, W_CO, W_CI);
    if (rc) return rc;
    SD_REQUIRE(output && pos, "inf_dist_forward_noalloc: null output or pos");
    a.y0 = output; a.p0 = pos;
    const size_t outputs = (size_t)B * CO * HW;
    SD_REQUIRE(outputs * 8 <= kScratchBytes, "inf_dist_forward_noalloc: %zu outputs exceed the maximum of %zu "
               "(8 bytes of built-in merge scratch per output, %zu bytes in all); use sd_inf_dist_forward",
               outputs, kScratchBytes / 8, kScratchBytes);
    void* buf = nullptr;
    if ((rc = scratch_address(&buf))) return rc;
    return run_chunk_pos<LinfChunk>(a, w_index_ci || w_index_co, static_cast<hipStream_t>(stream), buf, kScratchBytes);
}

// Factored mask on rows that cannot be loaded 16 bytes at a time: sets the shape of `a` and CI to that of copies whose rows are whole chunks,
// and returns their bytes, or 0 (as they were).  The kernel that loads value by value draws the keep bits of a tile as it stages it,
// again for every tile.  Without copies -> with them, q = 0.3, without / with positions, us: 91 x 799 x 1920 28 -> 25 / 47 -> 38, 250 x 3071 x
// 1021 92 -> 53 / 118 -> 67, 300 x 5001 x 3000 332 -> 214 / 497 -> 244, 512 x 5121 x 5120 839 -> 298 / 1441 -> 311, 20 x 7001 x 2001 59 -> 54 / 70 -> 61.
// Below 2^27 terms, where there is little to gain, the kernel stays; the smallest layers are streamed.
constexpr long long kMaskPadMinTerms = 1ll << 27;
static size_t masked_pad(FwdArgs& a, int B, int CO, int& CI, int G, int HW) {
    const int N = (CI + KT - 1) / KT * KT;
    if ((a.fast_x && a.fast_w) || G != 1 || HW != 1 || (long long)(B + CO) * N >= (1ll << 31) || B + CO > 4 * 65535 ||
        (long long)B * CO * CI < kMaskPadMinTerms) return 0;
    CI = a.CIg = a.W_CIg = N;
    a.fast_x = a.fast_w = 1;
    return (((size_t)B * N + 63) / 64 * 64 + (size_t)CO * N) * 4;
}

extern "C" int sd_masked_inf_dist_forward(const float* input, const float* weight,
                                          int B, int CO, int CI, int G, int HW, float* output, int* pos,
                                          float q, uint32_t seed, int mode, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    FwdArgs a;
    int rc = make_fwd_args(a, "masked_inf_dist_forward", input, nullptr, weight, B, CO, CI, G, HW, nullptr, nullptr, 0, 0);
    if (rc) return rc;
    SD_REQUIRE(output, "masked_inf_dist_forward: null output");
    SD_REQUIRE(q >= 0.f && q <= 1.f, "masked_inf_dist_forward: q=%g outside [0, 1]", (double)q);
    SD_REQUIRE(mode == SD_MASK_TERM || mode == SD_MASK_FACTORED, "masked_inf_dist_forward: unknown mask mode %d", mode);
    a.y0 = output; a.p0 = pos;
    a.q = q; a.seed = seed; a.mask_mode = mode;
    a.t8 = sd_mask_threshold8(q); a.t16 = sd_mask_threshold16(q);
    const bool small = a.R <= 32;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (mode == SD_MASK_TERM) {
        if (pos) return run_chunk_pos<MaskedTermChunk>(a, false, st);
        a.nsplit = pick_nsplit(a, small ? 32 : 64, 128);
        if (a.nsplit > 1 && (rc = fill_zero(output, (size_t)B * CO * HW, st))) return rc;
        return small ? launch_fwd<MaskedTermMax, 2, 8>(a, st) : launch_fwd<MaskedTermMax, 4, 8>(a, st);
    }
    // factored mask: dropped inputs / weights are replaced by NaN while staging the tiles and
    // NaN terms never win the maximum, so the plain l-inf policies apply unchanged.  On the
    // vector-load path, and for the kernels that stream the weights, the keep bits are built once per call into the
    // library workspace; elsewhere the kernels draw them term by term.
    int K = 0;          // depth of the candidate tables' bound (0: no tables)
    void* tables = nullptr;
    const int nchunks = (a.CIg + KT - 1) / KT;
    const long long xrows = (long long)a.R * G, wrows = (long long)CO;
    const size_t packed_bytes = pos ? (((size_t)a.R * CO * 8 + 255) / 256) * 256 : 0;
    const size_t mask_bytes = ((size_t)(xrows + wrows) * nchunks * 4 + 255) / 256 * 256;
    // (rows that are not streamed for speed need no scratch without positions, so a stream under capture must not ask for it)
    const bool streamed = g_linf_density.load(std::memory_order_relaxed) <= 0.f && row_stream_sizes_ok(a, kStreamMaskTerms) &&
                          ((a.fast_x && a.fast_w) || workspace_ready(packed_bytes + mask_bytes, st));
    // rows that cannot be loaded 16 bytes at a time: copies with zeros behind every row, which the keep bits drop
    const FwdArgs raw = a;
    const size_t copies = streamed ? 0 : masked_pad(a, B, CO, CI, G, HW);
    if (copies) {
        const int KE = max_cols_eligible(a, (float)a.t16 / 65536.f, B, CO, CI, G, HW);
        if (!workspace_ready(packed_bytes + mask_bytes + (KE ? max_tables_bytes(B, CO, CI, KE) : 0) + 256 + copies, st)) { a = raw; CI = raw.CIg; }
    }
    const bool vector = a.fast_x && a.fast_w, padded = vector && !(raw.fast_x && raw.fast_w);
    if (vector || streamed) {
        // one request for every user of the workspace: merge buffer, keep bits, candidate tables
        const int KE = max_cols_eligible(a, (float)a.t16 / 65536.f, B, CO, CI, G, HW);
        K = max_cols_wanted(a, KE, kHintSiteMasked, B, CO, CI, st);
        const size_t table_bytes = KE ? (max_tables_bytes(B, CO, CI, KE) + 255) / 256 * 256 : 0;
        char* base = static_cast<char*>(workspace(packed_bytes + mask_bytes + table_bytes + (padded ? copies : 0), st));
        if (!base) return SD_ERR_HIP;
        if (padded) {
            float* x = reinterpret_cast<float*>(base + packed_bytes + mask_bytes + table_bytes);
            float* w = x + ((size_t)a.R * a.CIg + 63) / 64 * 64;
            if ((rc = pad_rows({raw.x0, raw.x0, raw.w}, {x, x, w}, {a.R, 0, a.COg}, raw.CIg, a.CIg, st))) return rc;
            a.x0 = x;
            a.w = w;
        }
        tables = base + packed_bytes + mask_bytes;
        uint32_t* xm = reinterpret_cast<uint32_t*>(base + packed_bytes);
        uint32_t* wm = xm + xrows * nchunks;
        hipLaunchKernelGGL(build_masks_kernel, dim3((unsigned)(((xrows + wrows) * nchunks + 255) / 256)), dim3(256), 0, st,
                           xm, xrows, xrows + wrows, nchunks, raw.CIg, seed, a.t16);
        if ((rc = check_launch("build_masks_kernel"))) return rc;
        a.xmask = xm; a.wmask = wm;
        if (streamed) return row_stream_linf(a, st);
    }
    if (pos) {
        if (K && (rc = queue_max_cols(a, K, B, CO, CI, tables, st))) return rc;
        if (K) max_cols_expect(a, weight, kHintSiteMasked, B, CO, CI, st);
        rc = run_chunk_pos<LinfChunk>(a, false, st);
        if (rc) hint_forget(a.told);
        return rc;
    }
    static const int kTb42[] = {4, 2};   // 8 rows per work-item measured slower (168 registers, three waves per SIMD)
    const bool narrow = narrow_tiles(a);
    const int TB = narrow ? 2 : pick_tb(a, kTb42, 2, 128);
    a.nsplit = pick_nsplit(a, 16 * TB, narrow ? 32 : 128);
    if (a.nsplit > 1 && (rc = fill_zero(output, (size_t)B * CO * HW, st))) return rc;
    if (K && (rc = queue_max_cols(a, K, B, CO, CI, tables, st))) return rc;
    if (K) max_cols_expect(a, weight, kHintSiteMasked, B, CO, CI, st);
    rc = narrow ? launch_fwd<LinfNograd, 2, 2>(a, st) : TB == 2 ? launch_fwd<LinfNograd, 2, 8>(a, st) : launch_fwd<LinfNograd, 4, 8>(a, st);
    if (rc) hint_forget(a.told);
    return rc;
}

// Interval forward from tables per batch row (row_cands.h): what they need behind the tables per weight row, 0 where they do
// not serve
static size_t bound_rows_bytes(int B, int CO, int CI) {
    return CI <= 65536 && (long long)B * CO < (1ll << 32) ? row_cands_workspace(kRowsBound, B, CO, CI) : 0;
}

// Tables for the interval forward in front of the every-term kernel: per weight row (`cols`, bound_cols.h) and per batch row, or
// the latter alone, which are then built whatever the operands.  Afterwards a.gate[0] is non-zero when the every-term kernel is to run, and
// a.resolved (with positions) when the kernel of the tables per batch row has stored final values and positions.
// `ws`: bound_tables_bytes() bytes.
static size_t bound_tables_bytes(bool cols, int B, int CO, int CI) {
    return (cols ? bound_cols_workspace(B, CO, CI) : 0) + bound_rows_bytes(B, CO, CI);
}

static int queue_bound_tables(FwdArgs& a, bool cols, int B, int CO, int CI, float cap, char* ws, hipStream_t st) {
    const float density = g_bound_density.load(std::memory_order_relaxed);
    const unsigned long long* count = nullptr;
    const float* stat = nullptr;
    char* rows_ws = ws + (cols ? bound_cols_workspace(B, CO, CI) : 0);
    int rc = cols ? bound_cols_forward(a.x0, a.x1, a.w, B, CO, CI, a.y0, a.y1, a.packed0, a.packed1, ws, cap, &count, &stat, st) : SD_OK;
    if (rc) return rc;
    a.gate_above = 1;
    a.gate_limit = 0ull;
    if (cols) a.gate = count + 1;
    if (bound_rows_bytes(B, CO, CI) == 0) {
        note_term_counts(count, 1, (double)((B + 127) / 128) * CO * CI, 1.0);
        return SD_OK;
    }
    const unsigned long long* every = nullptr;
    rc = row_cands_forward(kRowsBound, a.x0, a.x1, a.w, nullptr, nullptr, B, CO, CI, 0.f, 1, a.y0, a.y1, a.p1, rows_ws,
                           density >= 0.f ? density : cols ? kBoundRowsCap : kBoundSmallRowsCap, density >= 0.f, stat, count, &every, st, a.p0);
    if (rc) return rc;
    a.gate = every;
    if (a.p0) a.resolved = every + 1;
    note_term_counts(every - 1, 3, (double)((CO + 127) / 128) * B * CI, (double)((B + 127) / 128) * CO * CI);
    return SD_OK;
}

// whether an interval forward gets tables, by shape and size alone: of both orientations (0: none; 1: per batch row; 2: both)
static int bound_tables_eligible(const FwdArgs& a, float cap, int B, int CO, int CI, int G, int HW) {
    const float density = g_bound_density.load(std::memory_order_relaxed);
    if (!(cap > 0.f && G == 1 && HW == 1 && CI % kColsChunk == 0 && a.fast_x && a.fast_w)) return 0;
    const long long terms = (long long)B * CO * CI;
    if (density >= 0.f || terms >= kBoundColsMinTerms) return 2;
    return terms >= kBoundRowsMinTerms + kBoundRowsMinOutputs * CI && bound_rows_bytes(B, CO, CI) > 0 ? 1 : 0;
}

// Interval layers whose rows are no whole number of table words (32 inputs) work on copies of bounds and weights with zeros behind every
// row, whose terms raise no bound.  Sets the shape of `a` and CI to the copies' and returns their bytes, or 0 (as they were).  Rows that
// can be loaded 16 bytes at a time are copied for tables that a probe of the operands goes before (without it, images gain 96 -> 74 us at
// 118 x 2596 x 2596, and rows that are alike pay 94 -> 103, one call in 32 with tables); others also for the kernels that load so.
// In us, without copies -> with them, inputs in [0, 1] / centred, spread 0.05, weights ~ N(0, 1 / inputs) / the same, weights ~ N(0, 1):
//   without positions  250 x 3071 x 1021 120 -> 56 / 118 -> 61 / 118 -> 99, 300 x 3001 x 3000 355 -> 134 / 360 -> 137 / 357 -> 70, 53 x 10187 x
//                      1472 (no tables) 162 -> 136, 100 x 1001 x 1400 34 -> 31
//   with them          250 x 3071 x 1021 155 -> 70 / 155 -> 75 / 154 -> 126, 300 x 3001 x 3000 621 -> 171 / 622 -> 166 / 620 -> 211, 53 x 10187 x
//                      1472 211 -> 149, 100 x 1001 x 1400 57 -> 51
constexpr long long kBoundPadMinTerms = 1ll << 27;
static size_t bound_pad(FwdArgs& a, float cap, int B, int CO, int& CI, int G, int HW) {
    const int N = (CI + kColsChunk - 1) / kColsChunk * kColsChunk;
    if (N == CI || a.G != 1 || a.HW != 1 || N > 65536 || (long long)(B + CO) * N >= (1ll << 31) || 2ll * B + CO > 4 * 65535) return 0;
    FwdArgs t = a;
    t.CIg = t.W_CIg = N;
    t.fast_x = t.fast_w = 1;
    const bool vectors = a.fast_x && a.fast_w;
    if (bound_tables_eligible(t, cap, B, CO, N, G, HW) < (vectors ? 2 : 1) && (vectors || (long long)B * CO * CI < kBoundPadMinTerms)) return 0;
    a = t;
    CI = N;
    return 2 * (((size_t)B * N * 4 + 255) / 256 * 256) + ((size_t)CO * N * 4 + 255) / 256 * 256;
}
static int bound_pad_copy(FwdArgs& a, const FwdArgs& raw, char* mem, hipStream_t st) {
    const size_t x = ((size_t)a.R * a.CIg * 4 + 255) / 256 * 256;
    float *l = reinterpret_cast<float*>(mem), *u = reinterpret_cast<float*>(mem + x), *w = reinterpret_cast<float*>(mem + 2 * x);
    const int rc = pad_rows({raw.x0, raw.x1, raw.w}, {l, u, w}, {a.R, a.R, a.COg}, raw.CIg, a.CIg, st);
    a.x0 = l; a.x1 = u; a.w = w;
    return rc;
}

// shift, *shifted: see linf_values
static int bound_values(const float* inputL, const float* inputU, const float* weight, int B, int CO, int CI, int G, int HW, float* outputL,
                        float* outputU, const float* shift, float sign, bool* shifted, sd_stream_t stream) {
    FwdArgs a;
    *shifted = false;
    SD_REQUIRE(inputU, "bound_inf_dist_forward_nograd: null upper input");
    int rc = make_fwd_args(a, "bound_inf_dist_forward_nograd", inputL, inputU, weight, B, CO, CI, G, HW,
                           nullptr, nullptr, 0, 0);
    if (rc) return rc;
    SD_REQUIRE(outputL && outputU, "bound_inf_dist_forward_nograd: null output");
    a.y0 = outputL; a.y1 = outputU;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (g_bound_density.load(std::memory_order_relaxed) <= 0.f && row_stream_ok(a, kStreamBoundTerms)) {
        a.shift = shift; a.shift_sign = sign;
        *shifted = true;
        return row_stream_bound(a, st);
    }
    // dense single-group layers: a kernel that works from per-weight-row candidate tables is queued in front of the
    // one that evaluates every term, and a count taken on the device decides which of the two runs
    const float bound_density = g_bound_density.load(std::memory_order_relaxed);
    const int bound_form = g_bound_form.load(std::memory_order_relaxed);
    const float cap = bound_density >= 0.f ? bound_density : kBoundColsCap;
    const FwdArgs raw = a;
    size_t copies = bound_pad(a, cap, B, CO, CI, G, HW);
    int tables = bound_tables_eligible(a, cap, B, CO, CI, G, HW);
    // The workspace is sized by shape alone (whatever the hints below decide), so that a call under graph capture, for
    // which they may decide otherwise, never needs more than the eager call before it did.
    char* wsbase = nullptr;
    size_t cbytes = 0;
    if (tables || copies) {
        const size_t both = !tables ? 0 : bound_tables_bytes(tables == 2, B, CO, CI), walk = tables == 2 && CI <= 65536 ? sort_cols_workspace(B, CO, CI) : 0;
        const size_t bytes = both > walk ? both : walk;
        cbytes = (bytes + 255) / 256 * 256;
        if ((bound_density < 0.f || copies) && !workspace_ready(cbytes + copies, st)) tables = 0;   // a first call under capture forms every term
        else if (!(wsbase = static_cast<char*>(workspace(cbytes + copies, st)))) return SD_ERR_HIP;   // the only request of this call
    }
    // with the built-in limit, a layer whose tables have not paid lately is not given any for a while
    const bool hinted = tables && bound_density < 0.f;
    if (hinted && !hint_build_tables(kHintSiteBound, weight, B, CO, CI, st, tables == 1)) tables = 0;
    if (copies) {
        // without tables the copies serve rows that could not be loaded 16 bytes at a time
        if (wsbase && (tables || !(raw.fast_x && raw.fast_w))) {
            if ((rc = bound_pad_copy(a, raw, wsbase + cbytes, st))) return rc;
        } else { a = raw; CI = raw.CIg; }
    }
    static const int kTb42[] = {4, 2};
    const bool narrow = narrow_tiles(a);
    const int TB = narrow ? 2 : pick_tb(a, kTb42, 2, 128);
    a.nsplit = pick_nsplit(a, 16 * TB, narrow ? 32 : 128);
    // Very few marks (weights of unit scale against rows that are alike: below 1 %): the staged kernel would spend its
    // time moving tiles through LDS, and the kernel that walks a weight row's marks over a transposed copy of the
    // inputs serves better.  Chosen by hand (sd_set_bound_candidate_form) or, with the built-in limit, for a layer
    // whose last three staged calls reported that few marks ("not building" the staged tables, in the hint's terms).
    bool sparse = tables == 2 && bound_form == 2 && CI <= 65536;
    if (tables == 2 && bound_form == 0 && hinted && CI <= 65536)
        sparse = !hint_build_tables(kHintSiteBoundSparse, weight, B, CO, CI, st);
    if (sparse) {
        void* ws = wsbase;
        if (a.nsplit > 1) {   // the every-term kernel, should it run, merges its slices into zeros
            if ((rc = fill_zero2(outputL, (size_t)B * CO * HW, outputU, (size_t)B * CO * HW, st))) return rc;
        }
        if ((rc = sort_cols_forward(a.x0, a.x1, a.w, B, CO, CI, 0.f, 1, outputL, outputU, nullptr, ws,
                                    bound_density > 0.f ? bound_density : kBoundSparseCap, &a.gate, &a.gate_limit, st)))
            return rc;
        a.gate_above = 1;
        return narrow ? launch_fwd<BoundNogradGated, 2, 2>(a, st) : TB == 2 ? launch_fwd<BoundNogradGated, 2, 8>(a, st) : launch_fwd<BoundNogradGated, 4, 8>(a, st);
    }
    if (a.nsplit > 1 || tables == 2) {
        if ((rc = fill_zero2(outputL, (size_t)B * CO * HW, outputU, (size_t)B * CO * HW, st))) return rc;
    }
    if (tables) {
        if ((rc = queue_bound_tables(a, tables == 2, B, CO, CI, cap, wsbase, st))) return rc;
        if (hinted) {
            a.told = hint_expect(kHintSiteBound, weight, B, CO, CI, st);
            if (tables == 2 && bound_form == 0) {   // 1: very few marks
                a.told2 = hint_expect(kHintSiteBoundSparse, weight, B, CO, CI, st);
                a.few = bound_cols_few(B, CO, CI, wsbase);
            }
        }
        rc = narrow ? launch_fwd<BoundNogradGated, 2, 2>(a, st) : TB == 2 ? launch_fwd<BoundNogradGated, 2, 8>(a, st) : launch_fwd<BoundNogradGated, 4, 8>(a, st);
        if (rc) { hint_forget(a.told); hint_forget(a.told2); }
        return rc;
    }
    if (narrow) return launch_fwd<BoundNograd, 2, 2>(a, st);
    if (TB == 2) return launch_fwd<BoundNograd, 2, 8>(a, st);
    return launch_fwd<BoundNograd, 4, 8>(a, st);
}

extern "C" int sd_bound_inf_dist_forward_nograd(const float* inputL, const float* inputU, const float* weight,
                                                int B, int CO, int CI, int G, int HW, float* outputL, float* outputU,
                                                sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    bool shifted;
    return bound_values(inputL, inputU, weight, B, CO, CI, G, HW, outputL, outputU, nullptr, 0.f, &shifted, stream);
}

extern "C" int sd_bound_inf_dist_forward_shifted(const float* inputL, const float* inputU, const float* weight,
                                                 int B, int CO, int CI, int G, int HW, float* outputL, float* outputU,
                                                 const float* shift, float sign, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    SD_REQUIRE(shift && (sign == 1.f || sign == -1.f), "bound_inf_dist_forward_shifted: null shift, or a sign (%g) other than 1 and -1",
               (double)sign);
    SD_REQUIRE(aligned16(shift) && aligned16(outputL) && aligned16(outputU), "bound_inf_dist_forward_shifted: shift and outputs must be 16-byte aligned");
    bool shifted;
    const int rc = bound_values(inputL, inputU, weight, B, CO, CI, G, HW, outputL, outputU, shift, sign, &shifted, stream);
    return rc || shifted ? rc : channel_shift_both(outputL, outputU, shift, B, CO, HW, sign, static_cast<hipStream_t>(stream));
}

extern "C" int sd_set_bound_candidate_density(float density) {
    SD_REQUIRE(density <= 1.f, "set_bound_candidate_density: %g is above 1", (double)density);
    g_bound_density = density;
    return SD_OK;
}

extern "C" int sd_set_bound_candidate_form(int form) {
    SD_REQUIRE(form >= 0 && form <= 2, "set_bound_candidate_form: %d is not 0 (automatic), 1 (staged tiles) or 2 (row walk)", form);
    g_bound_form = form;
    return SD_OK;
}

extern "C" int sd_bound_inf_dist_forward(const float* inputL, const float* inputU, const float* weight,
                                         int B, int CO, int CI, int G, int HW, float* outputL, float* outputU,
                                         int* posL, int* posU, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    FwdArgs a;
    SD_REQUIRE(inputU, "bound_inf_dist_forward: null upper input");
    int rc = make_fwd_args(a, "bound_inf_dist_forward", inputL, inputU, weight, B, CO, CI, G, HW,
                           nullptr, nullptr, 0, 0);
    if (rc) return rc;
    SD_REQUIRE(outputL && outputU && posL && posU, "bound_inf_dist_forward: null output or pos");
    a.y0 = outputL; a.y1 = outputU; a.p0 = posL; a.p1 = posU;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (g_bound_density.load(std::memory_order_relaxed) <= 0.f && row_stream_ok(a, kStreamBoundPosTerms)) return row_stream_bound(a, st);
    // dense single-group layers: the table kernel, tracking the chunk of every result, is queued in front
    // of the every-term kernel as for the forward without positions; both leave (value, chunk) pairs for the resolve
    const float bound_density = g_bound_density.load(std::memory_order_relaxed);
    const float cap = bound_density >= 0.f ? bound_density : kBoundPosColsCap;
    const FwdArgs raw = a;
    size_t copies = bound_pad(a, cap, B, CO, CI, G, HW);
    int tables = bound_tables_eligible(a, cap, B, CO, CI, G, HW);
    const size_t pairs = ((size_t)a.R * a.G * a.COg * 16 + 255) / 256 * 256;
    const size_t tbytes = tables ? (bound_tables_bytes(tables == 2, B, CO, CI) + 255) / 256 * 256 : 0;
    if ((tables || copies) && (bound_density < 0.f || copies) && !workspace_ready(pairs + tbytes + copies, st)) {   // a first call under capture
        tables = 0;
        if (copies) { a = raw; CI = raw.CIg; copies = 0; }
    }
    const bool elig = tables || copies;   // by shape alone: what the workspace is sized by (a captured call may build tables that an eager one does not)
    const bool hinted = tables && bound_density < 0.f;
    if (hinted && !hint_build_tables(kHintSiteBoundPos, weight, B, CO, CI, st, tables == 1)) tables = 0;
    const bool copied = copies && (tables || !(raw.fast_x && raw.fast_w));   // (as without positions)
    if (copies && !copied) { a = raw; CI = raw.CIg; }
    static const int kTb42[] = {4, 2};
    const bool narrow = narrow_tiles(a);
    const int TB = narrow ? 2 : pick_tb(a, kTb42, 2, 64);
    a.nsplit = pick_nsplit(a, 16 * TB, narrow ? 32 : 64);
    if (a.nsplit > 1 && !workspace_ready((size_t)a.R * a.G * a.COg * 16, st)) { a.coarse = 1; a.nsplit = pick_nsplit(a, 16 * TB, narrow ? 32 : 64); }
    if (tables == 2 && a.nsplit < 2) a.nsplit = 2;   // both kernels merge into the packed pairs
    if (a.nsplit > 1 || elig) {
        size_t n = (size_t)a.R * a.G * a.COg;
        char* ws = static_cast<char*>(workspace(pairs + (elig ? tbytes + copies : 0), st));   // the only request
        if (!ws) return SD_ERR_HIP;
        if (copied && (rc = bound_pad_copy(a, raw, ws + pairs + tbytes, st))) return rc;
        a.packed0 = reinterpret_cast<unsigned long long*>(ws);
        a.packed1 = a.packed0 + n;
        if (a.nsplit > 1 && (rc = fill_zero(a.packed0, n * 4, st))) return rc;
        if (tables && (rc = queue_bound_tables(a, tables == 2, B, CO, CI, cap, ws + pairs, st))) return rc;
    }
    if (hinted && tables) a.told = hint_expect(kHintSiteBoundPos, weight, B, CO, CI, st);
    // exact dense tiles: the LDS-direct kernel with the chunk numbers packed (same (value, chunk) pairs, same resolve)
    if (TB == 4 && a.nsplit > 1 && direct_ok<4, 4>(a) && (a.CIg / KT + a.nsplit - 1) / a.nsplit <= BoundChunkPacked::MAX_CHUNKS)
        rc = launch_fwd_direct<BoundChunkPacked, 4, 4>(a, st);
    else rc = narrow ? launch_fwd<BoundChunk, 2, 2>(a, st) : TB == 2 ? launch_fwd<BoundChunk, 2, 4>(a, st) : launch_fwd<BoundChunk, 4, 4>(a, st);
    if (rc) { hint_forget(a.told); return rc; }
    return launch_resolve_bound(a, st);
}
