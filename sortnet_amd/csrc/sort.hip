// Sort-neuron forward entry points (top-K order statistics with geometric weights), K = 2..25 as
// in the reference's instantiation table (core/cuda/sort_neuron.cu:403-534).
#include "fwd_tile.h"
#include "fwd_args.h"
#include "sort_cols.h"
#include "row_cands.h"
#include "row_stream.h"
#include <atomic>

using namespace sd;

#define SD_FOR_EACH_K(X) \
    X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) X(17) \
    X(18) X(19) X(20) X(21) X(22) X(23) X(24) X(25)

static int check_qk(const char* who, float q, int K, int CIg) {
    SD_REQUIRE(K >= 2 && K <= 25, "%s: K=%d outside 2..25", who, K);
    SD_REQUIRE(q > 0.f && q <= 1.f, "%s: q=%g outside (0, 1]", who, (double)q);
    (void)CIg;
    return SD_OK;
}

// Second pass of the two-level sort neuron.  One workgroup per weight row: the row is staged in LDS once
// (chunks of KT floats, each followed by 4 floats of padding so that work-items reading different chunks hit
// different banks) and every work-item resolves one output of that row at a time, reading the candidate
// chunks of its input row (128-bit loads) against the staged weights.  VALUES: the K largest candidate values
// by branch-free insertion; otherwise the reference's ordered insertion with indices over the candidates in
// ascending input order (the chunk numbers are sorted first), which ends in the same list as the scan over
// all inputs because every left-out term is smaller than the final K-th value.
constexpr int kSortRowMax = 12288;   // inputs per weight row this path stages
constexpr int kChunkPad = KT + 4;

template <int K, bool VALUES>
__global__ void __launch_bounds__(256) sort_rows_kernel(FwdArgs a, const int* __restrict__ keys) {
    constexpr int KP = K + kKeySlack;
    extern __shared__ __attribute__((aligned(16))) float wrow[];
    if (gate_closed(a.gate, a.gate_limit, a.gate_above)) return;   // one of two queued for the result
    const int c = blockIdx.x;                      // g * COg + m
    const int g = c / a.COg;
    const float* wsrc = a.w + (size_t)c * a.CIg;
    for (int n = threadIdx.x * 4; n < a.CIg; n += 1024)
        *reinterpret_cast<float4*>(wrow + (n / KT) * kChunkPad + (n % KT)) = *reinterpret_cast<const float4*>(wsrc + n);
    __syncthreads();
    const size_t size = (size_t)a.B * a.G * a.COg;
    const int nchunks = (a.CIg + KT - 1) / KT;
    const float sh = VALUES ? output_shift(a.shift, a.shift_sign, c) : 0.f;
    for (int b = threadIdx.x; b < a.B; b += 256) {
        const size_t o = (size_t)b * a.G * a.COg + c;
        const float* xr = a.x0 + (size_t)(b * a.G + g) * a.CIg;
        float res[K];
        int idx[K];
        #pragma unroll
        for (int k = 0; k < K; k++) { res[k] = 0.f; idx[k] = 0; }
        auto chunk = [&](int cid) {
            const int n0 = cid * KT;
            const float* wc = wrow + cid * kChunkPad;
            #pragma unroll
            for (int q4 = 0; q4 < KT / 4; q4++) {
                int n = n0 + 4 * q4;
                const bool in = n < a.CIg;           // CIg is a multiple of 4 on this path
                if (!in) n = a.CIg - 4;
                const float4 xv = *reinterpret_cast<const float4*>(xr + n);
                const float4 wv = *reinterpret_cast<const float4*>(wc + (n - n0));
                const float d[4] = {xv.x - wv.x, xv.y - wv.y, xv.z - wv.z, xv.w - wv.w};
                #pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float v = in ? fabsf(d[e]) : 0.f;
                    if (VALUES) topk_insert_values<K>(res, v);
                    else if (v > res[0]) topk_insert<K>(res, idx, v, (n + e) | (d[e] >= 0.f ? 0 : (int)kSign));
                }
            }
        };
        uint32_t key[KP];
        #pragma unroll
        for (int k = 0; k < KP; k++) key[k] = (uint32_t)keys[((size_t)k * a.G * a.COg + c) * a.B + b];
        // keys ascend: key[KP - K] is the K-th largest; chunks whose truncated maximum reaches it are candidates
        const uint32_t cut = key[KP - K] >> kKeyIdBits;
        if (cut != 0u && (key[0] >> kKeyIdBits) == cut) {
            for (int cid = 0; cid < nchunks; cid++) chunk(cid);     // too many chunks share the cut value
        } else {
            int ids[KP];
            #pragma unroll
            for (int k = 0; k < KP; k++) {
                const uint32_t bucket = key[k] >> kKeyIdBits;
                ids[k] = (bucket != 0u && bucket >= cut) ? (int)(key[k] & ((1u << kKeyIdBits) - 1u)) : 0x7fffffff;
            }
            if (!VALUES) {
                // ascending chunk numbers (odd-even transposition network; skipped slots sort to the end)
                #pragma unroll
                for (int i = 0; i < KP; i++) {
                    #pragma unroll
                    for (int k = i & 1; k + 1 < KP; k += 2) {
                        int lo = min(ids[k], ids[k + 1]), hi = max(ids[k], ids[k + 1]);
                        ids[k] = lo; ids[k + 1] = hi;
                    }
                }
            }
            #pragma unroll
            for (int k = 0; k < KP; k++) {
                if (ids[k] < nchunks) chunk(ids[k]);
            }
        }
        a.y0[o] = geo_sum<K>(res, a.q) + sh;
        if (!VALUES) {
            #pragma unroll
            for (int k = K - 1; k >= 0; k--) a.p0[(size_t)(K - 1 - k) * size + o] = idx[k];
        }
    }
}

// two-level path: dense vector-load case with a reduction long enough for the chunk lists to pay
static bool two_level_ok(const FwdArgs& a, int K) {
    const int nchunks = (a.CIg + KT - 1) / KT;
    return a.HW == 1 && a.fast_x && a.fast_w && a.CIg <= kSortRowMax && K <= 12 && nchunks >= 4 * K &&
           nchunks <= (1 << kKeyIdBits);
}

// bytes of the two-level path's key lists
static inline size_t align256(size_t b) { return (b + 255) / 256 * 256; }
static size_t two_level_bytes(const FwdArgs& a, int K) {
    return (size_t)(K + kKeySlack) * ((size_t)a.R * a.G * a.COg) * sizeof(int);
}

// `keys`: two_level_bytes() of workspace
template <int K, bool VALUES>
static int run_two_level(FwdArgs& a, bool small, int* keys, hipStream_t st) {
    FwdArgs t = a;
    t.p0 = keys;
    int rc = small ? launch_fwd<SortChunkKeys<K>, 1, 2>(t, st) : launch_fwd<SortChunkKeys<K>, 2, 4>(t, st);
    if (rc) return rc;
    const int nchunks = (a.CIg + KT - 1) / KT;
    hipLaunchKernelGGL((sort_rows_kernel<K, VALUES>), dim3((unsigned)(a.G * a.COg)), dim3(256),
                       (size_t)nchunks * kChunkPad * sizeof(float), st, a, keys);
    return check_launch("sort_rows_kernel");
}

// Dense single-group layers: a kernel that works from per-weight-row candidate tables is queued in front of the
// kernels that evaluate every term, and a count taken on the device decides which of the two runs (at most
// sort_cols_cap of the terms marked: the table kernel).  Negative g_sort_density: built-in limit, and only layers
// large enough for the tables to pay; 0 never; up to 1: that share, at any size.
static std::atomic<float> g_sort_density{-1.f};
// Every term / tables, us, by the marked share (activations of growing spread against unit weights, K = 10).  The time
// follows the marks that are left after a wavefront has cut its list, so the two meet late; positions, which walk their strong
// marks twice, meet first where a batch tile is not full.
//   values       512 x 5120 x 5120 1809 / 394 (12 %), 1813 / 766 (43 %), 1797 / 1212 (91 %); 256 x 2048 x 512 101 / 74 (21 %),
//                100 / 114 (61 %); 512 x 768 x 640 109 / 70 (36 %)
//   interval     512 x 5120 x 5120 3901 / 702 (14 %), 4120 / 1448 (47 %); 256 x 2048 x 512 241 / 106 (23 %), 252 / 169 (66 %)
//   positions    512 x 5120 x 5120 2447 / 818 (12 %), 2471 / 1592 (43 %); 128 x 5120 x 5120 583 / 305 (12 %), 600 / 561 (43 %);
//                256 x 2048 x 512 139 / 125 (21 %), 143 / 204 (61 %); 96 x 5120 x 300 216 / 150 (11 %), 220 / 256 (38 %)
// Smallest layers that have no kernel of their own (row_stream_sort_ok), values: 100 x 480 x 450 48 / 30 (15 %), 49 / 36 (39 %); 72 x
// 1024 x 1024 94 / 40 (23 %), 95 / 54 (49 %); 16 x 4096 x 4128 183 / 130 (29 %); 300 x 320 x 256 34 / 32 (20 %), 35 / 37 (47 %).  Rows of
// 256 inputs are formed before the tables are done: 512 x 256 x 256 30 / 35 (26 %), 256 x 256 x 300 29 / 31 (25 %).
static float sort_cols_cap(int form, int CI) {
    return form == kRowsSortPos ? 0.22f : form == kRowsSortValues && CI < 320 ? 0.10f : 0.40f;
}
constexpr long long kSortColsMinTerms = 1ll << 24;
// Positions have no kernel that streams the weights, and every term of a few outputs is formed by few wavefronts: tables from 2^20 terms on
// where rows are at least 320 inputs long.  Every term -> tables at spreads 0.05 / 0.3 of the inputs, K = 10: 99 x 2304 x 59 107 -> 36, 121 -> 66; 50 x
// 1000 x 64 238 -> 36, 286 -> 57; 128 x 5120 x 10 180 -> 39, 198 -> 82; 16 x 320 x 250 112 -> 33; where they do not serve (64 x 512 x 64 at
// 0.3, 185 us) building them takes 18 us, for one call in 32.
constexpr long long kSortPosMinTerms = 1ll << 20;
static long long sort_cols_min_terms(bool pos, int CI) { return pos && CI >= 320 ? kSortPosMinTerms : kSortColsMinTerms; }

// `site`: which entry point asks (with the built-in limit, a layer whose tables have not paid lately is not given
// any for a while, see hint_build_tables)
constexpr int kHintSiteSort = 2, kHintSiteBoundSort = 3, kHintSiteSortPos = 6;
constexpr int kHintSiteBox = 16;    // tables for values and bounds together
constexpr int kHintSiteRows = 10;   // and with the form added: whether the tables per batch row served
// shape and size alone: the workspace is sized by this, so that a call under graph capture (which always builds
// tables) never needs more than the eager call before it did
static bool sort_cols_eligible(const FwdArgs& a, bool pos, int B, int CO, int CI, int G, int HW) {
    const float density = g_sort_density.load(std::memory_order_relaxed);
    // the mark lists of the table kernels hold 16-bit input numbers
    if (density == 0.f || G != 1 || HW != 1 || CI % kSortColsChunk != 0 || CI > 65536 || !a.fast_x || !a.fast_w) return false;
    return density > 0.f || (long long)B * CO * CI >= sort_cols_min_terms(pos, CI);
}
// eligible, and (with the built-in limit) the layer's tables have paid lately
static bool sort_cols_ok(const float* weight, int site, int B, int CO, int CI, hipStream_t st) {
    return g_sort_density.load(std::memory_order_relaxed) > 0.f || hint_build_tables(site, weight, B, CO, CI, st);
}
// before the every-term kernels are queued behind the table kernel: where they report
static void sort_cols_expect(FwdArgs& a, const float* weight, int site, int B, int CO, int CI, hipStream_t st) {
    if (g_sort_density.load(std::memory_order_relaxed) < 0.f && a.gate) a.told = hint_expect(site, weight, B, CO, CI, st);
}

// Largest share of marked (tile of 128 weight rows, batch row, input) triples at which the kernel of the tables per
// batch row runs.  Every term / tables, us, on inputs in [0, 1] against weights of growing scale, K = 10:
//   values       512 x 5120 x 5120 1714 / 416 (7 %), 1763 / 905 (27 %); 128 x 3072 x 1024 132 / 90 (9 %), 130 / 117 (27 %), 131 / 151 (35 %)
//   interval     512 x 5120 x 5120 3225 / 675 (9 %), 3993 / 2025 (42 %); 128 x 3072 x 1024 312 / 116 (11 %), 335 / 217 (41 %); 64 x 2048 x 2048
//                231 / 152 (35 %), 237 / 188 (51 %)
//   positions    512 x 5120 x 5120 2332 / 778 (7 %), 2443 / 1748 (27 %); 128 x 3072 x 1024 182 / 132 (9 %), 179 / 176 (18 %)
static float sort_rows_cap(int form) { return form == kRowsSortInterval ? 0.45f : form == kRowsSortValues ? 0.27f : 0.22f; }
// Smallest layers (in terms) given tables per batch row under the built-in limit (128 x 3072 x 1024, 0.4 G terms:
// values 0.12 ms from tables against 0.14 ms for every term, with positions 0.16 against 0.19, interval bounds 0.17
// against 0.32)
constexpr long long kSortRowsMinTerms = 1ll << 28;

// bytes of both tables' workspace for one call: per weight row first (with the probe and the counter the per-batch-row
// tables read), per batch row behind it
static size_t sort_tables_bytes(int form, int B, int CO, int CI, int K) {
    const size_t cols = (sort_cols_workspace(B, CO, CI) + 255) / 256 * 256;
    return cols + (row_cands_supported(form, K) ? (row_cands_workspace(form, B, CO, CI) + 255) / 256 * 256 : 0);
}

// One table for the values and the bounds of a layer, and its kernel (sort_cols_box_tables, sort_cols_box_main), queued for both before either.
// own: the values' own tables behind it, for a layer that it does not serve.
struct SortBox {
    const unsigned long long* count;
    unsigned long long limit;
    void* ws;
    char* rest;             // workspace of the two forms, one after the other
    const float* layer;     // the weights as the caller has them, which the hints know the layer by
    bool own;
    bool own_tables(int form) const { return own && form == kRowsSortValues; }
};

// `ws`: sort_tables_bytes() bytes.  The gate it leaves in `a` points into `ws`: the kernels queued behind it must
// not be given memory that overlaps it, and `ws` must stay allocated until they have run (one workspace request
// per call, carved by the caller).  Afterwards a.gate[0] is non-zero when the every-term kernels are to run.
// A layer that the tables per weight row serve queues those per batch row in vain, three kernels that return at once (4.6 us each): where
// they ran in none of three calls they are left out of the next 31, unless the call before formed every term (hint_build_spare;
// evaluation pass of 6 x 5120 at batch 512 1636 -> 1575 us, attack on 128 x 5120 x 5120 225 -> 215).  `site`, `layer`: see sort_cols_ok;
// with a box it is the shared table that serves, or the values' own one beside it, and `site` hears only of tables that the call builds.
static int queue_sort_cols(FwdArgs& a, int site, const float* layer, int form, const float* xl, const float* xu, const float* w, int B, int CO, int CI,
                           float q, int K, float* outL, float* outU, int* pos, void* ws, const SortBox* box, hipStream_t st) {
    const float density = g_sort_density.load(std::memory_order_relaxed);
    const float cap = density > 0.f ? density : sort_cols_cap(form, CI);
    int rc = SD_OK;
    if (box) {
        a.gate = box->count;
        a.gate_limit = box->limit;
    }
    if (!rc && (!box || box->own_tables(form)))
        rc = sort_cols_forward(xl, xu, w, B, CO, CI, q, K, outL, outU, pos, ws, cap, &a.gate, &a.gate_limit, st, a.shift, a.shift_sign, box ? box->count : nullptr);
    a.gate_above = 1;
    const long long terms = (long long)B * CO * CI;
    auto served = [&] {
        if (box && !box->own_tables(form)) return hint_paid(kHintSiteBox, layer, B, CO, CI);
        return hint_paid(site, layer, B, CO, CI);
    };
    const bool rows = row_cands_supported(form, K) && (density > 0.f || terms >= kSortRowsMinTerms) &&
                      (density > 0.f || hint_build_spare(kHintSiteRows + form, layer, B, CO, CI, st, served()));
    if (rc || !rows) {
        // the every-term kernels read the flag behind the counter, as with both tables
        if (!rc) { a.gate = a.gate + 1; a.gate_limit = 0ull; }
        return rc;
    }
    const unsigned long long* col_count = a.gate;
    char* rows_ws = static_cast<char*>(ws) + (sort_cols_workspace(B, CO, CI) + 255) / 256 * 256;
    const unsigned long long* every = nullptr;
    rc = row_cands_forward(form, xl, xu, w, nullptr, nullptr, B, CO, CI, q, K, outL, outU, pos, rows_ws,
                           density > 0.f ? density : sort_rows_cap(form), density > 0.f, sort_cols_probe_sums(col_count), col_count, &every, st, nullptr, a.shift, a.shift_sign);
    if (rc) return rc;
    a.gate = every;
    a.gate_limit = 0ull;
    if (density < 0.f) {
        a.told2 = hint_expect(kHintSiteRows + form, layer, B, CO, CI, st);
        a.few = row_cands_idle(every);
    }
    note_term_counts(every - 1, 3, (double)((CO + 127) / 128) * B * CI, (double)((B + 127) / 128) * CO * CI);
    return SD_OK;
}

// Layers whose rows are no whole number of table words (32 inputs) work on copies of inputs and weights with zeros behind every
// row: a term of 0 enters no list.  The kernels that form every term then load 16 bytes at a time, too; rows that did so anyway
// are only copied for a call that builds tables.  Sets the shape of `a` and CI to the copies' and returns their bytes, or 0 (as they
// were) where there are too few terms for tables.
// In us, without copies -> with them, inputs of spread 0.05 / 0.3 / 3 against unit weights, K = 10:
//   values       128 x 1306 x 1306 160 -> 34 / 56 / 146, 250 x 3071 x 500 160 -> 42 / 70 / 108, 512 x 5001 x 2000 1660 -> 77 / 167 / 288
//   interval     128 x 1306 x 1306 258 -> 38 / 70 / 190, 14 x 4443 x 4443 668 -> 85 / 123 / 204, 512 x 5001 x 2000 2602 -> 96 / 258 / 450
//   positions    128 x 1306 x 1306 310 -> 45 / 153 / 179, 8 x 2198 x 2198 372 -> 51 / 65 / 152, 99 x 2303 x 59 450 -> 41 / 74 / 106
static size_t sort_pad(FwdArgs& a, bool pos, int B, int CO, int& CI, int G, int HW) {
    const int N = (CI + kSortColsChunk - 1) / kSortColsChunk * kSortColsChunk;
    if (N == CI || G != 1 || HW != 1 || N > 65536 || (long long)(B + CO) * N >= (1ll << 31) || 2ll * B + CO > 4 * 65535) return 0;
    const float density = g_sort_density.load(std::memory_order_relaxed);
    if (density == 0.f || (density < 0.f && (long long)B * CO * CI < sort_cols_min_terms(pos, N))) return 0;
    CI = a.CIg = a.W_CIg = N;
    a.fast_x = a.fast_w = 1;
    const size_t x = ((size_t)B * N * 4 + 255) / 256 * 256;
    return (a.x1 ? 2 : 1) * x + ((size_t)CO * N * 4 + 255) / 256 * 256;
}
// makes the copies; `raw`: the call's own operands
static int sort_pad_copy(FwdArgs& a, const FwdArgs& raw, void* mem, hipStream_t st) {
    const size_t x = ((size_t)a.B * a.CIg * 4 + 255) / 256 * 256;
    char* p = static_cast<char*>(mem);
    float* x0 = reinterpret_cast<float*>(p);
    float* x1 = a.x1 ? reinterpret_cast<float*>(p + x) : x0;
    float* w = reinterpret_cast<float*>(p + (a.x1 ? 2 : 1) * x);
    const int rc = pad_rows({raw.x0, raw.x1, raw.w}, {x0, x1, w}, {a.B, a.x1 ? a.B : 0, a.COg}, raw.CIg, a.CIg, st);
    a.x0 = x0;
    if (a.x1) a.x1 = x1;
    a.w = w;
    return rc;
}

// what a call does that has copies planned but builds no tables: whether it goes on without them
static bool sort_unpad(FwdArgs& a, const FwdArgs& raw, int& CI, bool tables) {
    if (tables || !(raw.fast_x && raw.fast_w)) return false;
    a = raw;
    CI = raw.CIg;
    return true;
}

extern "C" int sd_set_sort_candidate_density(float density) {
    SD_REQUIRE(density <= 1.f, "set_sort_candidate_density: %g is above 1", (double)density);
    g_sort_density = density;
    return SD_OK;
}

// few output tiles: 16 x 32 tiles instead of 32 x 64 (the top-K lists do not merge across a split reduction)
static bool few_tiles(const FwdArgs& a, int BB, int BM) {
    long long tiles = (long long)((a.R + BB - 1) / BB) * ((a.COg + BM - 1) / BM) * a.G;
    return tiles < 2ll * num_cus();
}

static int sort_values(const float* input, const float* weight, int B, int CO, int CI, int G, int HW, float* output, float q, int K,
                       const float* shift, float sign, const SortBox* box, sd_stream_t stream) {
    FwdArgs a;
    int rc = make_fwd_args(a, "sort_neuron_forward_nograd", input, nullptr, weight, B, CO, CI, G, HW, nullptr, nullptr, 0, 0);
    if (rc) return rc;
    if ((rc = check_qk("sort_neuron_forward_nograd", q, K, a.CIg))) return rc;
    SD_REQUIRE(output, "sort_neuron_forward_nograd: null output");
    a.y0 = output; a.q = q; a.shift = shift; a.shift_sign = sign;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (!box && g_sort_density.load(std::memory_order_relaxed) <= 0.f && row_stream_sort_ok(a))
        return row_stream_sort(a, K, st);
    const bool small = few_tiles(a, 32, 64), streamed = !box && g_sort_density.load(std::memory_order_relaxed) <= 0.f && row_stream_sort_before_terms(a);
    const FwdArgs raw = a;
    size_t copies = sort_pad(a, false, B, CO, CI, G, HW);
    if (copies && !workspace_ready(sort_tables_bytes(kRowsSortValues, B, CO, CI, K) + (two_level_ok(a, K) ? align256(two_level_bytes(a, K)) : 0) + copies, st)) {
        a = raw; CI = raw.CIg; copies = 0;
    }
    const bool two = K <= 12 && two_level_ok(a, K), elig = box || sort_cols_eligible(a, false, B, CO, CI, G, HW);
    const float* layer = box ? box->layer : weight;
    const bool cols = box || (elig && sort_cols_ok(layer, kHintSiteSort, B, CO, CI, st));
    if (streamed && !elig) return row_stream_sort(a, K, st);
    // one request for both users of the workspace: the tables (with the counter the gates read) first, the key
    // lists of the two-level path behind them
    const size_t tbytes = elig ? sort_tables_bytes(kRowsSortValues, B, CO, CI, K) : 0, kbytes = two ? align256(two_level_bytes(a, K)) : 0;
    char* base = nullptr;
    if (box) base = box->rest;
    else if (elig || two) {
        base = static_cast<char*>(workspace(tbytes + kbytes + copies, st));
        if (!base) return SD_ERR_HIP;
    }
    if (streamed && !cols) return row_stream_sort(raw, K, st);
    if (copies && !sort_unpad(a, raw, CI, cols) && (rc = sort_pad_copy(a, raw, base + tbytes + kbytes, st))) return rc;
    int* keys = reinterpret_cast<int*>(base + tbytes);
    if (cols && (rc = queue_sort_cols(a, kHintSiteSort, layer, kRowsSortValues, a.x0, nullptr, a.w, B, CO, CI, q, K, nullptr, output, nullptr, base, box, st))) return rc;
    if (cols && (!box || box->own)) sort_cols_expect(a, layer, kHintSiteSort, B, CO, CI, st);
    if (box && g_sort_density.load(std::memory_order_relaxed) < 0.f) {
        a.told3 = hint_expect(kHintSiteBox, layer, B, CO, CI, st);
        a.few3 = box->count + 1;
    }
    rc = SD_ERR_ARG;
    switch (K) {
#define X(k) case k: if (k <= 12 && two) rc = run_two_level<(k <= 12 ? k : 2), true>(a, small, keys, st); \
                     else rc = small ? launch_fwd<SortNograd<k>, 1, 2>(a, st) : launch_fwd<SortNograd<k>, 2, 4>(a, st); \
                     break;
        SD_FOR_EACH_K(X)
#undef X
    }
    if (rc) { hint_forget(a.told); hint_forget(a.told2); hint_forget(a.told3); }
    return rc;
}

extern "C" int sd_sort_neuron_forward_nograd(const float* input, const float* weight,
                                             int B, int CO, int CI, int G, int HW, float* output, float q, int K,
                                             sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    return sort_values(input, weight, B, CO, CI, G, HW, output, q, K, nullptr, 0.f, nullptr, stream);
}

extern "C" int sd_sort_neuron_forward_shifted(const float* input, const float* weight,
                                              int B, int CO, int CI, int G, int HW, float* output, float q, int K,
                                              const float* shift, float sign, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    SD_REQUIRE(shift && (sign == 1.f || sign == -1.f), "sort_neuron_forward_shifted: null shift, or a sign (%g) other than 1 and -1", (double)sign);
    return sort_values(input, weight, B, CO, CI, G, HW, output, q, K, shift, sign, nullptr, stream);
}

extern "C" int sd_sort_neuron_forward(const float* input, const float* weight,
                                      int B, int CO, int CI, int G, int HW, float* output, int* pos, float q, int K,
                                      sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    FwdArgs a;
    int rc = make_fwd_args(a, "sort_neuron_forward", input, nullptr, weight, B, CO, CI, G, HW, nullptr, nullptr, 0, 0);
    if (rc) return rc;
    if ((rc = check_qk("sort_neuron_forward", q, K, a.CIg))) return rc;
    SD_REQUIRE(output && pos, "sort_neuron_forward: null output or pos");
    SD_REQUIRE((long long)K * B * CO * HW < (1ll << 31), "sort_neuron_forward: pos too large for 32-bit indexing");
    a.y0 = output; a.p0 = pos; a.q = q;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool small = few_tiles(a, 32, 32);
    const FwdArgs raw = a;
    size_t copies = sort_pad(a, true, B, CO, CI, G, HW);
    const bool vectors = K <= 12 && two_level_ok(a, K);
    bool elig = sort_cols_eligible(a, true, B, CO, CI, G, HW);
    // (what was formed without scratch, or with the key lists alone, can be captured unprepared)
    if (elig && (copies || (long long)B * CO * CI < kSortColsMinTerms) &&
        !workspace_ready(sort_tables_bytes(kRowsSortPos, B, CO, CI, K) + (vectors ? align256(two_level_bytes(a, K)) : 0) + copies, st)) {
        elig = false;
        a = raw; CI = raw.CIg; copies = 0;
    }
    const bool two = K <= 12 && two_level_ok(a, K);
    const bool cols = elig && sort_cols_ok(weight, kHintSiteSortPos, B, CO, CI, st);
    // one request for both users of the workspace, as in sd_sort_neuron_forward_nograd
    const size_t tbytes = elig ? sort_tables_bytes(kRowsSortPos, B, CO, CI, K) : 0, kbytes = two ? align256(two_level_bytes(a, K)) : 0;
    char* base = nullptr;
    if (elig || two) {
        base = static_cast<char*>(workspace(tbytes + kbytes + copies, st));
        if (!base) return SD_ERR_HIP;
    }
    if (copies && !sort_unpad(a, raw, CI, cols) && (rc = sort_pad_copy(a, raw, base + tbytes + kbytes, st))) return rc;
    int* keys = reinterpret_cast<int*>(base + tbytes);
    if (cols && (rc = queue_sort_cols(a, kHintSiteSortPos, weight, kRowsSortPos, a.x0, nullptr, a.w, B, CO, CI, q, K, nullptr, output, pos, base, nullptr, st))) return rc;
    if (cols) sort_cols_expect(a, weight, kHintSiteSortPos, B, CO, CI, st);
    rc = SD_ERR_ARG;
    switch (K) {
#define X(k) case k: if (k <= 12 && two) rc = run_two_level<(k <= 12 ? k : 2), false>(a, few_tiles(a, 32, 64), keys, st); \
                     else rc = small ? launch_fwd<SortPos<k>, 1, 2>(a, st) : launch_fwd<SortPos<k>, 2, 2>(a, st); \
                     break;
        SD_FOR_EACH_K(X)
#undef X
    }
    if (rc) { hint_forget(a.told); hint_forget(a.told2); }
    return rc;
}

static int sort_bounds(const float* inputL, const float* inputU, const float* weight, int B, int CO, int CI, int G, int HW, float* outputL,
                       float* outputU, float q, int K, const float* shift, float sign, const SortBox* box, sd_stream_t stream) {
    FwdArgs a;
    SD_REQUIRE(inputU, "bound_sort_neuron_forward: null upper input");
    int rc = make_fwd_args(a, "bound_sort_neuron_forward", inputL, inputU, weight, B, CO, CI, G, HW, nullptr, nullptr, 0, 0);
    if (rc) return rc;
    if ((rc = check_qk("bound_sort_neuron_forward", q, K, a.CIg))) return rc;
    SD_REQUIRE(outputL && outputU, "bound_sort_neuron_forward: null output");
    a.y0 = outputL; a.y1 = outputU; a.q = q; a.shift = shift; a.shift_sign = sign;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (!box && g_sort_density.load(std::memory_order_relaxed) <= 0.f && row_stream_sort_ok(a))
        return row_stream_sort(a, K, st);
    const bool small = few_tiles(a, 32, 32);
    const FwdArgs raw = a;
    size_t copies = sort_pad(a, false, B, CO, CI, G, HW);
    if (copies && !workspace_ready(sort_tables_bytes(kRowsSortInterval, B, CO, CI, K) + copies, st)) { a = raw; CI = raw.CIg; copies = 0; }
    const bool elig = box || sort_cols_eligible(a, false, B, CO, CI, G, HW);
    const float* layer = box ? box->layer : weight;
    const bool cols = box || (elig && sort_cols_ok(layer, kHintSiteBoundSort, B, CO, CI, st));
    const bool streamed = !cols && g_sort_density.load(std::memory_order_relaxed) <= 0.f && row_stream_sort_before_terms(raw);
    if (elig) {
        const size_t tbytes = sort_tables_bytes(kRowsSortInterval, B, CO, CI, K);
        char* ws = box ? box->rest : static_cast<char*>(workspace(tbytes + copies, st));   // the only request of this call
        if (!ws) return SD_ERR_HIP;
        if (copies && !streamed && !sort_unpad(a, raw, CI, cols) && (rc = sort_pad_copy(a, raw, ws + tbytes, st))) return rc;
        if (cols && (rc = queue_sort_cols(a, kHintSiteBoundSort, layer, kRowsSortInterval, a.x0, a.x1, a.w, B, CO, CI, q, K, outputL, outputU, nullptr, ws, box, st))) return rc;
    }
    if (streamed) return row_stream_sort(raw, K, st);
    if (cols && !box) sort_cols_expect(a, layer, kHintSiteBoundSort, B, CO, CI, st);
    rc = SD_ERR_ARG;
    switch (K) {
#define X(k) case k: rc = small ? launch_fwd<BoundSort<k>, 1, 2>(a, st) : launch_fwd<BoundSort<k>, 2, 2>(a, st); break;
        SD_FOR_EACH_K(X)
#undef X
    }
    if (rc) { hint_forget(a.told); hint_forget(a.told2); }
    return rc;
}

extern "C" int sd_bound_sort_neuron_forward(const float* inputL, const float* inputU, const float* weight,
                                            int B, int CO, int CI, int G, int HW, float* outputL, float* outputU,
                                            float q, int K, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    return sort_bounds(inputL, inputU, weight, B, CO, CI, G, HW, outputL, outputU, q, K, nullptr, 0.f, nullptr, stream);
}

extern "C" int sd_bound_sort_neuron_forward_shifted(const float* inputL, const float* inputU, const float* weight,
                                                    int B, int CO, int CI, int G, int HW, float* outputL, float* outputU,
                                                    float q, int K, const float* shift, float sign, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    SD_REQUIRE(shift && (sign == 1.f || sign == -1.f), "bound_sort_neuron_forward_shifted: null shift, or a sign (%g) other than 1 and -1",
               (double)sign);
    return sort_bounds(inputL, inputU, weight, B, CO, CI, G, HW, outputL, outputU, q, K, shift, sign, nullptr, stream);
}

// Values and bounds of one layer.  Where both would be given tables per weight row they share one, and one walk: at 512 x 5120 x 5120, K = 10,
// ranges and table take 59 us where those of the two forms took 102, the walk 192 where theirs took 203 (certification of 6 x 5120 at batch 512
// 1503 -> 1406 us with the table, 1347 with the walk).  A layer whose shared table does not serve (intervals so wide that they
// mark nearly everything) goes on as the two calls by themselves: the values' own tables are queued behind the shared one, and return at
// once where that serves, until it has in several calls; where it did not in three calls it is left out of the next 31.
static int sort_box(const float* input, const float* inputL, const float* inputU, const float* weight, int B, int CO, int CI, int G, int HW,
                    float* output, float* outputL, float* outputU, float q, int K, const float* shift, float sign, sd_stream_t stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto apart = [&]() {
        const int rc = sort_values(input, weight, B, CO, CI, G, HW, output, q, K, shift, sign, nullptr, stream);
        return rc ? rc : sort_bounds(inputL, inputU, weight, B, CO, CI, G, HW, outputL, outputU, q, K, shift, sign, nullptr, stream);
    };
    FwdArgs v, b;
    int rc = make_fwd_args(v, "sort_neuron_box_forward", input, nullptr, weight, B, CO, CI, G, HW, nullptr, nullptr, 0, 0);
    if (rc) return rc;
    if ((rc = make_fwd_args(b, "sort_neuron_box_forward", inputL, inputU, weight, B, CO, CI, G, HW, nullptr, nullptr, 0, 0))) return rc;
    if ((rc = check_qk("sort_neuron_box_forward", q, K, v.CIg))) return rc;
    SD_REQUIRE(inputU && output && outputL && outputU, "sort_neuron_box_forward: null upper input or output");
    const float density = g_sort_density.load(std::memory_order_relaxed);
    const FwdArgs raw = v;
    int N = CI, NB = CI;
    const size_t copies = sort_pad(v, false, B, CO, N, G, HW), copies_b = sort_pad(b, false, B, CO, NB, G, HW);
    // (where the values do not stream the weights the bounds do not: their limits are lower. Asked of the operands as they come: copies count
    // as whole rows, whose limits are higher)
    if (K != kBoxK || (density <= 0.f && row_stream_sort_ok(raw)) || (copies == 0) != (copies_b == 0) ||
        !sort_cols_eligible(v, false, B, CO, N, G, HW) || !sort_cols_eligible(b, false, B, CO, NB, G, HW) ||
        sort_cols_cap(kRowsSortValues, N) != sort_cols_cap(kRowsSortInterval, N))
        return apart();
    auto al = [](size_t n) { return (n + 255) / 256 * 256; };
    const size_t shared = al(sort_cols_box_workspace(B, CO, N)), x = al((size_t)B * N * 4);
    const size_t values = sort_tables_bytes(kRowsSortValues, B, CO, N, K) + (two_level_ok(v, K) ? al(two_level_bytes(v, K)) : 0);
    const size_t bounds = sort_tables_bytes(kRowsSortInterval, B, CO, N, K), rest = al(values > bounds ? values : bounds);
    const size_t bytes = shared + rest + (copies ? 3 * x + al((size_t)CO * N * 4) : 0);
    if ((density < 0.f && !hint_build_tables(kHintSiteBox, weight, B, CO, N, st)) || !workspace_ready(bytes, st)) return apart();
    char* ws = static_cast<char*>(workspace(bytes, st));
    if (!ws) return SD_ERR_HIP;
    const float *xv = input, *xl = inputL, *xu = inputU, *w = weight;
    if (copies) {
        float* p = reinterpret_cast<float*>(ws + shared + rest);
        float *pv = p, *pl = p + x / 4, *pu = p + x / 2, *pw = p + 3 * (x / 4);
        if ((rc = pad_rows({input, weight, inputL}, {pv, pw, pl}, {B, CO, B}, CI, N, st))) return rc;
        if ((rc = pad_rows({inputU, inputU, inputU}, {pu, pu, pu}, {B, 0, 0}, CI, N, st))) return rc;
        xv = pv; xl = pl; xu = pu; w = pw;
    }
    SortBox box{nullptr, 0ull, ws, ws + shared, weight, density > 0.f || hint_stand_in(kHintSiteBox, weight, B, CO, N, st)};
    if ((rc = sort_cols_box_tables(xv, xl, xu, w, B, CO, N, ws, density > 0.f ? density : sort_cols_cap(kRowsSortValues, N), &box.count, &box.limit, st)))
        return rc;
    if ((rc = sort_cols_box_main(w, B, CO, N, q, output, outputL, outputU, ws, box.limit, shift, sign, st))) return rc;
    if ((rc = sort_values(xv, w, B, CO, N, G, HW, output, q, K, shift, sign, &box, stream))) return rc;
    return sort_bounds(xl, xu, w, B, CO, N, G, HW, outputL, outputU, q, K, shift, sign, &box, stream);
}

extern "C" int sd_sort_neuron_box_forward(const float* input, const float* inputL, const float* inputU, const float* weight,
                                          int B, int CO, int CI, int G, int HW, float* output, float* outputL, float* outputU,
                                          float q, int K, const float* shift, float sign, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    SD_REQUIRE(!shift || sign == 1.f || sign == -1.f, "sort_neuron_box_forward: a sign (%g) other than 1 and -1", (double)sign);
    return sort_box(input, inputL, inputU, weight, B, CO, CI, G, HW, output, outputL, outputU, q, K, shift, sign, stream);
}
