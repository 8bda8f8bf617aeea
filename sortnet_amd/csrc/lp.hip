// l-p norm distance: forward entry points and the fused backward kernel.
#include <atomic>
#include <cstdlib>
#include "fwd_tile.h"
#include "fwd_args.h"
#include "fwd_cols.h"
#include "lp_grad.h"
#include "lp_rows.h"

namespace sd {

// integral 0 <= p <= 8 selects a multiply chain, anything else the transcendental path
// (core/cuda/norm_dist.cpp:17-38)
// smallest thresholds from which the significance tests paid at B = 512, M = N = 5120 (p of about 32 for the
// vector-load forward, about 77 for the two-pass forward of the index lists)
constexpr float kLpSkipFrom = 0.5f, kLpSkipFromOnline = 0.75f;
// backward: the dense both-gradient kernel (p of about 97) and the general kernel (p of about 118)
constexpr float kLpSkipFromFused = 0.68f, kLpSkipFromGeneral = 0.73f;

// largest share of marked (tile, row, input) triples at which the candidate-table kernels run instead of the
// kernels that evaluate every term (sd_set_lp_candidate_density); negative: the built-in limits below
static std::atomic<float> g_rows_density{-1.f};
// Measured at B = 512, M = N = 5120 on three kinds of data (normal or uniform inputs against small weights,
// normal inputs against weights of the same size), in ms against the marked share d:
//   forward   table kernel 0.2 + 3.6 d    every term 2.8, with wave-level significance tests 1.3 .. 3.6
//   backward  both gradients 0.13 + 6 d   every term 3.5, with tests 2.8 .. 4.8
//             grad_input only 0.09 + 5 d  every term 3.15, with tests 1.45 .. 4.3
// The limits sit near where the table kernel meets the fastest case of the kernel it replaces: a little above it
// where that kernel's slow cases are far slower than its fast ones.
constexpr float kRowsCapForward = 0.55f, kRowsCapForwardSkip = 0.3f;
constexpr float kRowsCapBackward = 0.5f, kRowsCapBackwardSkip = 0.4f;
constexpr float kRowsCapBackwardInput = 0.55f, kRowsCapBackwardInputSkip = 0.3f;
// below this threshold (p of about 12 forward, 20 backward) most inputs are marked on all three
constexpr float kRowsFromThr = 0.15f;
static inline float rows_cap(float builtin, float thr) {
    const float density = g_rows_density.load(std::memory_order_relaxed);
    if (density >= 0.f) return density;
    return thr >= kRowsFromThr ? builtin : 0.f;
}

// Layers below 2^30 terms go without tables under the built-in limits: the passes that build them take about as long as
// every term there (normal inputs, p = 24, tables -> none, in us: forward 32 x 192 x 192 35 -> 18, 64 x 1024 x 1024
// 61 -> 34, 128 x 3072 x 1024 169 -> 110, 250 x 3072 x 1021 264 -> 213; backward of the last 511 -> 476).
constexpr long long kRowsMinTerms = 1ll << 30;
static inline bool rows_large(int R, int CO, int CI) {
    return g_rows_density.load(std::memory_order_relaxed) >= 0.f || (long long)R * CO * CI >= kRowsMinTerms;
}

static inline int int_power(float p) {
    if (p == (float)(int)p && p >= 0.f && p <= 8.f) return (int)p;
    return -1;
}

// ratio below which a term of r^p is dropped (see lp_add_significant); 0 when it is below `from`, i.e. when too
// many terms would pass for the wavefront-level tests to pay
static inline float lp_skip_threshold(float drop, float p, float from) {
    // the test only makes sense for an exponent above 1: then 0 < thr < 1 and ratios below it are small.  For
    // an exponent of at most 1 (backward with p <= 2) drop^(1/p) is no threshold at all (it exceeds 1 for
    // negative exponents) and every term is evaluated.
    if (!(p > 1.f)) return 0.f;
    const float thr = powf(drop, 1.f / p);
    return (thr >= from && thr < 1.f) ? thr : 0.f;
}

template <template <int> class Pol, int TB, int TM>
static int launch_lp(int ip, const FwdArgs& a, hipStream_t st) {
    switch (ip) {
        case 1: return launch_fwd<Pol<1>, TB, TM>(a, st);
        case 2: return launch_fwd<Pol<2>, TB, TM>(a, st);
        case 3: return launch_fwd<Pol<3>, TB, TM>(a, st);
        case 4: return launch_fwd<Pol<4>, TB, TM>(a, st);
        case 5: return launch_fwd<Pol<5>, TB, TM>(a, st);
        case 6: return launch_fwd<Pol<6>, TB, TM>(a, st);
        case 7: return launch_fwd<Pol<7>, TB, TM>(a, st);
        case 8: return launch_fwd<Pol<8>, TB, TM>(a, st);
        default: return launch_fwd<Pol<-1>, TB, TM>(a, st);
    }
}

// FwdArgs::redo and its kin for outputs of layers with one position per sample, whose tiles are BB rows by BM channels
struct LpRedo {
    uint32_t* flags;
    const uint32_t* only;
    int pow2, COg, G, BB, BM, gx, gy;
    __device__ __forceinline__ size_t tile(size_t o) const {
        const size_t t = o / (unsigned)COg;
        const unsigned m = (unsigned)(o - t * (unsigned)COg), r = (unsigned)(t / (unsigned)G), g = (unsigned)(t - (size_t)r * (unsigned)G);
        return ((size_t)g * gy + r / BB) * gx + m / BM;
    }
};

// merges the split-N slices of the l-p forward in slice order (deterministic) and takes the root:
// plain sums, sums relative to a known maximum (scale), or (sum, running maximum) pairs of the online form
__global__ void __launch_bounds__(256) lp_finalize_kernel(const float* __restrict__ part0, const float* __restrict__ part1,
                                                          const float* __restrict__ scale,
                                                          int nsplit, size_t total, float p, float inv_p,
                                                          float* __restrict__ y, const unsigned long long* gate,
                                                          unsigned long long gate_limit, int gate_above, LpRedo redo) {
    size_t o = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (o >= total || gate_closed(gate, gate_limit, gate_above)) return;
    if (redo.only && (redo.only[redo.tile(o)] == 0u || !lp_redo(y[o]))) return;
    if (part1 == nullptr) {
        float s = 0.f;
        #pragma unroll 16   // (loads in flight: 64 slices of 32 x 256 outputs 9.4 us one after the other)
        for (int k = 0; k < nsplit; k++) s += part0[(size_t)k * total + o];
        const float root = powf(scale ? s : fmaxf(s, FLT_MIN), inv_p);
        y[o] = scale ? root * (redo.pow2 ? pow2_above(scale[o]) : scale[o]) : root;
        if (redo.flags && !(root <= kSampledRoot)) {
            y[o] = __builtin_nanf("");
            redo.flags[redo.tile(o)] = 1u;
        }
    } else {
        float M = kEps;
        #pragma unroll 8
        for (int k = 0; k < nsplit; k++) M = fmaxf(M, part1[(size_t)k * total + o]);
        float s = 0.f;
        #pragma unroll 8
        for (int k = 0; k < nsplit; k++) {
            float Mk = part1[(size_t)k * total + o];
            s += part0[(size_t)k * total + o] * __builtin_amdgcn_exp2f(p * __builtin_amdgcn_logf(Mk / M));
        }
        y[o] = powf(s, inv_p) * M;
    }
}

// cuts the reduction range when the output tiles alone cannot fill the device; partial sums go to the
// library workspace and are merged by lp_finalize_kernel
static int lp_split_setup(FwdArgs& a, int BB, int BM, bool online, hipStream_t st) {
    a.nsplit = pick_nsplit(a, BB, BM);
    a.part_stride = (size_t)a.R * a.G * a.COg;
    auto bytes = [&] { return a.part_stride * a.nsplit * (online ? 2 : 1) * sizeof(float); };
    if (a.nsplit > 1 && !workspace_ready(bytes(), st)) { a.coarse = 1; a.nsplit = pick_nsplit(a, BB, BM); }
    if (a.nsplit > 1) {
        a.part0 = static_cast<float*>(workspace(bytes(), st));
        if (!a.part0) return SD_ERR_HIP;
        a.part1 = online ? a.part0 + a.part_stride * a.nsplit : nullptr;
    }
    return SD_OK;
}

static int lp_split_finish(const FwdArgs& a, hipStream_t st, const LpRedo& redo = LpRedo{}) {
    if (a.nsplit <= 1) return SD_OK;
    hipLaunchKernelGGL(lp_finalize_kernel, dim3((unsigned)((a.part_stride + 255) / 256)), dim3(256), 0, st,
                       a.part0, a.part1, a.part1 ? nullptr : a.aux, a.nsplit, a.part_stride, a.p, a.inv_p, a.y0,
                       a.gate, a.gate_limit, a.gate_above, redo);
    return check_launch("lp_finalize_kernel");
}

// General p on the vector path: the exact maximum of |x - w| per output first (l-inf kernel, 1.5
// instructions per term), then one pass of sums relative to it, instead of the online form's two passes over
// every LDS chunk.  Workspace: the maxima, then the partial sums of the split reduction.
//
// Where every term is formed whatever its size, the scale need not be the maximum: any M0 <= max |x - w| will do that leaves the result within
// kSampledRoot times it.  Layers of at least kSampledTerms terms take the maximum over a part of the inputs, one chunk of eight from all over the row,
// up to the next power of two, which spares the result a rounding.  The tiles of outputs beyond that (undefined or infinite operands
// among them) then run both steps on all inputs, which is what all of them did before, and store these outputs: those beside them keep
// their bits.  Index lists, 512 x 3840 x 3840 of 5120 at p = 24: 1741 -> 1467 us (maxima 312 -> 45,
// launches that return at once 10), with one weight 1e4 times the others 1713 -> 1750; lists 96 x 2250 x 3840, 8.3e8 terms, 229 -> 202; 250 x
// 3072 x 1021 203 -> 182, 64 x 10240 x 1024 179 -> 151.  Where most tiles have such outputs the layer takes twice as long.  Error against 64 bits, rms,
// lists of all 3840 inputs, with the maximum of all inputs -> now: p = 24 6.3e-8 -> 3.8e-8, images against small weights 4.6e-8 -> 3.8e-8, one input
// 6 / 300 times the others 3.2e-7 / 6.8e-7 -> 8.0e-8 / 1.7e-7; p = 10.5 6.9e-8 -> 4.3e-8, 3.0e-7 / 6.8e-7 -> 8.1e-8 / 1.6e-7; p = 31 6.2e-8 -> 3.4e-8,
// 3.1e-7 / 7.0e-7 -> 1.2e-7 / 2.0e-7.  Which outputs keep the scale is decided by the call's own operands alone, so equal calls have equal bits.
constexpr int kSampledPart = 8;
constexpr long long kSampledTerms = 1ll << 29;
static int lp_forward_max_first(FwdArgs& a, bool small, hipStream_t st) {
    const size_t total = (size_t)a.R * a.G * a.COg;
    // dense single-group layers: a kernel that works from per-row candidate tables and finds the maxima as it goes
    // is queued in front of the two steps below, and a count taken on the device decides which of the two runs
    const float thr_rows = powf(1e-6f / (float)a.CIg, 1.f / a.p);
    const float cap = rows_cap(a.skip_thr > 0.f ? kRowsCapForwardSkip : kRowsCapForward, thr_rows);
    const bool rows = cap > 0.f && rows_large(a.R, a.COg, a.CIg) && a.G == 1 && a.HW == 1 && !a.ci_idx &&
                      !a.co_idx && a.W_CIg == a.CIg &&
                      a.CIg % kRowsChunk == 0 && a.R < (1 << 22) && thr_rows > 0.f && thr_rows < 1.f;
    FwdArgs m = a;
    const bool narrow = narrow_tiles(a);
    m.nsplit = pick_nsplit(m, small || narrow ? 32 : 64, narrow ? 32 : 128);
    a.nsplit = m.nsplit;
    const int ns_rows = rows ? lp_rows_forward_nsplit(a.R, a.COg, a.CIg) : 1;
    const bool sampled = a.skip_thr == 0.f && !rows && (long long)a.R * a.G * a.COg * a.CIg >= kSampledTerms;
    const int BB = small || narrow ? 32 : 64, BM = narrow ? 32 : 128, gx = (a.COg + BM - 1) / BM, gy = (a.R + BB - 1) / BB;
    const size_t flag_words = sampled ? ((size_t)gx * gy * a.G + 63) / 64 * 64 : 0;
    // (a word per tile of outputs,) maxima, then the slice results of whichever sum kernel runs (the table kernel leaves two values per slice)
    const size_t table_bytes = rows ? lp_rows_workspace(a.R, a.COg, a.CIg) : 0;
    auto head_bytes = [&] {
        const int slots = a.nsplit > 1 ? a.nsplit : 0, slots_rows = ns_rows > 1 ? 2 * ns_rows : 0;
        const size_t head = total * (size_t)(1 + (slots > slots_rows ? slots : slots_rows)) * sizeof(float);
        return (head + 255) / 256 * 256 + flag_words * 4;
    };
    if (!workspace_ready(head_bytes() + table_bytes, st)) {
        m.coarse = 1;
        a.nsplit = m.nsplit = pick_nsplit(m, small || narrow ? 32 : 64, narrow ? 32 : 128);
    }
    const size_t head_al = head_bytes();
    float* base = static_cast<float*>(workspace(head_al + table_bytes, st));
    if (!base) return SD_ERR_HIP;
    int rc;
    uint32_t* const flags = reinterpret_cast<uint32_t*>(base);
    base += flag_words;
    const int slices = m.nsplit;
    if (sampled) {   // (slices that hold a chunk of the part each)
        const int most = (a.CIg + KT - 1) / KT / kSampledPart;
        m.sample = kSampledPart;
        m.nsplit = slices < most ? slices : most > 1 ? most : 1;
    }
    if (rows) {
        FwdArgs r = a;
        r.nsplit = ns_rows;
        r.part_stride = total;
        r.part0 = ns_rows > 1 ? base + total : nullptr;
        r.part1 = ns_rows > 1 ? base + total * (size_t)(1 + ns_rows) : nullptr;
        rc = lp_rows_forward(a.x0, a.w, nullptr, a.R, a.COg, a.CIg, a.p, thr_rows, ns_rows, a.y0, r.part0,
                             reinterpret_cast<char*>(base) + head_al, cap, &r.gate, &r.gate_limit, st);
        if (rc) return rc;
        r.gate_above = 0;
        if ((rc = lp_split_finish(r, st))) return rc;
        a.gate = r.gate; a.gate_limit = r.gate_limit; a.gate_above = 1;
        m.gate = r.gate; m.gate_limit = r.gate_limit; m.gate_above = 1;
    }
    m.y0 = base;
    if (sampled) rc = fill_zero(flags, flag_words + (m.nsplit > 1 ? total : 0), st);
    else rc = m.nsplit > 1 ? fill_zero(base, total, st) : SD_OK;
    if (rc) return rc;
    if (rows) rc = narrow ? launch_fwd<LinfNogradGated, 2, 2>(m, st) : small ? launch_fwd<LinfNogradGated, 2, 8>(m, st)
                                                             : launch_fwd<LinfNogradGated, 4, 8>(m, st);
    else rc = narrow ? launch_fwd<LinfNograd, 2, 2>(m, st) : small ? launch_fwd<LinfNograd, 2, 8>(m, st)
                                                             : launch_fwd<LinfNograd, 4, 8>(m, st);
    if (rc) return rc;
    a.aux = base;
    a.part_stride = total;
    a.part0 = a.nsplit > 1 ? base + total : nullptr;
    a.part1 = nullptr;
    LpRedo redo{nullptr, nullptr, 0, a.COg, a.G, BB, BM, gx, gy};
    auto sums = [&]() {
        if (a.skip_thr > 0.f) rc = narrow ? launch_fwd<LpWithMaxSkip, 2, 2>(a, st) : small ? launch_fwd<LpWithMaxSkip, 2, 8>(a, st) : launch_fwd<LpWithMaxSkip, 4, 8>(a, st);
        else rc = narrow ? launch_fwd<LpWithMax<-1>, 2, 2>(a, st) : small ? launch_fwd<LpWithMax<-1>, 2, 8>(a, st) : launch_fwd<LpWithMax<-1>, 4, 8>(a, st);
        return rc ? rc : lp_split_finish(a, st, redo);
    };
    if (!sampled) return sums();
    a.redo = redo.flags = flags;
    a.pow2_scale = redo.pow2 = 1;
    if ((rc = sums())) return rc;
    // (the maxima of all inputs meet those of the part in the same buffer)
    m.sample = 0;
    m.nsplit = slices;
    m.only = a.only = redo.only = flags;
    a.redo = redo.flags = nullptr;
    a.pow2_scale = redo.pow2 = 0;
    rc = narrow ? launch_fwd<LinfNogradGated, 2, 2>(m, st) : small ? launch_fwd<LinfNogradGated, 2, 8>(m, st)
                                                           : launch_fwd<LinfNogradGated, 4, 8>(m, st);
    return rc ? rc : sums();
}

// ---- backward -------------------------------------------------------------------------------
// u(b,m,n) = g[b,m] sgn(d) (|d| / y[b,m])^(p-1), d = x[b,n] - w[m,n]
// grad_x[b,n] = sum_m u,  grad_w[m,n] = - sum_b u      (core/cuda/norm_dist_cuda.cu:261-504)
//
// A workgroup owns 256 consecutive input channels (one per work-item) and RB = 32 batch rows.
// Each work-item keeps its 32 inputs and 32 grad_x partial sums in registers and walks all
// output channels in chunks of MC; per output channel it needs its own w[m,n] and the 32 wave-uniform
// pairs (g, 1/y), which are staged in LDS and read as broadcasts.  Everything a chunk needs is
// requested one chunk ahead, so that no load latency sits between two chunks: the weight rows of the
// next chunk (index lists: the row numbers of the chunk after it, one per lane, handed out with
// v_readlane), its weights (MC independent loads into registers) and its (g, 1/y) pairs (into the other
// half of the LDS buffer, one barrier per chunk).  The sum over the 32 rows of grad_w is formed in
// registers and added to memory with one coalesced atomic per work-item and output channel, or stored to the
// batch tile's own plane where the result has to be the same bits in every call (plan_lp_bwd).
constexpr int RB = 32;   // batch rows per workgroup (= one index-list sub-batch)
constexpr int MC = 8;    // output channels per chunk (the chunk body is unrolled: weights sit in named registers)
static_assert(MC * RB == 256, "one (g, 1/y) pair per work-item and chunk");

struct LpBwdArgs {
    const float* gy; const float* x; const float* w; const float* y;
    float* gx; float* gw;
    const int* ci_idx; const int* co_idx;
    int B, R, HW, G, COg, CIg, W_COg, W_CIg;
    float pm1;   // p - 1
    float skip_thr;  // general p: |d| / y below this cannot change the sums (0 = every term is evaluated)
    const unsigned long long* gate;   // see FwdArgs::gate
    unsigned long long gate_limit;
    int gate_above;
    const float* ry;                  // 1 / y when the caller already holds it, else null
    bool gx_is_zero;                  // grad_input (and grad_weight) were zero-filled by the caller
    int zsplit;      // slices of the output-channel range
    // floats between the planes of grad_input (one per slice) and grad_weight (one per batch tile) that gx and gw then point
    // to and lp_merge_kernel adds up; 0: slices and batch tiles add to gx and gw
    unsigned gx_plane, gw_plane;
};

// what becomes of the sums over a batch tile that make up grad_weight
enum LpGradWeight { kGwNone, kGwAdd, kGwStore };

template <int IP>
__device__ __forceinline__ float signed_pow(float d, float ry, float pm1) {
    float sr = d * ry;   // signed ratio
    float t1;
    switch (IP) {
        case 0: return d >= 0.f ? 1.f : -1.f;
        case 1: return sr;
        case 2: return fabsf(sr) * sr;
        case 3: return sr * sr * sr;
        case 4: t1 = sr * sr; return fabsf(sr) * sr * t1;
        case 5: t1 = sr * sr; return sr * t1 * t1;
        case 6: t1 = sr * sr; return fabsf(sr) * sr * t1 * t1;
        case 7: t1 = sr * sr; return sr * t1 * t1 * t1;
        case 8: t1 = sr * sr; return fabsf(sr) * sr * t1 * (t1 * t1);
        default: {
            float pw = __builtin_amdgcn_exp2f(pm1 * __builtin_amdgcn_logf(fabsf(sr)));
            return __builtin_copysignf(pw, sr);   // 1/y > 0: the ratio carries the sign of d (one v_bfi)
        }
    }
}

// general p from the signed ratio sr = d / y
__device__ __forceinline__ float signed_pow_ratio(float sr, float pm1) {
    float pw = __builtin_amdgcn_exp2f(pm1 * __builtin_amdgcn_logf(fabsf(sr)));
    return __builtin_copysignf(pw, sr);
}

// terms of output channel k of a chunk: FULL = all RB rows present
template <int IP, LpGradWeight GW, bool SKIP, bool FULL>
__device__ __forceinline__ void lp_bwd_channel(const LpBwdArgs& a, const float2 (&gr)[RB], const float (&xr)[RB],
                                               float (&acc)[RB], float wk, int rows, int row, bool n_ok,
                                               float* __restrict__ gwcol) {
    float wsum = 0.f;
    if (SKIP) {
        // large p: the two transcendentals only where some lane of the wavefront has a term that counts,
        // tested for eight batch rows together first (padded rows have x = 0, g = 0 and 1/y = 0)
        #pragma unroll
        for (int i0 = 0; i0 < RB; i0 += 8) {
            float sr[8], big = 0.f;
            #pragma unroll
            for (int e = 0; e < 8; e++) { sr[e] = (xr[i0 + e] - wk) * gr[i0 + e].y; big = fmaxf(big, fabsf(sr[e])); }
            if (__builtin_amdgcn_ballot_w64(big > a.skip_thr) == 0ull) continue;
            #pragma unroll
            for (int e = 0; e < 8; e++) {
                if (__builtin_amdgcn_ballot_w64(fabsf(sr[e]) > a.skip_thr) != 0ull) {
                    float u = gr[i0 + e].x * signed_pow_ratio(sr[e], a.pm1);
                    acc[i0 + e] += u;
                    wsum += u;
                }
            }
        }
    } else {
        // the last batch tile by groups of eight rows and a select per row: straight-line code is what hides the LDS
        // latency (250 x 3072 x 1021, 26 rows in the last tile, p = 8: 0.36 ms with a branch per row, 0.25 now)
        #pragma unroll
        for (int i0 = 0; i0 < RB; i0 += 8) {
            if (FULL || i0 < rows) {
                #pragma unroll
                for (int i = i0; i < i0 + 8; i++) {
                    float2 t = gr[i];
                    float pw = signed_pow<IP>(xr[i] - wk, t.y, a.pm1);
                    if (!FULL) pw = i < rows ? pw : 0.f;
                    acc[i] = fmaf(t.x, pw, acc[i]);
                    wsum = fmaf(t.x, pw, wsum);
                }
            }
        }
    }
    if (GW == kGwAdd && n_ok) unsafeAtomicAdd(gwcol + (size_t)row * a.W_CIg, -wsum);
    if (GW == kGwStore && n_ok) gwcol[(size_t)row * a.W_CIg] = -wsum;
}

// one chunk.  The multiply-chain and plain general-p forms unroll the channels (weights in named registers); the
// significance-test form is branchy and large, so it loops and picks its weight with selects.
template <int IP, LpGradWeight GW, bool SKIP, bool FULL>
__device__ __forceinline__ void lp_bwd_chunk(const LpBwdArgs& a, const float2 (&gr)[MC][RB], const float (&xr)[RB],
                                             float (&acc)[RB], const float (&wv)[MC], int rows, int mcount,
                                             int rowv, bool n_ok, float* __restrict__ gwcol) {
    if (SKIP) {
        #pragma unroll 1
        for (int k = 0; k < mcount; k++) {
            float wk = wv[0];
            #pragma unroll
            for (int j = 1; j < MC; j++) wk = k == j ? wv[j] : wk;
            lp_bwd_channel<IP, GW, SKIP, FULL>(a, gr[k], xr, acc, wk, rows, __builtin_amdgcn_readlane(rowv, k), n_ok, gwcol);
        }
    } else {
        #pragma unroll
        for (int k = 0; k < MC; k++) {
            if (k < mcount)
                lp_bwd_channel<IP, GW, SKIP, FULL>(a, gr[k], xr, acc, wv[k], rows, __builtin_amdgcn_readlane(rowv, k), n_ok, gwcol);
        }
    }
}

// RAGGED: the rows are no multiple of RB.  A kernel of its own: with the code for a part of a tile beside it the code for
// whole tiles lost 10 to 20 % to the registers (512 x 5120 x 2560, p = 8: 1.17 -> 1.43 ms).
template <int IP, LpGradWeight GW, bool SKIP, bool RAGGED>
__global__ void __launch_bounds__(256, (SKIP ? 4 : 1)) lp_bwd_kernel(LpBwdArgs a) {
    __shared__ float2 gr[2][MC][RB];   // (g, 1/y) of output channel m0+k, row r0+i; two chunks
    if (gate_closed(a.gate, a.gate_limit, a.gate_above)) return;

    const int tid = threadIdx.x;
    const int g = blockIdx.z % a.G, slice = blockIdx.z / a.G;
    // output channels of this slice, whole chunks
    const int per = ((a.COg + a.zsplit - 1) / a.zsplit + MC - 1) / MC * MC;
    const int m_lo = slice * per, m_hi = m_lo + per < a.COg ? m_lo + per : a.COg;
    if (m_lo >= m_hi) return;   // whole workgroup; no slice is empty where each has a plane of its own
    const int r0 = blockIdx.y * RB;
    const int n = blockIdx.x * 256 + tid;
    const bool n_ok = n < a.CIg;
    const int s = (r0 / a.HW) / kSubBatch;
    int rows = a.R - r0;
    if (rows > RB) rows = RB;

    const int wcol = n_ok ? (a.ci_idx ? a.ci_idx[(s * a.G + g) * a.CIg + n] : n) : 0;
    const int* __restrict__ co = a.co_idx ? a.co_idx + (size_t)(s * a.G + g) * a.COg : nullptr;
    const float* __restrict__ wcolp = a.w + (size_t)g * a.W_COg * a.W_CIg + wcol;
    float* __restrict__ gwcol = GW == kGwNone ? nullptr
        : a.gw + (GW == kGwStore ? (size_t)blockIdx.y * a.gw_plane : (size_t)0) + (size_t)g * a.W_COg * a.W_CIg + wcol;
    // weight row of output channel m0 + (lane mod MC), clamped into the slice so that every load stays inside W
    const int kl = tid & (MC - 1);
    auto row_of = [&](int m0) {
        int m = m0 + kl;
        m = m < m_hi ? m : m_hi - 1;
        return co ? co[m] : m;
    };
    // (g, 1/y) pair number tid of the chunk at m0: consecutive work-items take consecutive channels of one row
    const int sk = tid % MC, si = tid / MC;
    // returns (g, y); the reciprocal is taken when the pair is written to LDS, after the chunk's arithmetic, so
    // that nothing waits for these loads early (padding: g = 0, y = inf, i.e. 1/y = 0)
    auto pair_of = [&](int m0) {
        float2 v = make_float2(0.f, __builtin_inff());
        const int m = m0 + sk, r = r0 + si;
        if (m < m_hi && si < rows) {
            int b = r / a.HW, hw = r - b * a.HW;
            size_t o = ((size_t)(b * a.G + g) * a.COg + m) * a.HW + hw;
            v.x = a.gy[o];
            v.y = a.y[o];
        }
        return v;
    };

    float xr[RB], acc[RB];
    #pragma unroll
    for (int i = 0; i < RB; i++) {
        int r = r0 + i;
        float v = 0.f;
        if (n_ok && i < rows) {
            int b = r / a.HW, hw = r - b * a.HW;
            v = a.x[((size_t)(b * a.G + g) * a.CIg + n) * a.HW + hw];
        }
        xr[i] = v;
        acc[i] = 0.f;
    }

    int rowv = row_of(m_lo), rown = row_of(m_lo + MC);
    float wv[MC];
    #pragma unroll
    for (int k = 0; k < MC; k++) wv[k] = wcolp[(size_t)__builtin_amdgcn_readlane(rowv, k) * a.W_CIg];
    {
        const float2 p0 = pair_of(m_lo);
        gr[0][sk][si] = make_float2(p0.x, 1.f / p0.y);
    }
    __syncthreads();

    int buf = 0;
    for (int m0 = m_lo; m0 < m_hi; m0 += MC, buf ^= 1) {
        // requests for the next chunk (clamped rows: always inside W) and the row numbers of the one after it
        float wn[MC];
        #pragma unroll
        for (int k = 0; k < MC; k++) wn[k] = wcolp[(size_t)__builtin_amdgcn_readlane(rown, k) * a.W_CIg];
        const int rownn = row_of(m0 + 2 * MC);
        const float2 pn = pair_of(m0 + MC);

        const int mcount = m_hi - m0 < MC ? m_hi - m0 : MC;
        if (!RAGGED || rows == RB) lp_bwd_chunk<IP, GW, SKIP, true>(a, gr[buf], xr, acc, wv, rows, mcount, rowv, n_ok, gwcol);
        else lp_bwd_chunk<IP, GW, SKIP, false>(a, gr[buf], xr, acc, wv, rows, mcount, rowv, n_ok, gwcol);

        gr[buf ^ 1][sk][si] = make_float2(pn.x, 1.f / pn.y);   // last read in the previous iteration, before its barrier
        __syncthreads();
        #pragma unroll
        for (int k = 0; k < MC; k++) wv[k] = wn[k];
        rowv = rown;
        rown = rownn;
    }
    if (n_ok) {
        float* gx = a.gx + (size_t)slice * a.gx_plane;
        const bool add = a.zsplit > 1 && a.gx_plane == 0;
        #pragma unroll
        for (int i = 0; i < RB; i++) {
            if (i < rows) {
                int r = r0 + i;
                int b = r / a.HW, hw = r - b * a.HW;
                float* dst = gx + ((size_t)(b * a.G + g) * a.CIg + n) * a.HW + hw;
                if (add) unsafeAtomicAdd(dst, acc[i]);
                else *dst = acc[i];
            }
        }
    }
}

// ---- backward, dense single-group case with grad_weight and large p ------------------------------
// Fused dense backward for grad_input AND grad_weight: u(b, m, n) is formed once and feeds both sums.
// A workgroup owns FN = 8 consecutive input channels and a range of at most FMR weight rows; its 256
// work-items are 16 (row of W: m = tm + 16 j) x 16 (batch row: b = tb + 16 i) with a 4 x 2 x 8 block of terms
// each per (batch tile, weight tile) pair.  Outer loop = batch tiles, inner loop = weight tiles:
//   grad_x partial sums of the 4 batch rows stay in registers across the inner loop, are reduced over the 16
//   work-items that share the rows and added to memory (one atomic per row and channel and weight range);
//   grad_w partial sums of a pair are combined through LDS into an accumulator that covers the whole weight
//   range and is written out once at the end (the workgroup sees every batch row, so grad_weight needs no
//   global atomics).
// All operands sit in vector registers; the only LDS traffic is that combination.
constexpr int FN = 8, FMR = 1024;

__global__ void __launch_bounds__(256) lp_recip_kernel(const float* __restrict__ y, size_t n, float* __restrict__ ry) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) ry[i] = 1.f / y[i];
}

template <int IP, bool SKIP>
__global__ void __launch_bounds__(256, 3) lp_bwd_fused_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                              const float* __restrict__ g, const float* __restrict__ ry,
                                                              int B, int M, int N, int mr, float pm1, float skip_thr,
                                                              float* __restrict__ gx, float* __restrict__ gw,
                                                              const unsigned long long* gate, unsigned long long gate_limit,
                                                              int gate_above) {
    constexpr int TI = 4, TJ = 2;                 // batch rows / weight rows per work-item
    constexpr int PSTRIDE = FN * 16 * TJ + 16;    // plane of one batch-row group, skewed by 16 banks
    constexpr int GSTRIDE = FMR + 32;
    static_assert(FN * 16 * TJ == 256, "one accumulator per work-item and weight tile");
    __shared__ float gwl[FN * GSTRIDE];
    __shared__ float part[16 * PSTRIDE];
    if (gate_closed(gate, gate_limit, gate_above)) return;
    const int tid = threadIdx.x, tm = tid & 15, tb = tid >> 4;
    const int n0 = blockIdx.x * FN;
    const int m_lo = blockIdx.y * mr, m_hi = m_lo + mr < M ? m_lo + mr : M;
    for (int e = tid; e < FN * GSTRIDE; e += 256) gwl[e] = 0.f;
    __syncthreads();

    for (int b0 = 0; b0 < B; b0 += 16 * TI) {
        float xr[TI][FN], gxp[TI][FN];
        int bi[TI];
        #pragma unroll
        for (int i = 0; i < TI; i++) {
            int b = b0 + tb + 16 * i;
            bi[i] = b < B ? b : -1;
            const float* xp = x + (size_t)(b < B ? b : B - 1) * N + n0;
            float4 v0 = *reinterpret_cast<const float4*>(xp), v1 = *reinterpret_cast<const float4*>(xp + 4);
            xr[i][0] = v0.x; xr[i][1] = v0.y; xr[i][2] = v0.z; xr[i][3] = v0.w;
            xr[i][4] = v1.x; xr[i][5] = v1.y; xr[i][6] = v1.z; xr[i][7] = v1.w;
            #pragma unroll
            for (int t = 0; t < FN; t++) gxp[i][t] = 0.f;
        }
        for (int m0 = m_lo; m0 < m_hi; m0 += 16 * TJ) {
            float wr[TJ][FN], gwp[TJ][FN];
            int mj[TJ];
            #pragma unroll
            for (int j = 0; j < TJ; j++) {
                int m = m0 + tm + 16 * j;
                mj[j] = m < m_hi ? m : -1;
                const float* wp = w + (size_t)(m < m_hi ? m : m_hi - 1) * N + n0;
                float4 v0 = *reinterpret_cast<const float4*>(wp), v1 = *reinterpret_cast<const float4*>(wp + 4);
                wr[j][0] = v0.x; wr[j][1] = v0.y; wr[j][2] = v0.z; wr[j][3] = v0.w;
                wr[j][4] = v1.x; wr[j][5] = v1.y; wr[j][6] = v1.z; wr[j][7] = v1.w;
                #pragma unroll
                for (int t = 0; t < FN; t++) gwp[j][t] = 0.f;
            }
            // (g, 1/y) of the TI x TJ pairs first, so that the branches below do not serialise their loads
            float gvs[TI][TJ], rvs[TI][TJ];
            #pragma unroll
            for (int i = 0; i < TI; i++) {
                #pragma unroll
                for (int j = 0; j < TJ; j++) {
                    const bool ok = bi[i] >= 0 && mj[j] >= 0;
                    // padded rows reuse the last valid row of x / w and its own 1/y, so the ratio stays <= 1
                    const size_t o = (size_t)(bi[i] >= 0 ? bi[i] : B - 1) * M + (mj[j] >= 0 ? mj[j] : m_hi - 1);
                    gvs[i][j] = ok ? g[o] : 0.f;
                    rvs[i][j] = ry[o];
                }
            }
            #pragma unroll
            for (int i = 0; i < TI; i++) {
                #pragma unroll
                for (int j = 0; j < TJ; j++) {
                    const float gv = gvs[i][j], rv = rvs[i][j];
                    if (SKIP) {
                        // large p: transcendentals only where some lane of the wavefront has a term that counts,
                        // tested for the eight channels together first
                        float sr[FN], big = 0.f;
                        #pragma unroll
                        for (int t = 0; t < FN; t++) { sr[t] = (xr[i][t] - wr[j][t]) * rv; big = fmaxf(big, fabsf(sr[t])); }
                        if (__builtin_amdgcn_ballot_w64(big > skip_thr) != 0ull) {
                            #pragma unroll
                            for (int t = 0; t < FN; t++) {
                                if (__builtin_amdgcn_ballot_w64(fabsf(sr[t]) > skip_thr) != 0ull) {
                                    float pw = signed_pow_ratio(sr[t], pm1);
                                    gxp[i][t] = fmaf(gv, pw, gxp[i][t]);
                                    gwp[j][t] = fmaf(gv, pw, gwp[j][t]);
                                }
                            }
                        }
                        continue;
                    }
                    #pragma unroll
                    for (int t = 0; t < FN; t++) {
                        float pw = signed_pow<IP>(xr[i][t] - wr[j][t], rv, pm1);
                        gxp[i][t] = fmaf(gv, pw, gxp[i][t]);
                        gwp[j][t] = fmaf(gv, pw, gwp[j][t]);
                    }
                }
            }
            // the 16 work-items that share a weight row publish their partial sums; work-item (t, row) of the
            // tile then adds the 16 of them to the accumulator it owns (LDS float atomics are far too slow)
            #pragma unroll
            for (int j = 0; j < TJ; j++) {
                #pragma unroll
                for (int t = 0; t < FN; t++) part[tb * PSTRIDE + t * (16 * TJ) + tm + 16 * j] = gwp[j][t];
            }
            __syncthreads();
            {
                const int t = tid / (16 * TJ), ml = tid % (16 * TJ);
                float sum = 0.f;
                #pragma unroll
                for (int k = 0; k < 16; k++) sum += part[k * PSTRIDE + t * (16 * TJ) + ml];
                if (m0 + ml < m_hi) gwl[t * GSTRIDE + (m0 - m_lo) + ml] += sum;
            }
            __syncthreads();
        }
        // sum over the 16 work-items that share the batch rows, then one atomic per row and channel
        #pragma unroll
        for (int i = 0; i < TI; i++) {
            #pragma unroll
            for (int t = 0; t < FN; t++) {
                float v = gxp[i][t];
                v += __shfl_xor(v, 1); v += __shfl_xor(v, 2); v += __shfl_xor(v, 4); v += __shfl_xor(v, 8);
                gxp[i][t] = v;
            }
        }
        if (tm == 0) {
            #pragma unroll
            for (int i = 0; i < TI; i++) {
                if (bi[i] >= 0) {
                    #pragma unroll
                    for (int t = 0; t < FN; t++) unsafeAtomicAdd(gx + (size_t)bi[i] * N + n0 + t, gxp[i][t]);
                }
            }
        }
    }
    __syncthreads();
    for (int e = tid; e < (m_hi - m_lo) * 2; e += 256) {
        int row = e >> 1, h = (e & 1) * 4;
        const float* src = gwl + h * GSTRIDE + row;
        *reinterpret_cast<float4*>(gw + (size_t)(m_lo + row) * N + n0 + h) =
            make_float4(-src[0], -src[GSTRIDE], -src[2 * GSTRIDE], -src[3 * GSTRIDE]);
    }
}

static int launch_lp_bwd_fused(int ip, const LpBwdArgs& a, hipStream_t st) {
    const int B = a.R, M = a.COg, N = a.CIg;
    const size_t n = (size_t)B * M;
    int rc;
    const float* ry = a.ry;   // with it comes a zero-filled grad_input
    if (!ry) {
        float* buf = static_cast<float*>(workspace(n * sizeof(float), st));
        if (!buf) return SD_ERR_HIP;
        hipLaunchKernelGGL(lp_recip_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a.y, n, buf);
        if ((rc = check_launch("lp_recip_kernel"))) return rc;
        if ((rc = fill_zero(a.gx, (size_t)B * N, st))) return rc;
        ry = buf;
    }
    const int ranges = (M + FMR - 1) / FMR;
    const int mr = (((M + ranges - 1) / ranges) + 31) / 32 * 32;   // equal ranges, whole weight tiles
    dim3 grid(N / FN, (M + mr - 1) / mr);
    (void)ip;
    hipLaunchKernelGGL((lp_bwd_fused_kernel<-1, true>), grid, dim3(256), 0, st, a.x, a.w, a.gy, ry, B, M, N, mr, a.pm1,
                       a.skip_thr, a.gx, a.gw, a.gate, a.gate_limit, a.gate_above);
    return check_launch("lp_bwd_fused_kernel");
}

// grad[o] (+)= sum of `planes` partial sums, in plane order: the same bits in every call.  A work-item adds four neighbouring
// elements over a quarter of the planes, the quarters meet in LDS (a few planes of a small layer: what counts is how many
// loads are in flight: 32 slices of 32 x 784 take 3.9 us; 8 tiles of 1021 x 3072, 113 MB read and written, 21.7).  The blocks of grad_input first, then those of grad_weight, in one launch.
struct LpMerge { const float* part; float* out; size_t total, plane; int planes; unsigned blocks; bool add; };
__global__ void __launch_bounds__(256) lp_merge_kernel(LpMerge gx, LpMerge gw, const unsigned long long* gate,
                                                       unsigned long long gate_limit, int gate_above) {
    __shared__ float4 sums[4][64];
    if (gate_closed(gate, gate_limit, gate_above)) return;
    const LpMerge m = blockIdx.x < gx.blocks ? gx : gw;
    const int lane = threadIdx.x & 63, quarter = threadIdx.x >> 6;
    const size_t o = ((size_t)(blockIdx.x < gx.blocks ? blockIdx.x : blockIdx.x - gx.blocks) * 64 + lane) * 4;
    const int per = (m.planes + 3) / 4, lo = quarter * per, hi = lo + per < m.planes ? lo + per : m.planes;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    if (o < m.total) {      // (a plane is a whole number of 16-byte words)
        // Every fourth plane to a sum of its own: a small layer is cut into slices of four channels, and one sum over a quarter of them was
        // further off than with fewer planes (relative error of grad_input, 16 x 164 x 1417 at p = 1: 178 planes 1.4e-7, 355 planes 1.7e-7, with
        // these sums 1.1e-7; 4.1 us either way).
        auto add = [&](float4& t, int k) __attribute__((always_inline)) {
            const float4 v = *reinterpret_cast<const float4*>(m.part + k * m.plane + o);
            t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w;
        };
        float4 t[3] = {s, s, s};
        int k = lo;
        #pragma unroll 2
        for (; k + 4 <= hi; k += 4) { add(s, k); add(t[0], k + 1); add(t[1], k + 2); add(t[2], k + 3); }
        for (; k < hi; k++) add(s, k);
        s.x = (s.x + t[0].x) + (t[1].x + t[2].x);
        s.y = (s.y + t[0].y) + (t[1].y + t[2].y);
        s.z = (s.z + t[0].z) + (t[1].z + t[2].z);
        s.w = (s.w + t[0].w) + (t[1].w + t[2].w);
    }
    sums[quarter][lane] = s;
    __syncthreads();
    if (quarter != 0 || o >= m.total) return;
    #pragma unroll
    for (int k = 1; k < 4; k++) {
        const float4 v = sums[k][lane];
        s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    const float r[4] = {s.x, s.y, s.z, s.w};
    if (o + 4 <= m.total && !m.add) *reinterpret_cast<float4*>(m.out + o) = s;
    else {
        for (int k = 0; k < 4 && o + k < m.total; k++) m.out[o + k] = m.add ? m.out[o + k] + r[k] : r[k];
    }
}

int lp_merge_planes(const float* part, float* out, size_t total, size_t plane, int planes, hipStream_t st) {
    const LpMerge m{part, out, total, plane, planes, (unsigned)((total + 255) / 256), false};
    hipLaunchKernelGGL(lp_merge_kernel, dim3(m.blocks), dim3(256), 0, st, m, LpMerge{}, nullptr, 0ull, 0);
    return check_launch("lp_merge_kernel");
}

// How the general kernel's sums are cut and merged.  Sums of up to two addends have one result; more of them are merged in
// a fixed order, from planes in the workspace, or by atomic additions in any order.
struct LpBwdPlan {
    int zsplit;                  // slices of the output-channel range
    int rows;                    // batch rows per launch
    size_t gx_plane, gw_plane;   // floats per plane of partial sums, 0: no planes, the sums meet by atomic additions
    size_t gx_words, gw_words;   // floats of all planes of a launch
    size_t words() const { return gx_words + gw_words; }
};

// workgroups run in rounds of (resident workgroups per CU) x CUs: the slice count whose last round is fullest, a smaller count
// unless a larger one gains 3 %, slices of at least 64 channels
int lp_even_slices(long long blocks, int slots, int channels) {
    int slices = 1;
    double best = 0.0;
    for (int z = 1; z <= 16 && (z == 1 || channels / z >= 64); z++) {
        const double rounds = (double)blocks * z / slots, eff = rounds / std::ceil(rounds);
        if (eff > best * 1.03) { best = eff; slices = z; }
    }
    return slices;
}

// same_bits: the planes that make the gradients of a dense layer the same bits in every call
static LpBwdPlan plan_lp_bwd(const LpBwdArgs& a, bool same_bits, bool planes) {
    LpBwdPlan plan{1, a.R, 0, 0, 0, 0};
    int tiles = (a.R + RB - 1) / RB;
    if (planes && same_bits && a.gw && tiles > 2) {
        // planes of at most 128 MB: a larger batch is taken in several launches
        const size_t most = ((size_t)1 << 25) / ((size_t)a.COg * a.CIg);
        if ((size_t)tiles > most) { tiles = most > 4 ? (int)most : 4; plan.rows = tiles * RB; }
        plan.gw_plane = ((size_t)a.COg * a.CIg + 3) / 4 * 4;
        plan.gw_words = plan.gw_plane * tiles;
    }
    // a workgroup covers 256 input channels x 32 rows and walks the output channels; when that leaves the
    // device mostly idle (index lists: a few hundred kept inputs per sub-batch) the output-channel range is
    // cut in slices
    const long long blocks = (long long)((a.CIg + 255) / 256) * tiles * a.G;
    plan.zsplit = lp_even_slices(blocks, (a.skip_thr > 0.f ? 4 : 3) * num_cus(), a.COg);
    if (!planes || !aligned16(a.gx)) return plan;
    // small layers: slices down to one chunk of MC channels until every compute unit has two workgroups, merged in slice order
    // (p = 8, both gradients, in us, slices of 64 channels -> this, in brackets with atomic additions in any order:
    // 32 x 784 x 256 61 -> 20 (17), 90 x 1600 x 230 199 -> 37 (31), 64 x 1024 x 1024 64 -> 35 (36); with four per unit 51)
    const long long fill = 2ll * num_cus();
    const bool fine = blocks * plan.zsplit < fill;
    if (fine) {
        const long long more = (fill + blocks - 1) / blocks, most = (a.COg + MC - 1) / MC;
        plan.zsplit = (int)(more < most ? more : most);
        const int per = ((a.COg + plan.zsplit - 1) / plan.zsplit + MC - 1) / MC * MC;   // as the kernel cuts
        plan.zsplit = (a.COg + per - 1) / per;
    }
    if (plan.zsplit > 2 && (fine || same_bits)) {
        plan.gx_plane = ((size_t)(plan.rows < a.R ? plan.rows : a.R) * a.G * a.CIg + 3) / 4 * 4;
        plan.gx_words = plan.gx_plane * plan.zsplit;
    }
    return plan;
}

template <LpGradWeight GW>
static int launch_lp_bwd(int ip, const LpBwdArgs& a, hipStream_t st) {
    dim3 grid((a.CIg + 255) / 256, (a.R + RB - 1) / RB, a.G * a.zsplit);
    const bool ragged = a.R % RB != 0;
#define SD_LAUNCH(k, skip)                                                                               \
    do {                                                                                                 \
        if (ragged) hipLaunchKernelGGL((lp_bwd_kernel<k, GW, skip, true>), grid, dim3(256), 0, st, a);   \
        else hipLaunchKernelGGL((lp_bwd_kernel<k, GW, skip, false>), grid, dim3(256), 0, st, a);         \
    } while (0)
#define SD_CASE(k) case k: if constexpr (GW != kGwStore) SD_LAUNCH(k, false); break;   // (planes of grad_weight: p from about 20)
    switch (ip) {
        SD_CASE(0) SD_CASE(1) SD_CASE(2) SD_CASE(3) SD_CASE(4) SD_CASE(5) SD_CASE(6) SD_CASE(7) SD_CASE(8)
        default:
            if (a.skip_thr > 0.f) SD_LAUNCH(-1, true);
            else SD_LAUNCH(-1, false);
            break;
    }
#undef SD_CASE
#undef SD_LAUNCH
    return check_launch("lp_bwd_kernel");
}

// the general kernel as `plan` cuts it; `part`: room for the planes
static int run_lp_bwd(int ip, LpBwdArgs& a, const LpBwdPlan& plan, float* part, hipStream_t st) {
    a.zsplit = plan.zsplit;
    a.gx_plane = (unsigned)plan.gx_plane; a.gw_plane = (unsigned)plan.gw_plane;
    float *gx = a.gx, *const gw = a.gw;
    float *const gx_part = plan.gx_words ? part : nullptr, *const gw_part = plan.gw_words ? part + plan.gx_words : nullptr;
    const size_t w_words = gw ? (size_t)a.G * a.W_COg * a.W_CIg : 0;
    int rc = SD_OK;
    if (!a.gx_is_zero) {   // what atomics add to
        const size_t nx = a.zsplit > 1 && !gx_part ? (size_t)a.R * a.G * a.CIg : 0, nw = gw_part ? 0 : w_words;
        if (nx && nw) rc = fill_zero2(gx, nx, gw, nw, st);
        else if (nx + nw) rc = nx ? fill_zero(gx, nx, st) : fill_zero(gw, nw, st);
        if (rc) return rc;
    }
    for (int left = a.R, first = 1; left > 0; left -= plan.rows, first = 0) {
        a.R = left < plan.rows ? left : plan.rows;
        a.gx = gx_part ? gx_part : gx;
        a.gw = gw_part ? gw_part : gw;
        rc = !gw ? launch_lp_bwd<kGwNone>(ip, a, st) : gw_part ? launch_lp_bwd<kGwStore>(ip, a, st) : launch_lp_bwd<kGwAdd>(ip, a, st);
        if (rc) return rc;
        const size_t x_words = (size_t)a.R * a.G * a.CIg;
        if (plan.words()) {
            LpMerge mx{}, mw{};
            if (gx_part) mx = LpMerge{gx_part, gx, x_words, plan.gx_plane, a.zsplit, (unsigned)((x_words + 255) / 256), false};
            if (gw_part) mw = LpMerge{gw_part, gw, w_words, plan.gw_plane, (a.R + RB - 1) / RB, (unsigned)((w_words + 255) / 256), !first};
            hipLaunchKernelGGL(lp_merge_kernel, dim3(mx.blocks + mw.blocks), dim3(256), 0, st, mx, mw, a.gate, a.gate_limit, a.gate_above);
            if ((rc = check_launch("lp_merge_kernel"))) return rc;
        }
        // (only dense single-group layers are taken in several launches)
        a.x += x_words; gx += x_words;
        a.gy += (size_t)a.R * a.COg; a.y += (size_t)a.R * a.COg;
    }
    return SD_OK;
}

// Whether the gradients are formed from scalar registers (lp_grad.hip) or by the general kernel.  That one leaves out groups of eight rows
// without work where a tile of 32 is not full, and takes a launch less; it loads strided inputs one value per cache line.  Both
// gradients / the inputs' alone, us, general kernel -> from scalar registers, rows x inputs x outputs (x positions):
//   whole p (p = 8)  1 x 2001 x 2000 31 -> 37 / 20 -> 33, 8 x 1024 x 1024 18 -> 21 / 14 -> 20, 17 x 640 x 640 22 -> 21 / 18 -> 20, 1 x 5120 x 5120 157 -> 147
//                    / 104 -> 128, 10 x 5120 x 5120 208 -> 151 / 153 -> 130; lists 8 x 2048 x 2048 28 -> 38 / 20 -> 28, 32 x 512 x 512 22 -> 20 / 19 -> 19
//                    positions: 6 x 2700 x 256 x 2 +51 % / +99 %, 144 x 64 x 64 with 512 rows +21 % / +35 %, 288 x 512 with 2048 rows -62 % / -66 %
//   p = 17.3         1 x 5120 x 2560 76 -> 171 / 56 -> 139, 17 x 3072 x 1024 57 -> 52 / 45 -> 48, 33 x 3072 x 1024 80 -> 84 / 69 -> 75, 33 x 800 x 800 40 -> 32 / 35 ->
//                    30, 65 x 2001 x 2000 141 -> 167 / 121 -> 148, 250 x 3072 x 1021 301 -> 245 / 233 -> 218, 500 x 5120 x 2560 1941 -> 1810 / 1586 -> 1608; whole
//                    tiles 512 x 5120 x 2560 1730 -> 1800, 128 x 3072 x 1024 128 -> 144; lists 8 x 1024 x 1024 19 -> 26, 100 x 512 x 512 31 -> 28, 512 x 1024 x 1024
//                    129 -> 153; positions 4: 128 x 800 x 256 (105 M terms) +38 %, 512 x 2700 x 256 (354 M) -9 %, 16 and more: 64 x 64 x 27 x 1024 -55 %
// (Both gradients of layers with positions stay with scalar registers at whole p from 17 rows on, also where they take longer, 8 x 2700 x 256 x 4
// 32 -> 36 us, 32 x 288 x 512 x 2 23 -> 29: their error against 64 bits is smaller, 32 x 2700 x 256 x 4 3.7e-7 -> 2.5e-7.)
static bool lp_grad_pays(const FwdArgs& f, bool both, bool whole) {
    const long long weights = (long long)f.G * f.COg * f.CIg, terms = weights * f.R;
    if (f.HW > 1) return f.R > 16 && ((whole && both) || terms >= (f.HW >= 16 ? 1ll << 23 : f.HW >= 9 ? 1ll << 26 : 1ll << 28));
    if (f.ci_idx || f.co_idx) return whole ? f.R > (both ? 8 : 16) : f.R > 16 && terms < (1ll << 26);
    if (whole) return both ? f.R > 8 || weights >= (1ll << 23) : f.R > 8 && terms >= (1ll << 24) && (f.R > 16 || weights >= (1ll << 24));
    // rows that the two kernels go through
    const int tiles = (f.R + RB - 1) / RB * RB, eights = (f.R + 7) / 8 * 8;
    return f.R % RB != 0 && f.R > 16 && (7ll * tiles <= 8ll * eights || terms < (1ll << 26));
}

static int lp_backward(const char* who, const float* grad_output, const float* input, const float* weight,
                       const float* output, int B, int CO, int CI, int G, int HW, float* grad_input,
                       float* grad_weight, float p, const int* ci_idx, const int* co_idx, int W_CO, int W_CI,
                       sd_stream_t stream) {
    FwdArgs f;
    int rc = make_fwd_args(f, who, input, nullptr, weight, B, CO, CI, G, HW, ci_idx, co_idx, W_CO, W_CI);
    if (rc) return rc;
    SD_REQUIRE(grad_output && output && grad_input, "%s: null pointer", who);
    SD_REQUIRE(p > 0.f && !std::isinf(p), "%s: p=%g must be positive and finite", who, (double)p);
    LpBwdArgs a{};
    a.gy = grad_output; a.x = input; a.w = weight; a.y = output; a.gx = grad_input; a.gw = grad_weight;
    a.ci_idx = ci_idx; a.co_idx = co_idx;
    a.B = B; a.R = f.R; a.HW = HW; a.G = G; a.COg = f.COg; a.CIg = f.CIg; a.W_COg = f.W_COg; a.W_CIg = f.W_CIg;
    a.pm1 = p - 1.f;
    // a dropped term has (|d| / y)^(p-1) < 1e-16: the reference trains with AdamW at eps = 1e-10 (main.py:38,432), which
    // turns gradient entries far below the parity bar into full-size updates, so the cut sits where even the sum of
    // all dropped terms of an entry (at most 1e-16 x terms x |grad_output|) cannot move such an update visibly
    a.skip_thr = int_power(p - 1.f) < 0 ? lp_skip_threshold(1e-16f, p - 1.f, kLpSkipFrom) : 0.f;
    hipStream_t st = static_cast<hipStream_t>(stream);
    int ip = int_power(p - 1.f);
    // from scalar registers where that pays, the scratch for it is at hand (a stream under capture may lack it) and the gradients are
    // aligned to 16 bytes; else, and for what is left, the general kernel below
    const bool pays = lp_grad_pays(f, grad_weight != nullptr, ip >= 0);
    auto from_scalars = [&](int power) -> int {
        if (!aligned16(grad_input) || !aligned16(grad_weight)) return -1;
        const LpGradArgs b{grad_output, input, weight, output, grad_input, grad_weight, ci_idx, co_idx,
                           f.R, HW, G, f.COg, f.CIg, f.W_COg, f.W_CIg};
        const size_t bytes = lp_grad_workspace(b);
        if (!workspace_ready(bytes, st)) return -1;
        void* ws = workspace(bytes, st);
        return ws ? lp_grad(power, a.pm1, b, ws, st) : SD_ERR_HIP;
    };
    if (ip >= 0 && pays && (rc = from_scalars(ip)) >= 0) return rc;
    // large p with both gradients in the dense single-group case: the kernel that forms every term once for both
    // sums and owns its grad_weight block tests significance more cheaply than the general kernel, whose
    // test only pays from a higher threshold; everything else goes through the general kernel
    const bool dense = G == 1 && HW == 1 && !ci_idx && !co_idx && f.CIg % FN == 0 && aligned16(input) &&
                       aligned16(weight) && aligned16(grad_weight);
    // dense layers at general p: a kernel that works from per-row candidate tables is queued in front of the one
    // that evaluates every term, and a count taken on the device decides which of the two runs
    const float thr_rows = (ip < 0 && a.pm1 > 1.f) ? powf(1e-16f, 1.f / a.pm1) : 0.f;
    // which kernel evaluates every term, and whether it runs its own wave-level tests
    // (and enough workgroups for it: 512 x 600 x 600 at p = 100, 75 of them, took 480 us against 101)
    const long long fused_groups = (long long)(f.CIg / FN) * ((f.COg + FMR - 1) / FMR);
    const bool fused_p = dense && grad_weight && a.skip_thr >= kLpSkipFromFused, fused = fused_p && fused_groups >= 2 * num_cus();
    const bool tests = fused || a.skip_thr >= kLpSkipFromGeneral;
    const float cap = rows_cap(grad_weight ? (tests ? kRowsCapBackwardSkip : kRowsCapBackward)
                                           : (tests ? kRowsCapBackwardInputSkip : kRowsCapBackwardInput), thr_rows);
    const bool rows_p = cap > 0.f && dense && thr_rows > 0.f && thr_rows < 1.f && f.CIg % kRowsChunk == 0 &&
                        f.W_CIg == f.CIg && B < (1 << 22);
    const bool rows = rows_p && rows_large(f.R, f.COg, f.CIg);
    if (!fused && a.skip_thr < kLpSkipFromGeneral) a.skip_thr = 0.f;
    // At such p the table kernel and the fused kernel form a grad_weight that is the same bits in every call, and grad_input
    // too where few weight rows meet; so does the general kernel where it takes the place of one of them for want of size
    // (both gradients, in us, by atomic additions -> from planes: 250 x 3072 x 1021 at p = 24 297 -> 312, 512 x 600 x 600
    // at p = 100 94 -> 101, 2048 x 1024 x 1024 at p = 120 in eight launches 639 -> 717, the fused kernel 3215).
    const bool same_bits = !fused && (fused_p || (rows_p && !rows));
    // other powers without significance tests, as far as none of the above takes them
    if (ip < 0 && pays && a.pm1 > 0.f && a.skip_thr == 0.f && !rows && !fused && !same_bits && (rc = from_scalars(-1)) >= 0) return rc;
    // one request for every user of the workspace: the tables and 1 / y, then the planes of partial sums
    const size_t table_bytes = rows ? (lp_rows_workspace(f.R, f.COg, f.CIg) + (size_t)f.R * f.COg * sizeof(float) + 255) / 256 * 256 : 0;
    LpBwdPlan plan{};
    char* ws = nullptr;
    if (!fused) {
        plan = plan_lp_bwd(a, same_bits, true);
        if (plan.words() && !(ws = static_cast<char*>(workspace(table_bytes + plan.words() * sizeof(float), st))))
            plan = plan_lp_bwd(a, same_bits, false);   // no room for planes (a stream under capture)
    }
    if (rows) {
        if (!ws && !(ws = static_cast<char*>(workspace(table_bytes, st)))) return SD_ERR_HIP;
        // the general kernel adds to a zero-filled grad_weight, which the table kernel must not find cleared after it ran
        if (grad_weight && !fused && !plan.gw_words && (rc = fill_zero(grad_weight, (size_t)G * f.W_COg * f.W_CIg, st))) return rc;
        if ((rc = lp_rows_backward(grad_output, input, weight, output, f.R, f.COg, f.CIg, a.pm1, thr_rows, grad_input,
                                   grad_weight, ws, cap, &a.ry, &a.gate, &a.gate_limit, st))) return rc;
        a.gate_above = 1;
        a.gx_is_zero = true;
    }
    if (fused) return launch_lp_bwd_fused(ip, a, st);
    return run_lp_bwd(ip, a, plan, reinterpret_cast<float*>(ws + table_bytes), st);
}

}  // namespace sd

using namespace sd;

extern "C" int sd_set_lp_candidate_density(float density) {
    SD_REQUIRE(density <= 1.f, "set_lp_candidate_density: %g is above 1", (double)density);
    g_rows_density = density;
    return SD_OK;
}

extern "C" int sd_norm_dist_forward(const float* input, const float* weight,
                                    int B, int CO, int CI, int G, int HW, float* output, float p,
                                    const int* w_index_ci, const int* w_index_co, int W_CO, int W_CI,
                                    sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    FwdArgs a;
    int rc = make_fwd_args(a, "norm_dist_forward", input, nullptr, weight, B, CO, CI, G, HW,
                           w_index_ci, w_index_co, W_CO, W_CI);
    if (rc) return rc;
    SD_REQUIRE(output, "norm_dist_forward: null output");
    SD_REQUIRE(p > 0.f && !std::isinf(p), "norm_dist_forward: p=%g must be positive and finite", (double)p);
    a.y0 = output; a.p = p; a.inv_p = 1.f / p;
    hipStream_t st = static_cast<hipStream_t>(stream);
    static const int kTb42[] = {4, 2};
    const bool narrow = narrow_tiles(a) && p <= 10.f;
    const bool small = w_index_ci || w_index_co || narrow || pick_tb(a, kTb42, 2, 128) == 2 ||
                       !(a.fast_x && a.fast_w);   // (these take the scalar-load kernel, built for 32 rows)
    const bool online = p > 10.f;   // core/cuda/norm_dist.cpp:4,51-55
    const bool lists = w_index_ci || w_index_co;
    // p > 10: the exact maximum per output first, then one pass of sums relative to it.  On the vector path, and with
    // index lists as well: there the gather kernel's two passes over every LDS chunk (the online form) cost more than
    // a second launch (index-list training step at keep 0.75: 17.6 -> 13.7 ms at p = 256, 20.4 -> 20.1 at p = 24).
    const bool max_first = online && ((a.fast_x && a.fast_w && !w_index_co) || (lists && a.HW == 1));
    a.skip_thr = lp_skip_threshold(1e-6f / (float)a.CIg, p, max_first ? kLpSkipFrom : kLpSkipFromOnline);
    if (max_first) return lp_forward_max_first(a, small, st);
    if (int_power(p) > 0 && cols_ok(a, kColsHW, kColsLpTerms)) {
        a.nsplit = cols_nsplit(a);
        a.part_stride = (size_t)a.R * a.G * a.COg;
        const size_t weights = (cols_workspace(a) + 255) / 256 * 256, parts = a.nsplit > 1 ? a.part_stride * a.nsplit * 4 : 0;
        if (workspace_ready(weights + parts, st)) {
            char* ws = static_cast<char*>(workspace(weights + parts, st));
            if (!ws) return SD_ERR_HIP;
            a.part0 = reinterpret_cast<float*>(ws + weights);
            if ((rc = cols_lp(int_power(p), a, ws, st))) return rc;
            return lp_split_finish(a, st);
        }
    }
    if ((rc = lp_split_setup(a, small ? 32 : 64, narrow ? 32 : 128, online, st))) return rc;
    if (!online) {
        int ip = int_power(p);
        rc = narrow ? launch_lp<LpPlain, 2, 2>(ip, a, st) : small ? launch_lp<LpPlain, 2, 8>(ip, a, st) : launch_lp<LpPlain, 4, 8>(ip, a, st);
    } else {
        if (a.skip_thr > 0.f) rc = small ? launch_fwd<LpOnlineSkip, 2, 8>(a, st) : launch_fwd<LpOnlineSkip, 4, 8>(a, st);
        else rc = small ? launch_fwd<LpOnline<-1>, 2, 8>(a, st) : launch_fwd<LpOnline<-1>, 4, 8>(a, st);
    }
    if (rc) return rc;
    return lp_split_finish(a, st);
}

extern "C" int sd_norm_dist_forward_with_max(const float* input, const float* weight, const float* max_output,
                                             int B, int CO, int CI, int G, int HW, float* output, float p,
                                             const int* w_index_ci, const int* w_index_co, int W_CO, int W_CI,
                                             sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    FwdArgs a;
    int rc = make_fwd_args(a, "norm_dist_forward_with_max", input, nullptr, weight, B, CO, CI, G, HW,
                           w_index_ci, w_index_co, W_CO, W_CI);
    if (rc) return rc;
    SD_REQUIRE(output && max_output, "norm_dist_forward_with_max: null output or max_output");
    SD_REQUIRE(p > 0.f && !std::isinf(p), "norm_dist_forward_with_max: p=%g must be positive and finite", (double)p);
    a.y0 = output; a.aux = max_output; a.p = p; a.inv_p = 1.f / p;
    return launch_lp<LpWithMax, 2, 8>(int_power(p), a, static_cast<hipStream_t>(stream));
}

extern "C" int sd_norm_dist_backward_input(const float* grad_output, const float* input, const float* weight,
                                           const float* output, int B, int CO, int CI, int G, int HW,
                                           float* grad_input, float p,
                                           const int* w_index_ci, const int* w_index_co, int W_CO, int W_CI,
                                           sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    return lp_backward("norm_dist_backward_input", grad_output, input, weight, output, B, CO, CI, G, HW,
                       grad_input, nullptr, p, w_index_ci, w_index_co, W_CO, W_CI, stream);
}

extern "C" int sd_norm_dist_backward_input_weight(const float* grad_output, const float* input, const float* weight,
                                                  const float* output, int B, int CO, int CI, int G, int HW,
                                                  float* grad_input, float* grad_weight, float p,
                                                  const int* w_index_ci, const int* w_index_co, int W_CO, int W_CI,
                                                  sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    SD_REQUIRE(grad_weight, "norm_dist_backward_input_weight: null grad_weight");
    return lp_backward("norm_dist_backward_input_weight", grad_output, input, weight, output, B, CO, CI, G, HW,
                       grad_input, grad_weight, p, w_index_ci, w_index_co, W_CO, W_CI, stream);
}
