// Shared definitions of the gfx950 distance-neuron kernels: argument block, counter RNG,
// error reporting and small utility kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include "../../include/sortdist.h"

namespace sd {

constexpr float kEps = 1e-10f;            // floor of every distance (core/cuda/inf_dist_cuda.cu:14)
constexpr uint32_t kSign = 0x80000000u;   // bit 31 of pos
constexpr uint32_t kNanId = 0xffffffffu;  // "no lower-bound gradient" sentinel (bound_inf_dist_cuda.cu:12)
constexpr int kSubBatch = 32;             // samples sharing one index list (inf_dist_cuda.cu:8)

// ---- counter RNG: word = mix(mix((seed ^ stream * C1) + row) + (col + 1) * C2) ------------------
__host__ __device__ __forceinline__ uint32_t rng_mix(uint32_t h) {
    h ^= h >> 16; h *= 0x21f0aaadu;
    h ^= h >> 15; h *= 0x735a2d97u;
    h ^= h >> 15;
    return h;
}
__host__ __device__ __forceinline__ uint32_t rng_row_key(uint32_t seed, uint32_t stream, uint32_t row) {
    return rng_mix((seed ^ (stream * 0x9e3779b9u)) + row);
}
__host__ __device__ __forceinline__ uint32_t rng_word(uint32_t key, uint32_t col) {
    return rng_mix(key + (col + 1u) * 0x85ebca6bu);
}

// ---- arguments shared by every forward tile kernel -------------------------------------------
struct FwdArgs {
    const float* x0;      // input, or lower bound
    const float* x1;      // upper bound (interval kernels)
    const float* w;
    const float* aux;     // max_output of the with-max l-p forward
    float* y0;            // output, or lower output
    float* y1;            // upper output
    int* p0;              // pos / posL / sort pos (K, B, CO, HW)
    int* p1;              // posU
    unsigned long long* packed0;  // (value bits << 32 | ~chunk) merge buffer of split-N position kernels
    unsigned long long* packed1;  // same for the upper bound of the interval kernel
    float* part0;         // split-N partial sums of the l-p forward, [nsplit][part_stride]
    float* part1;         // split-N partial maxima (online form)
    size_t part_stride;   // B * CO * HW
    const uint32_t* xmask;  // factored mask: keep bits of x rows, one word per (row, chunk), or null
    const uint32_t* wmask;  // same for w rows
    const int* ci_idx;    // (S, G, CIg) or null
    const int* co_idx;    // (S, G, COg) or null
    int B, R, HW, G;      // R = B * HW rows of the batch tile
    int COg, CIg;         // per-group output / input channels (compact sizes with index lists)
    int W_COg, W_CIg;     // per-group rows / row length of the weight tensor
    int nsplit;           // number of slices the reduction range is cut in (grid.z = G * nsplit)
    int coarse;           // slices of four chunks at least: the scratch that more of them merge in is not at hand
    int fast_x, fast_w;   // 128-bit loads allowed for the x / w tiles
    float p, inv_p, q;
    const float* shift;   // vector added to the finished values, one entry per output channel, times shift_sign (+1 or -1); or null
    float shift_sign;
    int sample;           // above 1: of the row only every so many'th chunk (l-inf as a scale, see lp_forward_max_first)
    uint32_t* redo;       // l-p relative to a scale: one word per tile of outputs, set to 1 where a result is too far above its scale (kSampledRoot), and left undefined (null: not asked for)
    const uint32_t* only; // not null: gated policies run on the tiles whose word is set, l-p sums for the undefined outputs
    int pow2_scale;       // the scale is aux rounded up to a power of two
    float skip_thr;       // l-p, large p: ratios to the running scale below this cannot change the fp32 result (0 = unused)
    uint32_t seed, t8, t16;
    int mask_mode;        // -1 none, SD_MASK_TERM, SD_MASK_FACTORED
    // device-side choice between two kernels queued for the same result (gated policies only): the kernel runs
    // when gate is null or (*gate > gate_limit) == gate_above, and returns at once otherwise
    const unsigned long long* gate;
    unsigned long long gate_limit;
    int gate_above;
    // pinned words that the gated kernel leaves its outcome in, for the table hints (null: none): 1 in the first when it
    // runs, 0 when it does not; in the second whether *few is not zero
    unsigned long long* told;
    unsigned long long* told2;
    const unsigned long long* few;
    unsigned long long* told3;   // the same for another word of the device
    const unsigned long long* few3;
    // interval forward with positions: non-null and non-zero on the device when a table kernel has already stored the
    // final values and positions, so that resolve_bound_kernel has nothing to do
    const unsigned long long* resolved;
};

// What an evaluation pass adds to the values of output channel c (its running mean, or a bias): the sum is the one that a kernel of its
// own would form from the stored value, 0 leaves it (results are at least 1e-10).  That kernel is bound by its launch: 3.7 us at 1 x 5120,
// 5.6 at 512 x 5120, three of them per certified layer (6 x 5120, batch 512: 1571 -> 1503 us; one image 141 -> 134).
__device__ __forceinline__ float output_shift(const float* shift, float sign, int c) { return shift ? sign * shift[c] : 0.f; }

__device__ __forceinline__ bool gate_closed(const unsigned long long* gate, unsigned long long limit, int above) {
    return gate != nullptr && (*gate > limit) != (above != 0);
}

// the same for a forward tile kernel, whose first work-item reports the outcome (nothing is reported without a gate)
__device__ __forceinline__ bool gate_closed(const FwdArgs& a) {
    if (a.only && a.only[((blockIdx.z % a.G) * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] == 0u) return true;
    if (a.gate == nullptr) return false;
    const bool closed = gate_closed(a.gate, a.gate_limit, a.gate_above);
    if ((a.told || a.told2 || a.told3) && threadIdx.x == 0 && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0) {
        if (a.told) __hip_atomic_store(a.told, closed ? 0ull : 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (a.told2) __hip_atomic_store(a.told2, *a.few != 0ull ? 1ull : 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (a.told3) __hip_atomic_store(a.told3, *a.few3 != 0ull ? 1ull : 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    return closed;
}

// v > 0 rounded up to a power of two, to the largest there is above it
__device__ __forceinline__ float pow2_above(float v) {
    const uint32_t up = (__float_as_uint(v) + 0x7fffffu) & 0x7f800000u;
    return __uint_as_float(up < 0x7f000000u ? up : 0x7f000000u);
}

// ---- error reporting ---------------------------------------------------------------------------
void set_error(const char* fmt, ...);
int check_launch(const char* what);
// records which forward tile kernel the calling thread dispatched last (sd_last_forward_kernel)
void note_forward_kernel(const char* kind, int tb, int tm);
// With sd_time_forward_kernels(1): an event on `stream` before and after a forward tile kernel's launch, for
// sd_last_forward_kernel_ms.  Nothing while the stream is being captured.
void forward_kernel_timer(hipStream_t stream, bool after);

// What sd_last_forward_term_share reads: where the candidate-table counters of the calling thread's last forward
// call lie on the device and how to turn them into the share of the terms that the call formed.
//   kind 0: no tables were queued (every term is formed)
//   kind 1: counts[0] = marked (tile, weight row, input) triples of denom0, counts[1] != 0 when the every-term kernel ran
//   kind 3: counts[0] = marks of the table per batch row (of denom0), counts[1] != 0 when the every-term kernels ran,
//           counts[2] != 0 when the per-batch-row table served, counts[3] = marks of the table per weight row (of denom1)
void note_term_counts(const unsigned long long* counts, int kind, double denom0, double denom1);

#define SD_REQUIRE(cond, ...)                                   \
    do {                                                        \
        if (!(cond)) { sd::set_error(__VA_ARGS__); return SD_ERR_ARG; } \
    } while (0)

// number of compute units of the current device (cached)
int num_cus();

// grow-only scratch buffer owned by the library, one per (device, stream): split-N merges, bit masks, partial
// sums.  Work queued on different streams never shares one; calls on ONE stream use it in queue order.
// Growing waits for that stream and re-allocates (bytes == 0 returns the current buffer).
void* workspace(size_t bytes, hipStream_t stream);
// the same for paths that use scratch for speed where another needs none: whether the buffer holds so many bytes, grown if it has to be.
// False while `stream` records a graph and its buffer is smaller, and where the memory is not to be had.
bool workspace_ready(size_t bytes, hipStream_t stream);

// Held by an entry point while it queues its kernels.  The calls of several host threads then reach their streams
// one after the other, whole, so that a stream's workspace is used in call order even when threads share the stream
// (as they do by default); only the queueing is serialised, the work of different streams still overlaps.
class CallGuard {
public:
    CallGuard();
    ~CallGuard();
    CallGuard(const CallGuard&) = delete;
    CallGuard& operator=(const CallGuard&) = delete;
};

// Whether a call site's candidate tables have paid lately.  Calls that queue a table kernel and an every-term kernel
// for one result let the device choose, and report afterwards which ran: hint_expect returns a pinned word that the
// every-term kernel stores its outcome in (FwdArgs::told; a copy and an event behind every call cost 10 us), read by a later
// call once it is there; nothing waits.  When the every-term kernel ran kHintStreak times in a row for a (site, weight matrix,
// shape) - a layer - the next kHintSkip calls do not build tables at all (hint_build_tables returns false), then one call
// probes again.  A performance hint only: results do not depend on it.  Nothing is expected or remembered while `stream` is
// being captured: tables are then always built, except those that no probe of the operands goes before (`unprobed`), which a
// graph would pay for in every replay where they do not serve; they are captured where they served the layer's last call that
// is known of.  hint_forget: the kernel was not launched after all.
constexpr int kHintStreak = 3, kHintSkip = 31;
bool hint_build_tables(int site, const void* weight, int B, int CO, int CI, hipStream_t stream, bool unprobed = false);
// The same for tables that the layer's other tables make spare (`served`: these served the last call that is known of): built wherever
// those did not serve.  A call that formed every term without the spare ones may have wanted them (operands of one layer that alternate:
// 512 x 2048 x 2048, sort neuron, 150 us from them, 490 for every term), so four times as many calls in a row must not have needed them before
// they are left out again, up to kHintSpareMost: a call in vain costs 14 us.
constexpr int kHintSpareMost = 192;
bool hint_build_spare(int site, const void* weight, int B, int CO, int CI, hipStream_t stream, bool served);
// Whether to queue tables that stand in for those of `site` where these do not serve: left out once those have served kHintStreak
// calls in a row, and, each time they then do not, only after four times as many (up to kHintSpareMost); never while a graph is recorded.
// The slot is that of `site`: nothing is expected for the tables that stand in.
bool hint_stand_in(int site, const void* weight, int B, int CO, int CI, hipStream_t stream);
// whether the layer's last call whose outcome is there was served from tables
bool hint_paid(int site, const void* weight, int B, int CO, int CI);
unsigned long long* hint_expect(int site, const void* weight, int B, int CO, int CI, hipStream_t stream);
void hint_forget(unsigned long long* word);

// zero-fill n floats on `stream` with a kernel (graph-capture friendly, no memset node)
int fill_zero(void* ptr, size_t n_words, hipStream_t stream);
// the same for two buffers with one launch
int fill_zero2(void* a, size_t na_words, void* b, size_t nb_words, hipStream_t stream);
// y = x + sign * shift[channel] on (B, C, HW) tensors, x and y may be one
int channel_shift(const float* x, const float* shift, int B, int C, int HW, float sign, float* y, hipStream_t stream);
// the same in place for two tensors with one launch
int channel_shift_both(float* a, float* b, const float* shift, int B, int C, int HW, float sign, hipStream_t stream);
// copies up to three matrices whose rows hold n values to rows of np, zeros behind the values, with one launch (rows: 0 for none)
int pad_rows(const float* const (&src)[3], float* const (&dst)[3], const int (&rows)[3], int n, int np, hipStream_t stream);

}  // namespace sd
