// Gradients of the l-p distance (core/cuda/norm_dist_cuda.cu:261-504)
//   u(b,m,n) = g[b,m] sgn(d) (|d| / y[b,m])^(p-1), d = x[b,n] - w[m,n];  grad_x[b,n] = sum_m u,  grad_w[m,n] = - sum_b u
// from scalar registers: a wavefront owns 64 inputs (one per lane) and 32 rows of the batch, whose inputs and grad_x sums
// stay in vector registers, and walks a slice of the output channels.  All that a term needs of the pair (row, channel)
// is the same for the 64 lanes; it is laid out by tile, channel and row beforehand and read with scalar loads, 16 rows at a
// time and one block ahead, straight into an operand of the vector instructions.
//
// Vector issue bounds it: 7 instructions per term at p = 8 and no LDS read, at 54 to 59 T lane instructions/s from one card to
// another (a loop of the same instructions on registers alone: 60; with the pairs (g, 1/y) read from LDS, 8 instructions and 3
// wavefronts per SIMD it was 43).  Both gradients in us, that kernel -> this, p = 8: 512 x 5120 x 5120 2460 -> 1720, 250 x 3072 x 1021 258
// -> 151, 90 x 1600 x 230 40 -> 31, 32 x 192 x 192 24 -> 20; convolutions of 80 x 27 x 576 on 32 x 32 positions 1735 -> 610, of
// 64 x 288 x 256 on 16 x 16 1000 -> 224; index lists, 512 x 3840 x 3840 of 5120 1436 -> 1310 (16 additions per weight go to memory,
// 0.4 ms), the inputs' gradient alone 1049 -> 802.
#include <cmath>
#include <type_traits>
#include "fwd_args.h"
#include "lp_grad.h"

namespace sd {

namespace {

constexpr int RB = 32;   // batch rows of a tile (= one index-list sub-batch)
constexpr int MC = 4;    // output channels of a chunk: their weights are loaded a chunk ahead
constexpr int kTiles = 4;   // batch tiles of a workgroup of four wavefronts

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f8v __attribute__((ext_vector_type(8)));
typedef uint32_t u8v __attribute__((ext_vector_type(8)));
// memory that no kernel writes while this one runs, read at wave-uniform addresses: scalar loads
template <class T> using Const = const __attribute__((address_space(4))) T*;
template <class T> __device__ __forceinline__ Const<T> as_const(const void* p) { return (Const<T>)(uintptr_t)p; }

// d^(p-1) g y^(1-p) is formed as the product of two factors, d^I g y^(1-p) and d^J with I + J = p - 1 (power_pair), one multiplication less
// per term than the power of the ratio.  That holds where |d| <= y, as in every output, keeps both factors and d^(p-1) itself below 2^120 and
// makes them normal numbers wherever (|d| / y)^(p-1) is above 2^-56.  Chunks with an output (or its gradient) outside form the ratio.
constexpr int second_factor(int ip) { return ip <= 2 ? 1 : ip == 3 ? 2 : ip == 4 || ip == 6 ? 3 : ip == 8 ? 5 : 4; }
constexpr double two_to(int e) { double v = 1.0; for (; e > 0; e--) v *= 2.0; for (; e < 0; e++) v *= 0.5; return v; }
template <int IP> struct Limits {
    static constexpr int J = second_factor(IP), I = IP - J;
    static constexpr float kYLow = (float)two_to(-70 / IP), kYHigh = (float)two_to(120 / IP);
    static constexpr float kFirstLow = (float)two_to(-126 + (56 * I + IP - 1) / IP), kFirstHigh = 0x1p+120f;   // |g| y^-J, the first factor at |d| = y
    static constexpr float kScaleLow = 0x1p-125f, kScaleHigh = 0x1p+120f;                                  // |g| y^(1-p)
};
template <int N> __device__ __forceinline__ double power(double v) {
    if constexpr (N <= 1) return N ? v : 1.0;
    else { const double h = power<N / 2>(v); return N % 2 ? h * h * v : h * h; }
}

struct Batch {          // the batch side as the kernel reads it
    float* scale;       // [tile][group][channel][row]: g y^(1-p), or g in a chunk that forms ratios; 0 for rows past the batch.
                        // Any other power (IP < 0): pairs (g, 1 / y), and nothing in the two below
    float* recip;       // the same layout: 1 / y in chunks that form ratios, 0 for rows past the batch
    uint32_t* ratio;    // [tile][group][chunk]: the chunk forms ratios
};

struct Args {
    LpGradArgs a;
    Batch s;
    int COp;        // channels of a group, whole chunks
    int tile0;         // first batch tile of the launch (the tables begin with it)
    int zsplit, per;   // slices of the output channels, channels of a slice
    size_t gx_plane;   // floats between the planes of grad_x that the slices write, 0: they add to grad_x
    unsigned nblocks, pairs, groups;   // blocks of 64 inputs; (block, group, slice) triples; groups of WAVES batch tiles
    int span;          // the largest power of two up to 32 and the positions per image: rows that lie side by side
    bool by_die;       // the triples fill the eight dies evenly
    float pm1;         // p - 1 where it is no whole number up to 8
    bool gw_store;     // a workgroup holds the whole batch: its sums are grad_weight
};

constexpr int TS = 65;   // row stride of a tile in LDS
constexpr int lds_words(int waves, bool strided) { return strided ? RB * TS : waves > 1 ? 2 * MC * 64 : 0; }

// u = (first of the pair times the second) from the difference and g y^(1-p)
template <int IP>
__device__ __forceinline__ float2 power_pair(float d, float s) {
    const float t2 = d * d;
    switch (IP) {
        case 0: return make_float2(d >= 0.f ? s : -s, 1.f);
        case 1: return make_float2(s, d);
        case 2: return make_float2(fabsf(d) * s, d);
        case 3: return make_float2(d * s, t2);
        case 4: return make_float2(fabsf(d) * s, t2 * d);
        case 5: return make_float2(d * s, t2 * t2);
        case 6: { const float t3 = t2 * d; return make_float2(fabsf(t3) * s, t3); }
        case 7: return make_float2(t2 * d * s, t2 * t2);
        default: { const float t3 = t2 * d; return make_float2(fabsf(t3) * s, t3 * t2); }
    }
}

template <int IP>
__device__ __forceinline__ float ratio_power(float sr) {
    const float t = sr * sr;
    switch (IP) {
        case 0: return sr >= 0.f ? 1.f : -1.f;
        case 1: return sr;
        case 2: return fabsf(sr) * sr;
        case 3: return sr * t;
        case 4: return fabsf(sr) * sr * t;
        case 5: return sr * t * t;
        case 6: return fabsf(sr) * sr * t * t;
        case 7: return sr * t * t * t;
        default: return fabsf(sr) * sr * t * (t * t);
    }
}

// ---- batch side ---------------------------------------------------------------------------------------------------
// A workgroup lays out 32 rows x 64 channels; workgroups behind those clear grad_weight and, where slices add to it, grad_x.
template <int IP>
__global__ void __launch_bounds__(256) lp_grad_batch_kernel(Args k, float* __restrict__ zero0, size_t zero0_n,
                                                            float* __restrict__ zero1, size_t zero1_n, unsigned fill_from) {
    const LpGradArgs& a = k.a;
    const int tid = threadIdx.x;
    if (blockIdx.x >= fill_from) {
        const size_t step = (size_t)(gridDim.x - fill_from) * 256, i0 = (size_t)(blockIdx.x - fill_from) * 256 + tid;
        for (size_t i = i0; i < zero0_n / 4; i += step) reinterpret_cast<float4*>(zero0)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        for (size_t i = i0 + zero0_n / 4 * 4; i < zero0_n; i += step) zero0[i] = 0.f;
        for (size_t i = i0; i < zero1_n / 4; i += step) reinterpret_cast<float4*>(zero1)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        for (size_t i = i0 + zero1_n / 4 * 4; i < zero1_n; i += step) zero1[i] = 0.f;
        return;
    }
    __shared__ float gs[RB][65], ys[RB][65];
    const unsigned cols = (unsigned)(k.COp + 63) / 64;
    const int c = blockIdx.x % cols, g = (blockIdx.x / cols) % a.G, t = blockIdx.x / cols / a.G;
    const int r0 = (k.tile0 + t) * RB, m0 = c * 64;
    // neighbouring work-items read neighbouring channels (one position per image) or rows
    #pragma unroll
    for (int e = 0; e < 8; e++) {
        const int f = tid + 256 * e, i = a.HW == 1 ? f / 64 : f % RB, j = a.HW == 1 ? f % 64 : f / RB;
        const int r = r0 + i, m = m0 + j;
        float gv = 0.f, yv = IP < 0 ? __builtin_inff() : 1.f;
        if (r < a.R && m < a.COg) {
            const int b = a.HW == 1 ? r : r / a.HW, hw = r - b * a.HW;
            const size_t o = ((size_t)(b * a.G + g) * a.COg + m) * a.HW + hw;
            gv = a.gy[o];
            yv = a.y[o];
        }
        gs[i][j] = gv;
        ys[i][j] = yv;
    }
    __syncthreads();
    // a work-item owns four rows of two channels; eight of them make a channel, 32 a chunk
    const size_t base = ((size_t)t * a.G + g) * k.COp;
    const int i0 = (tid & 7) * 4;
    #pragma unroll
    for (int e = 0; e < 2; e++) {
        const int j = (tid >> 3) + 32 * e, m = m0 + j;
        float s[4], yv[4], gv[4];
        if (IP < 0) {
            if (m < k.COp) {
                float4* dst = reinterpret_cast<float4*>(k.s.scale + ((base + m) * RB + i0) * 2);
                #pragma unroll
                for (int i = 0; i < 4; i += 2) dst[i / 2] = make_float4(gs[i0 + i][j], 1.f / ys[i0 + i][j], gs[i0 + i + 1][j], 1.f / ys[i0 + i + 1][j]);
            }
            continue;
        }
        bool bad = false;
        #pragma unroll
        for (int i = 0; i < 4; i++) {
            gv[i] = gs[i0 + i][j]; yv[i] = ys[i0 + i][j];
            if constexpr (IP > 0) {
                using L = Limits<IP>;
                // (few operations on 64 bits, and the limits tested on 32: they are this kernel's time)
                const double v = 1.0 / (double)yv[i], first = (double)gv[i] * power<L::J>(v);
                s[i] = (float)(first * power<L::I>(v));
                const float size = fabsf(s[i]), part = fabsf((float)first);
                const bool fits = (size >= L::kScaleLow) & (size <= L::kScaleHigh) & (part >= L::kFirstLow) & (part <= L::kFirstHigh);
                bad |= !((yv[i] >= L::kYLow) & (yv[i] <= L::kYHigh) & (fits | (gv[i] == 0.f)));   // (never a row past the batch: 0 and 1)
            } else s[i] = gv[i];
        }
        const bool ratio = ((__builtin_amdgcn_ballot_w64(bad) >> (threadIdx.x & 32)) & 0xffffffffull) != 0ull;
        if (m < k.COp) {
            float* dst = k.s.scale + (base + m) * RB + i0;
            *reinterpret_cast<float4*>(dst) = ratio ? make_float4(gv[0], gv[1], gv[2], gv[3]) : make_float4(s[0], s[1], s[2], s[3]);
            if (ratio) {
                const int real = m < a.COg ? a.R - r0 - i0 : 0;
                *reinterpret_cast<float4*>(k.s.recip + (base + m) * RB + i0) =
                    make_float4(real > 0 ? 1.f / yv[0] : 0.f, real > 1 ? 1.f / yv[1] : 0.f, real > 2 ? 1.f / yv[2] : 0.f, real > 3 ? 1.f / yv[3] : 0.f);
            }
            if ((threadIdx.x & 31) == 0) k.s.ratio[(base + m) / MC] = ratio ? 1u : 0u;
        }
    }
}

// ---- terms --------------------------------------------------------------------------------------------------------
// rows i0 .. i0 + 15 of one channel; `rest` is called behind the first row, when the loads before have arrived
template <int IP, bool GW, class Rest>
__device__ __forceinline__ void product_rows(const float* xr, float* acc, float (&ws)[2], f16v s, float wk, Rest rest) {
    #pragma unroll
    for (int i = 0; i < 16; i++) {
        const float2 f = power_pair<IP>(xr[i] - wk, s[i]);
        acc[i] = fmaf(f.x, f.y, acc[i]);
        asm volatile("" : "+v"(acc[i]));   // added here: put off behind the chunk, the factors of 128 rows would spill
        if (GW) ws[i & 1] = fmaf(f.x, f.y, ws[i & 1]);
        if (i == 0) { __builtin_amdgcn_sched_barrier(0); rest(); }
        if (i % 4 == 0) __builtin_amdgcn_sched_barrier(0);   // more rows at once would take the registers of a fourth wavefront
    }
}
// eight rows of one channel from the ratio
template <int IP, bool GW, class Rest>
__device__ __forceinline__ void ratio_rows(const float* xr, float* acc, float (&ws)[2], f8v g, f8v recip, float wk, Rest rest) {
    #pragma unroll
    for (int i = 0; i < 8; i++) {
        const float pw = ratio_power<IP>((xr[i] - wk) * recip[i]);
        acc[i] = fmaf(g[i], pw, acc[i]);
        asm volatile("" : "+v"(acc[i]));
        if (GW) ws[i & 1] = fmaf(g[i], pw, ws[i & 1]);
        if (i == 0) { __builtin_amdgcn_sched_barrier(0); rest(); }
        if (i % 4 == 0) __builtin_amdgcn_sched_barrier(0);
    }
}
// eight rows of one channel at any power; rows past the batch have g = 1 / y = 0.  (The transcendentals bound it, at any number of
// wavefronts: four rows side by side took 4 % longer.)
template <bool GW, class Rest>
__device__ __forceinline__ void any_power_rows(const float* xr, float* acc, float (&ws)[2], f16v pairs, float wk, float pm1, Rest rest) {
    #pragma unroll
    for (int i = 0; i < 8; i++) {
        const float sr = (xr[i] - wk) * pairs[2 * i + 1];
        const float pw = __builtin_copysignf(__builtin_amdgcn_exp2f(pm1 * __builtin_amdgcn_logf(fabsf(sr))), sr);   // 1 / y > 0: the sign of d
        acc[i] = fmaf(pairs[2 * i], pw, acc[i]);
        asm volatile("" : "+v"(acc[i]));
        if (GW) ws[i & 1] = fmaf(pairs[2 * i], pw, ws[i & 1]);
        if (i == 0) { __builtin_amdgcn_sched_barrier(0); rest(); }
        if (i % 4 == 0) __builtin_amdgcn_sched_barrier(0);
    }
}

enum Form { kProduct, kRatio, kNothing };

// WAVES = kTiles: the wavefronts of a workgroup take neighbouring batch tiles of the same inputs and their sums of grad_weight
// meet in LDS, so that memory sees one addition per 128 rows.  WAVES = 1: they have nothing to do with each
// other, and four of them make a workgroup where there are many, so that every SIMD holds as many (index lists, 512 x 3840 x 3840 of
// 5120, p = 24: 2.7 ms in workgroups of one wavefront).  STRIDED: several positions per image, whose inputs are not side by side in a row.  LISTS: index lists on either side.
template <int IP, bool GW, int WAVES, bool STRIDED, bool LISTS>
__global__ void __launch_bounds__(256, 4) lp_grad_kernel(Args k) {
    const LpGradArgs& a = k.a;
    // the tile on its way between memory and registers where a row's inputs are strided; then sums of grad_weight
    extern __shared__ float shared[];
    constexpr int kLds = lds_words(WAVES, STRIDED);   // of a wavefront
    static_assert(2 * MC * 64 <= RB * TS, "both halves of the sums fit");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* const lds = shared + wave * kLds;
    // all batch tiles of a (block of inputs, slice) run on one die one after the other: they share its weights there
    const unsigned die = blockIdx.x % 8, waves = WAVES > 1 ? 1 : blockDim.x / 64, own = WAVES > 1 ? 0 : wave;
    const unsigned unit = (k.by_die ? blockIdx.x / 8 : blockIdx.x) * waves + own;
    // (in scalar registers, with all that follows from them: the compiler kept some of it in vector registers)
    const unsigned pair = __builtin_amdgcn_readfirstlane(k.by_die ? die + 8 * (unit / k.groups) : unit % k.pairs);
    const unsigned group = __builtin_amdgcn_readfirstlane(k.by_die ? unit % k.groups : unit / k.pairs);
    if (pair >= k.pairs || group >= k.groups) return;
    const int nblock = pair % k.nblocks, g = pair / k.nblocks % a.G, slice = pair / k.nblocks / a.G;
    const int m_lo = slice * k.per, m_hi = m_lo + k.per < a.COg ? m_lo + k.per : a.COg;
    if (m_lo >= m_hi) return;
    const int tile = (int)group * WAVES + (WAVES > 1 ? wave : 0), r0 = (k.tile0 + tile) * RB;
    const int n = nblock * 64 + lane;
    const bool n_ok = n < a.CIg;
    const int nc = n_ok ? n : a.CIg - 1;
    int rows = a.R - r0;
    rows = rows < 0 ? 0 : rows > RB ? RB : rows;
    // rows past the batch repeat one of their tile, with g = 0; a tile behind the batch holds row 0, whose terms are left out
    const int last = rows > 0 ? rows - 1 : 0, rx = rows > 0 ? r0 : 0;
    const int sub = (rx / a.HW) / kSubBatch;   // (one tile to a sub-batch where there are index lists)

    const int wcol = a.ci_idx ? a.ci_idx[(sub * a.G + g) * a.CIg + nc] : nc;
    const float* __restrict__ wbase = a.w + (size_t)g * a.W_COg * a.W_CIg + wcol;
    float* __restrict__ gwbase = GW ? a.gw + (size_t)g * a.W_COg * a.W_CIg + wcol : nullptr;
    // weight rows of the channels from m on, inside the slice; LISTS: fetched ahead, one per lane
    const int* __restrict__ co = LISTS && a.co_idx ? a.co_idx + (size_t)(sub * a.G + g) * a.COg : nullptr;
    auto rows_of = [&](int m) {
        m += lane & (MC - 1);
        m = m < m_hi ? m : m_hi - 1;
        return LISTS && co ? co[m] : m;
    };
    auto row_of = [&](int m0, int j, int rows) {
        if (LISTS) return __builtin_amdgcn_readlane(rows, j);
        return m0 + j < m_hi ? m0 + j : m_hi - 1;
    };

    // where row i of the tile begins, in lane i (the tensors hold fewer than 2^31 values)
    const int rl = rx + ((lane & (RB - 1)) < last ? (lane & (RB - 1)) : last);
    const int begin = ((rl / a.HW) * a.G + g) * a.CIg * a.HW + rl % a.HW;

    // step t of a walk over the tile as memory holds it where a row's inputs are strided: `span` rows side by side, then the
    // next inputs; the row and the input of this lane
    auto strided = [&](int t) {
        const int per = RB / k.span;
        return make_int2((lane & (k.span - 1)) + k.span * (t % per), lane / k.span + 64 / k.span * (t / per));
    };

    const size_t base = ((size_t)tile * a.G + g) * k.COp;
    const Const<float> scale = as_const<float>(k.s.scale + base * RB * (IP < 0 ? 2 : 1)), recip = as_const<float>(k.s.recip + base * RB);
    const Const<uint32_t> ratio = as_const<uint32_t>(k.s.ratio + base / MC);
    const uint32_t* modes = k.s.ratio + base / MC;
    const int c_hi = (m_hi + MC - 1) / MC;
    uint32_t mode = IP > 0 && m_lo / MC + lane < c_hi ? modes[m_lo / MC + lane] : 0u;

    float xr[RB], acc[RB];
    if constexpr (STRIDED) {
        #pragma unroll
        for (int t = 0; t < RB; t++) {
            const int2 at = strided(t);
            const int c = nblock * 64 + at.y < a.CIg ? nblock * 64 + at.y : a.CIg - 1;
            xr[t] = (a.x + __shfl(begin, at.x))[(unsigned)c * (unsigned)a.HW];
        }
        #pragma unroll
        for (int t = 0; t < RB; t++) { const int2 at = strided(t); lds[at.x * TS + at.y] = xr[t]; }
        #pragma unroll
        for (int i = 0; i < RB; i++) { xr[i] = lds[i * TS + lane]; acc[i] = 0.f; }
        if (WAVES > 1) __syncthreads();
    } else {
        #pragma unroll
        for (int i = 0; i < RB; i++) {
            xr[i] = (a.x + __builtin_amdgcn_readlane(begin, i))[(unsigned)nc];
            acc[i] = 0.f;
            if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);
        }
    }

    const int m_end = k.COp;   // channels that the tables hold
    auto block = [&](int m, int i0) { return *(Const<f16v>)(scale + (size_t)m * RB + i0); };

    int rowv = LISTS ? rows_of(m_lo) : 0, rown = LISTS ? rows_of(m_lo + MC) : 0;
    float wv[MC];
    #pragma unroll
    for (int j = 0; j < MC; j++) wv[j] = wbase[(size_t)row_of(m_lo, j, rowv) * a.W_CIg];
    for (int c = m_lo / MC + 64 + lane; IP > 0 && c < c_hi; c += 64) mode |= modes[c];
    // A slice without a chunk that forms ratios runs a loop without them, one instruction less per term (both gradients of 512 x 5120 x
    // 512 with such chunks / without, us: p = 3 198 / 148, p = 8 231 / 190; row by row, with loads of one value, 507 and 519).
    const bool ratios = __builtin_amdgcn_ballot_w64(mode != 0u) != 0ull;

    auto add_weight = [&](int row, float v) {
        float* dst = gwbase + (size_t)row * a.W_CIg;
        if (k.gw_store) *dst = v;
        else unsafeAtomicAdd(dst, v);
    };

    auto walk = [&](auto tag) {
        constexpr Form FORM = decltype(tag)::value;
        int buf = 0;
        for (int m0 = m_lo; m0 < m_hi; m0 += MC, buf ^= 1) {
            float wn[MC];
            #pragma unroll
            for (int j = 0; j < MC; j++) wn[j] = wbase[(size_t)row_of(m0 + MC, j, rown) * a.W_CIg];
            float sum[MC] = {};
            if constexpr (IP < 0) {
                f16v s0 = block(2 * m0, 0);
                float next = 0.f;
                #pragma unroll
                for (int j = 0; j < MC; j++) {
                    float ws[2] = {0.f, 0.f};
                    #pragma unroll
                    for (int q = 0; q < 4; q++) {
                        f16v s1 = s0;
                        any_power_rows<GW>(xr + 8 * q, acc + 8 * q, ws, s0, wv[j], k.pm1, [&] {
                            if (j * 4 + q + 1 < 4 * MC) s1 = block(2 * (m0 + j), 16 * (q + 1));
                            else next = scale[(size_t)(m0 + MC < m_end ? m0 + MC : m0) * RB * 2];
                        });
                        s0 = s1;
                    }
                    sum[j] = ws[0] + ws[1];
                    asm volatile("" : "+v"(sum[j]));
                }
                asm volatile("" :: "s"(next));
            } else if constexpr (FORM == kProduct) {
                f16v s0 = block(m0, 0);
                float next = 0.f;   // brings the next chunk's first block as far as the scalar cache
                #pragma unroll
                for (int j = 0; j < MC; j++) {
                    float ws[2] = {0.f, 0.f};
                    f16v s1;
                    product_rows<IP, GW>(xr, acc, ws, s0, wv[j], [&] { s1 = block(m0 + j, 16); });
                    product_rows<IP, GW>(xr + 16, acc + 16, ws, s1, wv[j], [&] {
                        if (j + 1 < MC) s0 = block(m0 + j + 1, 0);
                        else next = scale[(size_t)(m0 + MC < m_end ? m0 + MC : m0) * RB];
                    });
                    sum[j] = ws[0] + ws[1];
                    asm volatile("" : "+v"(sum[j]));
                }
                asm volatile("" :: "s"(next));
            } else if constexpr (FORM == kRatio) {
                // (a chunk of products: d^(p-1) is the power of the "ratio" d * 1)
                const bool form = ratio[m0 / MC] != 0u;
                const Const<float> g = scale + (size_t)m0 * RB, r = recip + (size_t)m0 * RB;
                auto recips = [&](int at) {
                    u8v v = *(Const<u8v>)(r + at);   // (whole numbers: a choice between floats would take vector instructions)
                    #pragma unroll
                    for (int i = 0; i < 8; i++) v[i] = form ? v[i] : 0x3f800000u;
                    return __builtin_bit_cast(f8v, v);
                };
                f8v g0 = *(Const<f8v>)g, r0 = recips(0);
                #pragma unroll
                for (int j = 0; j < MC; j++) {
                    float ws[2] = {0.f, 0.f};
                    #pragma unroll
                    for (int q = 0; q < 4; q++) {
                        f8v g1 = g0, r1 = r0;
                        ratio_rows<IP, GW>(xr + 8 * q, acc + 8 * q, ws, g0, r0, wv[j], [&] {
                            if (j * 4 + q + 1 < 4 * MC) {
                                g1 = *(Const<f8v>)(g + (j * 4 + q + 1) * 8);
                                r1 = recips((j * 4 + q + 1) * 8);
                            }
                        });
                        g0 = g1; r0 = r1;
                    }
                    sum[j] = ws[0] + ws[1];
                    asm volatile("" : "+v"(sum[j]));
                }
            }
            if (GW && WAVES > 1) {
                #pragma unroll
                for (int j = 0; j < MC; j++) lds[(buf * MC + j) * 64 + lane] = sum[j];
                __syncthreads();   // the other half is written behind the next barrier but one
            }
            // the next weights have arrived before the additions below are queued: waiting for them later would wait for these
            #pragma unroll
            for (int j = 0; j < MC; j++) { asm volatile("" : "+v"(wn[j])); wv[j] = wn[j]; }
            if (GW && WAVES > 1) {
                static_assert(WAVES == 1 || WAVES == MC, "a wavefront adds up one channel of the chunk");
                float v = 0.f;
                #pragma unroll
                for (int j = 0; j < WAVES; j++) v += shared[j * kLds + (buf * MC + wave) * 64 + lane];
                if (n_ok && m0 + wave < m_hi) add_weight(m0 + wave, -v);
            } else if (GW) {
                #pragma unroll
                for (int j = 0; j < MC; j++)
                    if (n_ok && m0 + j < m_hi) add_weight(row_of(m0, j, rowv), -sum[j]);
            }
            if (LISTS) { rowv = rown; rown = rows_of(m0 + 2 * MC); }
        }
    };
    // (0 times the power of a difference is not 0 where the power overflows, and no output says that it does not in a tile behind the batch)
    if (WAVES > 1 && IP >= 0 && rows == 0) walk(std::integral_constant<Form, kNothing>{});
    else if (IP <= 0 || !ratios) walk(std::integral_constant<Form, kProduct>{});
    else walk(std::integral_constant<Form, IP <= 0 ? kProduct : kRatio>{});
    // what only the end needs is read again here: it would take scalar registers all the way
    Const<Args> late = (Const<Args>)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(late));
    float* gx = late->a.gx + (size_t)slice * late->gx_plane;
    const bool add = late->zsplit > 1 && late->gx_plane == 0;
    if constexpr (STRIDED) {
        if (WAVES > 1) __syncthreads();
        #pragma unroll
        for (int i = 0; i < RB; i++) lds[i * TS + lane] = acc[i];
        #pragma unroll 8
        for (int t = 0; t < RB; t++) {
            const int2 at = strided(t);
            float* dst = gx + __shfl(begin, at.x) + (unsigned)(nblock * 64 + at.y) * (unsigned)a.HW;
            const float v = lds[at.x * TS + at.y];
            if (at.x >= rows || nblock * 64 + at.y >= a.CIg) continue;
            if (add) unsafeAtomicAdd(dst, v);
            else *dst = v;
        }
    } else if (n_ok) {
        #pragma unroll
        for (int i = 0; i < RB; i++) {
            if (i < rows) {
                float* dst = gx + __builtin_amdgcn_readlane(begin, i) + (unsigned)n;
                if (add) unsafeAtomicAdd(dst, acc[i]);
                else *dst = acc[i];
            }
            if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

struct Plan {
    int waves, zsplit, per;
    int tiles, launch_tiles;   // batch tiles, whole workgroups of them; of one launch
    size_t words, plane;       // floats of a launch's table (each of the two); of a plane of grad_x, 0: no planes
    size_t bytes;
};

size_t align256(size_t b) { return (b + 255) / 256 * 256; }

Plan make_plan(const LpGradArgs& a) {
    Plan p{};
    const int real = (a.R + RB - 1) / RB, nb = (a.CIg + 63) / 64, COp = (a.COg + MC - 1) / MC * MC;
    const int whole = (real + kTiles - 1) / kTiles * kTiles;
    const bool lists = a.ci_idx || a.co_idx;
    const long long waves = (long long)nb * real * a.G;   // before the output channels are cut
    p.waves = !lists && a.gw && whole * 8 <= real * 9 && waves >= 4ll * num_cus() ? kTiles : 1;
    p.tiles = p.waves > 1 ? whole : real;
    // four rounds of the wavefronts that the device holds at once (four per SIMD; the first round is not dealt evenly, and the last
    // one not filled), slices of at least 64 channels
    const long long units = (long long)nb * p.tiles * a.G, rounds = (64ll * num_cus() + units - 1) / units, longest = a.COg / 64;
    p.zsplit = (int)(rounds > 16 ? 16 : rounds);
    if (p.zsplit > longest) p.zsplit = longest > 1 ? (int)longest : 1;
    // and no fewer than the general kernel's, so that no sum of grad_x runs over more channels (large batches; relative error of grad_x,
    // 8192 x 2048 x 1024 at p = 2: 3 slices there 3.4e-7, 2 slices here 4.0e-7, 3 3.4e-7 and 1310 us instead of 1390)
    const int even = lp_even_slices((long long)((a.CIg + 255) / 256) * real * a.G, 3 * num_cus(), a.COg);
    if (p.zsplit < even) p.zsplit = even;
    // small layers: slices down to one chunk until every SIMD has two wavefronts; their sums are merged in slice order
    const long long fill = 8ll * num_cus();
    bool planes = false;
    if (waves * p.zsplit < fill && aligned16(a.gx)) {
        const long long more = (fill + waves - 1) / waves, most = COp / MC;
        p.zsplit = (int)(more < most ? more : most);
        planes = p.zsplit > 2;
    }
    p.per = ((a.COg + p.zsplit - 1) / p.zsplit + MC - 1) / MC * MC;
    p.zsplit = (a.COg + p.per - 1) / p.per;
    if (planes && p.zsplit > 2) p.plane = ((size_t)a.R * a.G * a.CIg + 3) / 4 * 4;
    // tables of at most 128 MB each: a larger batch is taken in several launches
    const size_t tile_words = (size_t)a.G * COp * RB;
    size_t most = ((size_t)1 << 25) / tile_words / kTiles * kTiles;
    if (most < (size_t)kTiles) most = kTiles;
    p.launch_tiles = (size_t)p.tiles > most ? (int)most : p.tiles;
    p.words = tile_words * p.launch_tiles;
    p.bytes = align256(p.words * 4) * 2 + align256(p.words / RB / MC * 4) + p.plane * p.zsplit * 4;
    return p;
}

template <int IP, bool STRIDED>
void launch_tiles(const Args& k, int waves, hipStream_t st) {
    const bool lists = k.a.ci_idx || k.a.co_idx;
    const unsigned units = k.pairs * k.groups, pack = waves > 1 ? 1 : units >= 8u * num_cus() ? 4 : 1;   // units of a workgroup
    const unsigned per_die = (k.pairs + 7) / 8 * k.groups;
    const dim3 grid(k.by_die ? 8 * ((per_die + pack - 1) / pack) : (units + pack - 1) / pack), block(64 * waves * pack);
    const size_t lds = (size_t)lds_words(waves, STRIDED) * waves * pack * sizeof(float);
    if (lists && k.a.gw) hipLaunchKernelGGL((lp_grad_kernel<IP, true, 1, STRIDED, true>), grid, block, lds, st, k);
    else if (lists) hipLaunchKernelGGL((lp_grad_kernel<IP, false, 1, STRIDED, true>), grid, block, lds, st, k);
    else if (waves > 1) hipLaunchKernelGGL((lp_grad_kernel<IP, true, kTiles, STRIDED, false>), grid, block, lds, st, k);
    else if (k.a.gw) hipLaunchKernelGGL((lp_grad_kernel<IP, true, 1, STRIDED, false>), grid, block, lds, st, k);
    else hipLaunchKernelGGL((lp_grad_kernel<IP, false, 1, STRIDED, false>), grid, block, lds, st, k);
}

template <int IP>
int launch(Args& k, const Plan& p, float* part, hipStream_t st) {
    LpGradArgs& a = k.a;
    float* const gx = a.gx;
    const size_t nx = (size_t)a.R * a.G * a.CIg, nw = a.gw ? (size_t)a.G * a.W_COg * a.W_CIg : 0;
    int rc;
    if (part) { a.gx = part; k.gx_plane = p.plane; }
    for (k.tile0 = 0; k.tile0 < p.tiles; k.tile0 += p.launch_tiles) {
        const int tiles = p.tiles - k.tile0 < p.launch_tiles ? p.tiles - k.tile0 : p.launch_tiles;
        const unsigned lay = (unsigned)((k.COp + 63) / 64) * a.G * tiles;
        k.groups = (unsigned)(tiles / p.waves);
        k.gw_store = !a.ci_idx && !a.co_idx && tiles == p.tiles && k.groups == 1;
        const size_t z0 = k.tile0 == 0 && k.zsplit > 1 && !part ? nx : 0, z1 = k.tile0 == 0 && !k.gw_store ? nw : 0;
        size_t fill = ((z0 > z1 ? z0 : z1) / 4 + 255) / 256;
        if (z0 + z1 && fill == 0) fill = 1;
        if (fill > 16u * num_cus()) fill = 16u * num_cus();
        hipLaunchKernelGGL((lp_grad_batch_kernel<IP>), dim3(lay + (unsigned)fill), dim3(256), 0, st, k, a.gx, z0, a.gw, z1, lay);
        if ((rc = check_launch("lp_grad_batch_kernel"))) return rc;
        if (a.HW > 1) launch_tiles<IP, true>(k, p.waves, st);
        else launch_tiles<IP, false>(k, p.waves, st);
        if ((rc = check_launch("lp_grad_kernel"))) return rc;
    }
    return part ? lp_merge_planes(part, gx, nx, p.plane, k.zsplit, st) : SD_OK;
}

}  // namespace

size_t lp_grad_workspace(const LpGradArgs& a) { return make_plan(a).bytes; }

int lp_grad(int ip, float pm1, const LpGradArgs& a, void* ws, hipStream_t st) {
    const Plan p = make_plan(a);
    Args k{};
    k.a = a;
    k.pm1 = pm1;
    k.COp = (a.COg + MC - 1) / MC * MC;
    k.zsplit = p.zsplit; k.per = p.per;
    k.nblocks = (unsigned)(a.CIg + 63) / 64;
    k.pairs = k.nblocks * a.G * k.zsplit;
    k.by_die = (k.pairs + 7) / 8 * 8 * 32 <= k.pairs * 33;
    for (k.span = 1; k.span < RB && k.span * 2 <= a.HW; ) k.span *= 2;
    char* at = static_cast<char*>(ws);
    k.s.scale = reinterpret_cast<float*>(at); at += align256(p.words * 4);
    k.s.recip = reinterpret_cast<float*>(at); at += align256(p.words * 4);
    k.s.ratio = reinterpret_cast<uint32_t*>(at); at += align256(p.words / RB / MC * 4);
    float* part = p.plane ? reinterpret_cast<float*>(at) : nullptr;
    switch (ip) {
        case 0: return launch<0>(k, p, part, st);
        case 1: return launch<1>(k, p, part, st);
        case 2: return launch<2>(k, p, part, st);
        case 3: return launch<3>(k, p, part, st);
        case 4: return launch<4>(k, p, part, st);
        case 5: return launch<5>(k, p, part, st);
        case 6: return launch<6>(k, p, part, st);
        case 7: return launch<7>(k, p, part, st);
        case 8: return launch<8>(k, p, part, st);
        default: return launch<-1>(k, p, part, st);   // (scale and recip together: the pairs)
    }
}

}  // namespace sd
