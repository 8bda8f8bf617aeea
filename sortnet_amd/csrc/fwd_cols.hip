// Forward with the positions on the lanes: a wavefront owns 64 rows of the batch (a row is one position of one sample, and
// neighbouring positions lie side by side in memory) and 8 output channels, whose weights are the same for all lanes and go
// straight into the vector instructions as scalar operands.  Inputs are loaded from memory into registers, eight at a time and one
// step ahead, without a tile in LDS; results leave in the order of memory.  The kernel that stages tiles read one input of a
// row per cache line and stored one result per line, and the pass that finds positions behind it read 32 lines per output.
//
// Scalar loads and vector issue bound it: l-p at p = 8 runs at 51 to 56 T lane instructions/s, the maximum at 37 to 40.  Finding the
// positions is a gather of four inputs per output, a third of the time at 400 inputs, half at 800.  In us, tiles -> this:
//   samples x inputs x outputs x positions   l-inf with positions   without        p = 8
//   64 x 288 x 256 x 64                      135 -> 57              39 -> 31       50 -> 47
//   64 x 288 x 256 x 256                     548 -> 102             91 -> 69       128 -> 113
//   100 x 144 x 100 x 1024                   1101 -> 160            150 -> 81      226 -> 152
//   80 x 27 x 576 x 1024                     3131 -> 252            173 -> 98      297 -> 242
//   32 x 400 x 512 x 1024                    2304 -> 505            321 -> 277     592 -> 522
//   128 x 800 x 1024 x 256                   5397 -> 1809           1071 -> 1036   2153 -> 1938
// Two rows per lane (half the scalar loads per term, four wavefronts per SIMD) were slower, by 13 % at 64 x 288 x 256 x 256
// without positions; a maximum per eight inputs, with positions, by 21 % there and 26 % on the last.
#include "fwd_cols.h"
#include "fwd_args.h"
#include "fwd_tile.h"
#include <type_traits>

namespace sd {

namespace {

constexpr int RC = 8;          // output channels of a wavefront
constexpr int kWaves = 4;      // wavefronts of a workgroup: the same rows, channels next to each other
constexpr int kStep = 8;       // inputs of a step
// Inputs whose powers are added up by themselves: a layer is cut into fewer slices here than by the kernel that stages tiles, and one sum
// over a slice was further off (rms of the relative error of 24 x 800 x 512 x 256 at p = 2 / 8: 4 slices there 6.7e-8 / 4.3e-8, 2 slices
// here 1.1e-7 / 5.3e-8, with these sums 4.7e-8 / 3.9e-8).  Time from 5 % less (p = 2) to 2 % more (p = 8).
constexpr int kRun = 64;

typedef float f16s __attribute__((ext_vector_type(16)));
// memory that no kernel writes while this one runs, read at wave-uniform addresses: scalar loads
template <class T> using Const = const __attribute__((address_space(4))) T*;

struct Quad { f16s h[2]; };    // four inputs of eight channels

inline int quads_of(int CIg) { return (CIg + kStep - 1) / kStep * 2; }
inline int blocks_of(int COg) { return (COg + RC * kWaves - 1) / (RC * kWaves) * kWaves; }

// l-inf distance with positions: the maximum and the quad of inputs that it sits in, which is gone through again at the end (an
// input's number with every term would take 4 instructions of each instead of 2.25; chunks of 32 inputs 1.6, and eight times the loads)
struct LinfQuad : PolicyBase {
    struct Acc { float best; int quad; };
    static __device__ __forceinline__ void init(Acc& A, const FwdArgs&, size_t, bool, int) { A.best = kEps; A.quad = -1; }
    static __device__ __forceinline__ void step4(Acc& A, const FwdArgs&, const float4& x, const float4&, const float4& w, int n, int) {
        const float v = fmaxf(fmaxf(fmaxf(fabsf(x.x - w.x), fabsf(x.y - w.y)), fabsf(x.z - w.z)), fabsf(x.w - w.w));
        if (v > A.best) { A.best = v; A.quad = n / 4; }   // (the lowest quad that attains the value; undefined terms do not count)
    }
};

// Weights as the kernels read them: [block of 8 channels][group][input / 4][channel][input % 4], 0 where there is no channel or
// input.  A workgroup takes 32 channels and 32 inputs.
__global__ void __launch_bounds__(256) cols_layout_kernel(const float* __restrict__ w, float* __restrict__ out, int COg, int CIg,
                                                          int G, int quads, bool vec) {
    const int q = blockIdx.x * 8 + ((threadIdx.x >> 3) & 7), g = blockIdx.z;
    const int block = blockIdx.y * kWaves + (threadIdx.x >> 6), i = threadIdx.x & 7, m = block * RC + i, n = 4 * q;
    if (q >= quads) return;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (m < COg && n < CIg) {
        const float* src = w + (size_t)(g * COg + m) * CIg + n;
        if (vec) v = *reinterpret_cast<const float4*>(src);
        else {
            v.x = src[0];
            if (n + 1 < CIg) v.y = src[1];
            if (n + 2 < CIg) v.z = src[2];
            if (n + 3 < CIg) v.w = src[3];
        }
    }
    reinterpret_cast<float4*>(out)[((size_t)(block * G + g) * quads + q) * RC + i] = v;
}

// first input of a quad whose term is `best` (one of them is), with the sign of its difference.  xp: input 0 of the row; wq: quad 0
// of the channel
__device__ __forceinline__ int find_input(const float* __restrict__ xp, const float4* __restrict__ wq, int HW, int CIg, int quad, float best) {
    const int n0 = 4 * quad;
    float xv[4];
    #pragma unroll
    for (int e = 0; e < 4; e++) xv[e] = xp[(size_t)(n0 + e < CIg ? n0 + e : n0) * HW];
    const float4 w = wq[(size_t)quad * RC];
    const float wv[4] = {w.x, w.y, w.z, w.w};
    int pos = 0;
    #pragma unroll
    for (int e = 3; e >= 0; e--) {
        const float d = xv[e] - wv[e];
        if (n0 + e < CIg && fabsf(d) == best) pos = (n0 + e) | (d < 0.f ? (int)kSign : 0);
    }
    return pos;
}

template <class P>
__global__ void __launch_bounds__(64 * kWaves, 4) fwd_cols_kernel(FwdArgs a, const float* __restrict__ wl, int quads) {
    constexpr bool POS = std::is_same<P, LinfQuad>::value, SUM = !POS && !std::is_same<P, LinfNograd>::value;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = blockIdx.z % a.G, split = blockIdx.z / a.G;
    const int r0 = blockIdx.x * 64, block = blockIdx.y * kWaves + wave, m0 = block * RC;
    if (m0 >= a.COg) return;   // (no barrier below)
    const int nchunks = (a.CIg + KT - 1) / KT;
    const int n_begin = (int)((long long)split * nchunks / a.nsplit) * KT;
    int n_end = (int)((long long)(split + 1) * nchunks / a.nsplit) * KT;
    if (n_end > a.CIg) n_end = a.CIg;
    const int n_full = n_end - (n_end - n_begin) % kStep;

    // inputs: byte offset of the lane's row from the first row's sample (cols_ok: below 2^32); rows past the batch repeat the last
    const int b0 = r0 / a.HW, r = r0 + lane, rr = r < a.R ? r : a.R - 1;
    const int b = rr / a.HW, hw = rr - b * a.HW;
    const float* const xfirst = a.x0 + (size_t)(b0 * a.G + g) * a.CIg * a.HW;
    const size_t plane = (size_t)a.HW;
    const uint32_t xoff = ((uint32_t)(b - b0) * (uint32_t)(a.G * a.CIg) * (uint32_t)a.HW + (uint32_t)hw) * 4u;
    const Const<f16s> wq = (Const<f16s>)(uintptr_t)(wl + (size_t)(block * a.G + g) * quads * (4 * RC));

    struct Inputs { float v[kStep]; };
    auto xload = [&](Inputs& o, int n) __attribute__((always_inline)) {
        #pragma unroll
        for (int e = 0; e < kStep; e++) {
            const int ne = n + e < a.CIg ? n + e : a.CIg - 1;
            const char* base = reinterpret_cast<const char*>(xfirst + plane * (size_t)ne);   // (wave-uniform)
            o.v[e] = *reinterpret_cast<const float*>(base + xoff);
        }
    };
    auto wload = [&](Quad& o, int q) __attribute__((always_inline)) {
        asm volatile("" : "+s"(q));   // (quads apart: loads of two at once would not fit the scalar registers)
        o.h[0] = wq[2 * q]; o.h[1] = wq[2 * q + 1];
    };

    typename P::Acc acc[RC];
    #pragma unroll
    for (int i = 0; i < RC; i++) P::init(acc[i], a, 0, false, split);
    auto terms = [&](const Inputs& x, const Quad& w, int half, int i, int n) __attribute__((always_inline)) {
        const f16s& h = w.h[i / 4];
        const int e = i % 4 * 4;
        const float4 wv = make_float4(h[e], h[e + 1], h[e + 2], h[e + 3]);
        const float4 xv = make_float4(x.v[4 * half], x.v[4 * half + 1], x.v[4 * half + 2], x.v[4 * half + 3]);
        P::step4(acc[i], a, xv, xv, wv, n, 0);
    };

    Quad w;
    Inputs x;
    if (n_begin < n_full) { xload(x, n_begin); wload(w, n_begin / 4); }
    // The first channel's terms wait for the weights of the quad; behind them the next quad's are requested, so that they are on their
    // way while the other channels' terms are formed (scalar loads return in any order: a wait covers all).
    auto step = [&](const Inputs& x, Inputs& xn, int n) __attribute__((always_inline)) {
        const int next = n + kStep < n_full ? n + kStep : n;
        Quad w1, wn;
        xload(xn, next);
        terms(x, w, 0, 0, n);
        __builtin_amdgcn_sched_barrier(0);
        wload(w1, n / 4 + 1);
        __builtin_amdgcn_sched_barrier(0);
        #pragma unroll
        for (int i = 1; i < RC; i++) terms(x, w, 0, i, n);
        __builtin_amdgcn_sched_barrier(0);
        terms(x, w1, 1, 0, n + 4);
        __builtin_amdgcn_sched_barrier(0);
        wload(wn, next / 4);
        __builtin_amdgcn_sched_barrier(0);
        #pragma unroll
        for (int i = 1; i < RC; i++) terms(x, w1, 1, i, n + 4);
        w = wn;
    };
    auto steps = [&](int n, int to) __attribute__((always_inline)) {
        Inputs x1;
        for (; n + 2 * kStep <= to; n += 2 * kStep) { step(x, x1, n); step(x1, x, n + kStep); }
        if (n < to) { step(x, x1, n); x = x1; }
    };
    float total[RC] = {};   // of the runs that are done
    if constexpr (SUM) {
        for (int n0 = n_begin; n0 < n_full; n0 += kRun) {
            steps(n0, n0 + kRun < n_full ? n0 + kRun : n_full);
            #pragma unroll
            for (int i = 0; i < RC; i++) {
                asm volatile("" : "+v"(acc[i].s));
                total[i] += acc[i].s;
                acc[i].s = 0.f;
            }
        }
    } else steps(n_begin, n_full);
    if (n_full < n_end) {   // the end of a row: inputs behind it are 0 on both sides
        xload(x, n_full);
        #pragma unroll
        for (int e = 0; e < kStep; e++) x.v[e] = n_full + e < n_end ? x.v[e] : 0.f;
        #pragma unroll
        for (int half = 0; half < 2; half++) {
            wload(w, n_full / 4 + half);
            #pragma unroll
            for (int i = 0; i < RC; i++) terms(x, w, half, i, n_full + 4 * half);
        }
    }
    if constexpr (SUM) {
        #pragma unroll
        for (int i = 0; i < RC; i++) acc[i].s += total[i];
    }

    if (r >= a.R) return;
    const size_t o0 = ((size_t)(b * a.G + g) * a.COg + m0) * a.HW + hw;
    #pragma unroll
    for (int i = 0; i < RC; i++) {
        if (m0 + i >= a.COg) break;   // (wave-uniform)
        const size_t o = o0 + (size_t)i * a.HW;
        if constexpr (POS) {
            if (a.nsplit > 1) store_chunk_winner(a, o, acc[i].best, acc[i].quad);
            else {
                a.y0[o] = acc[i].best;
                const float4* wrow = reinterpret_cast<const float4*>(wl) + (size_t)(block * a.G + g) * quads * RC + i;
                a.p0[o] = acc[i].quad < 0 ? 0 : find_input(reinterpret_cast<const float*>(reinterpret_cast<const char*>(xfirst) + xoff),
                                                           wrow, a.HW, a.CIg, acc[i].quad, acc[i].best);
            }
        } else P::store(acc[i], a, o, split);
    }
}

// positions of a reduction that was cut into slices, from the merged (value, quad) pairs; neighbouring lanes take neighbouring outputs
__global__ void __launch_bounds__(256) cols_resolve_kernel(FwdArgs a, const float* __restrict__ wl, int quads) {
    const long long total = (long long)a.R * a.G * a.COg;
    const long long o = (long long)blockIdx.x * 256 + threadIdx.x;
    if (o >= total) return;
    const unsigned long long v = a.packed0[o];
    const uint32_t low = (uint32_t)v;
    const float best = low ? __uint_as_float((uint32_t)(v >> 32)) : kEps;
    int pos = 0;
    if (low) {
        const int hw = (int)(o % a.HW), c = (int)(o / a.HW % (a.G * a.COg)), b = (int)(o / a.HW / (a.G * a.COg));
        const int g = c / a.COg, m = c - g * a.COg;
        const float4* wrow = reinterpret_cast<const float4*>(wl) + ((size_t)(m / RC * a.G + g) * quads) * RC + m % RC;
        pos = find_input(a.x0 + (size_t)(b * a.G + g) * a.CIg * a.HW + hw, wrow, a.HW, a.CIg, (int)(0xffffffffu - low), best);
    }
    a.y0[o] = best;
    a.p0[o] = pos;
}

template <class P>
int run(const FwdArgs& a, void* ws, hipStream_t st) {
    float* wl = static_cast<float*>(ws);
    const int quads = quads_of(a.CIg), groups = blocks_of(a.COg) / kWaves;
    hipLaunchKernelGGL(cols_layout_kernel, dim3((quads + 7) / 8, groups, a.G), dim3(256), 0, st, a.w, wl, a.COg, a.CIg, a.G, quads,
                       a.CIg % 4 == 0 && aligned16(a.w));
    int rc = check_launch("cols_layout_kernel");
    if (rc) return rc;
    note_forward_kernel("fwd_cols_kernel", 1, RC);
    forward_kernel_timer(st, false);
    hipLaunchKernelGGL((fwd_cols_kernel<P>), dim3((a.R + 63) / 64, groups, a.G * a.nsplit), dim3(64 * kWaves), 0, st, a, wl, quads);
    rc = check_launch("fwd_cols_kernel");
    forward_kernel_timer(st, true);
    return rc;
}

}  // namespace

bool cols_ok(const FwdArgs& a, int hw, long long terms) {
    const long long samples = 64 / a.HW + 2;   // that the rows of a wavefront reach into
    return a.HW >= hw && a.HW <= kColsMostHW && (long long)a.R * a.G * a.COg * a.CIg >= terms && !a.ci_idx && !a.co_idx && !a.x1 && a.mask_mode < 0 &&
           samples * a.G * a.CIg * a.HW < (1ll << 30) && (a.COg + RC * kWaves - 1) / (RC * kWaves) <= 65535 && a.G <= 1023;
}

int cols_nsplit(const FwdArgs& a) { return pick_nsplit(a, 64, RC * kWaves); }

size_t cols_workspace(const FwdArgs& a) { return (size_t)blocks_of(a.COg) * a.G * quads_of(a.CIg) * (16 * RC); }

int cols_linf(const FwdArgs& a, void* ws, hipStream_t st) {
    if (!a.p0) return run<LinfNograd>(a, ws, st);
    int rc = run<LinfQuad>(a, ws, st);
    if (rc || a.nsplit == 1) return rc;
    const long long total = (long long)a.R * a.G * a.COg;
    hipLaunchKernelGGL(cols_resolve_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, a, static_cast<const float*>(ws), quads_of(a.CIg));
    return check_launch("cols_resolve_kernel");
}

int cols_lp(int ip, const FwdArgs& a, void* ws, hipStream_t st) {
    switch (ip) {
        case 1: return run<LpPlain<1>>(a, ws, st);
        case 2: return run<LpPlain<2>>(a, ws, st);
        case 3: return run<LpPlain<3>>(a, ws, st);
        case 4: return run<LpPlain<4>>(a, ws, st);
        case 5: return run<LpPlain<5>>(a, ws, st);
        case 6: return run<LpPlain<6>>(a, ws, st);
        case 7: return run<LpPlain<7>>(a, ws, st);
        case 8: return run<LpPlain<8>>(a, ws, st);
    }
    set_error("cols_lp: power %d not supported", ip);
    return SD_ERR_ARG;
}

}  // namespace sd
