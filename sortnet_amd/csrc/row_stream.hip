// Few batch rows (one image up to a small batch in evaluation): the layer is a pass over its weights, so its floor is
// the time to read them (5120 x 5120: 105 MB).  The tile kernels cut such a layer into workgroups of 32 batch rows, most
// of them padding, and the candidate tables read the weights three times to save arithmetic that costs nothing here.
//
// A wavefront owns one weight row: every lane loads its share of the row once (NE inputs, all loads in flight together)
// and keeps it in registers; the batch rows pass by in LDS, shared by the four wavefronts of the workgroup.
//   l-inf: 1.5 vector instructions per term and a reduction over the lanes; with positions, the first group of inputs
//   that holds the maximum is found by one comparison per group.
//   sort neuron: the K largest of the row without sorting it.  The K-th largest of the 64 lane maxima is a lower bound T
//   of the K-th largest term (each of the K lanes above it holds one), found bit by bit with ballots; the terms of at
//   least T, about K + 1 of them on data without ties, hold the K largest.  The groups of four inputs that reach T (as
//   many) go to LDS, one term per lane, are ranked against each other and added up in the order of the other kernels
//   (largest first, every product rounded on its own), so the result has the same bits.
// More than 16 such groups, or more than 64 such terms (many equal terms): slower exact paths of the same kernel.
//
// The selection bounds it from about three batch rows on, the weights below.  It starts at the bits that all lane maxima share, ranks up
// to 16 terms in one step of 64 lanes and weighs every term in its own lane; a pass reads at most four groups of a staged row ahead, so
// that rows of 5120 inputs leave room for four wavefronts per SIMD (three, an odd number, issue at three quarters of the rate) and rows of
// 3072 for six.  K = 10, us, before -> now: 1 x 5120 x 5120 28.8 -> 23.4 (4.5 TB/s), 8 x 5120 x 5120 103 -> 81, 33 x 1658 x 1658 83 -> 61,
// 64 x 640 x 640 38 -> 28, 256 x 10240 x 10 31 -> 19; intervals 8 x 5120 x 5120 225 -> 162.
#include "fwd_tile.h"
#include "row_stream.h"

namespace sd {
namespace {

enum StreamOp { kStreamMax, kStreamPos, kStreamSort };
// weight rows (wavefronts) per workgroup: eight share a staged batch row, four where the registers of the sort neuron
// leave room for twelve wavefronts per compute unit
constexpr int stream_waves(StreamOp op) { return op == kStreamSort ? 4 : 8; }

// wavefronts per SIMD that the registers are to leave room for, and how many to count on (rows of up to 1024 inputs leave room for
// twice as many; the staged ends of intervals leave room for fewer)
constexpr int stream_occupancy(int NE, int NX, StreamOp op, bool one = false, bool vec = true) {
    if (one) return NE <= 16 ? 8 : NE == 48 ? (vec ? 8 : 6) : NE == 80 ? (vec ? 5 : 4) : 2;
    return NE == 48 && NX == 1 && op == kStreamSort ? 6 : NE <= 80 ? 4 : 2;
}
constexpr int stream_resident(int NE, int NX, StreamOp op) {
    if (NE <= 16) return NX == 2 && op == kStreamPos ? 7 : 8;
    if (NX == 2 && op == kStreamSort && NE > 48) return NE <= 80 ? 3 : 1;
    return stream_occupancy(NE, NX, op);
}

// maximum over the wavefront, in every lane (row-wise shifts, then the two row broadcasts; v >= 0)
__device__ __forceinline__ float wave_max(float v) {
#define SD_DPP_MAX(ctrl, rows) \
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), ctrl, rows, 0xf, false)))
    SD_DPP_MAX(0x111, 0xf);      // row_shr:1
    SD_DPP_MAX(0x112, 0xf);      // row_shr:2
    SD_DPP_MAX(0x114, 0xf);      // row_shr:4
    SD_DPP_MAX(0x118, 0xf);      // row_shr:8
    SD_DPP_MAX(0x142, 0xa);      // row_bcast:15 into rows 1 and 3
    SD_DPP_MAX(0x143, 0xc);      // row_bcast:31 into rows 2 and 3
#undef SD_DPP_MAX
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
// the minimum of values that are not negative: the maximum of their complements
__device__ __forceinline__ float wave_min(float v) {
    uint32_t u = ~__float_as_uint(v);
#define SD_DPP_MAX(ctrl, rows) { const uint32_t t = __builtin_amdgcn_update_dpp(u, u, ctrl, rows, 0xf, false); u = t > u ? t : u; }
    SD_DPP_MAX(0x111, 0xf) SD_DPP_MAX(0x112, 0xf) SD_DPP_MAX(0x114, 0xf) SD_DPP_MAX(0x118, 0xf) SD_DPP_MAX(0x142, 0xa) SD_DPP_MAX(0x143, 0xc)
#undef SD_DPP_MAX
    return __uint_as_float(~(uint32_t)__builtin_amdgcn_readlane(u, 63));
}

__device__ __forceinline__ int lanes_below(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// LDS operations of one wavefront complete in order; this keeps the compiler from moving them across
__device__ __forceinline__ void wave_fence() { __builtin_amdgcn_wave_barrier(); }

// NE inputs per lane in groups of four.  VEC: a group is four neighbouring inputs (rows a multiple of four long and
// aligned), otherwise inputs 64 apart, so that loads coalesce either way.  grid.y: slices of the batch rows.
// NX = 1: terms |x - w|.  NX = 2: interval bounds, terms -min(w - l, u - w) for the lower (side 0) and
// max(w - l, u - w) for the upper result (side 1), inverted intervals repaired as everywhere.
// ONE: every workgroup meets one batch row (sort neuron, values): the terms take the place of the weights as these arrive, behind an
// input row that is asked for before them.
template <int NE, bool VEC, int NX, StreamOp OP, bool ONE>
__global__ void __launch_bounds__(64 * stream_waves(OP), (stream_occupancy(NE, NX, OP, ONE, VEC)))
row_stream_kernel(FwdArgs a, int K) {
    constexpr int NG = NE / 4, kWaves = stream_waves(OP);
    static_assert(!ONE || (NX == 1 && OP == kStreamSort), "one set of terms per weight row");
    constexpr bool MASKABLE = NX == 1 && OP != kStreamSort;
    __shared__ __attribute__((aligned(16))) float xs[NX][NE * 64];
    __shared__ __attribute__((aligned(16))) float cand[OP == kStreamSort ? kWaves : 1][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tiles = (a.COg + kWaves - 1) / kWaves, g = blockIdx.x / tiles;
    const int CI = a.CIg, m = (blockIdx.x - g * tiles) * kWaves + wave;
    const bool mine = m < a.COg;
    const int c = g * a.COg + (mine ? m : a.COg - 1);
    const float* wrow = a.w + (size_t)c * CI;
    // factored mask: inputs and weights that the mask drops are undefined, and undefined terms never win a maximum
    const int nchunks = (CI + KT - 1) / KT;
    const uint32_t* wkeep = MASKABLE && a.xmask ? a.wmask + (size_t)c * nchunks : nullptr;
    auto masked = [](float v, const uint32_t* keep, int n) {
        return keep == nullptr || ((keep[n >> 5] >> (n & 31)) & 1u) ? v : __builtin_nanf("");
    };
    // the row as a buffer of 4 CI bytes
    const uint64_t wbits = reinterpret_cast<uint64_t>(wrow);
    void* wuni = reinterpret_cast<void*>(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(wbits >> 32)) << 32) |
                                         (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)wbits));
    const auto wrsrc = __builtin_amdgcn_make_buffer_rsrc(wuni, 0, 4 * CI, 0x00020000);

    // ONE: the batch row is on its way before the weights, so that none of them has to have arrived when it is staged
    constexpr int XV = ONE ? (NE + 4 * kWaves - 1) / (4 * kWaves) : 1;
    float4 xfirst[XV];
    if constexpr (ONE) {
        #pragma unroll
        for (int i = 0; i < XV; i++) {
            const int n = 4 * (tid + 64 * kWaves * i);
            const float* src = a.x0 + (size_t)((int)blockIdx.y * a.G + g) * CI;
            if (VEC) {
                xfirst[i] = *reinterpret_cast<const float4*>(src + (n < CI ? n : 0));
                if (n >= CI) xfirst[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            } else
                xfirst[i] = make_float4(n < CI ? src[n] : 0.f, n + 1 < CI ? src[n + 1] : 0.f, n + 2 < CI ? src[n + 2] : 0.f, n + 3 < CI ? src[n + 3] : 0.f);
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    // inputs of group e of this lane: VEC: 4 (64 e + lane) + j, else 256 e + 64 j + lane; beyond the row x = w = 0
    float w[NG][4];
    auto load_weights = [&](int e) {
        if (VEC && ONE) {   // (one address for all groups)
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(wrsrc, 16 * lane, 1024 * e, 0);
            #pragma unroll
            for (int j = 0; j < 4; j++) w[e][j] = __uint_as_float(v[j]);
        } else if (VEC) {
            const int n = 4 * (64 * e + lane);
            const bool in = n < CI;
            const int nn = in ? n : 0;
            float4 v = *reinterpret_cast<const float4*>(wrow + nn);
            if (wkeep) v = make_float4(masked(v.x, wkeep, nn), masked(v.y, wkeep, nn + 1), masked(v.z, wkeep, nn + 2), masked(v.w, wkeep, nn + 3));
            w[e][0] = in ? v.x : 0.f; w[e][1] = in ? v.y : 0.f; w[e][2] = in ? v.z : 0.f; w[e][3] = in ? v.w : 0.f;
        } else {
            #pragma unroll
            for (int j = 0; j < 4; j++) {
                const int n = 256 * e + 64 * j + lane;
                // (a buffer load returns 0 beyond the row: a select per input would keep a lane mask alive for each)
                w[e][j] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(wrsrc, 4 * n, 0, 0));
                if (wkeep && n < CI) w[e][j] = masked(w[e][j], wkeep, n);
            }
        }
    };
    #pragma unroll
    for (int e = 0; e < NG - (ONE ? XV : 0); e++) load_weights(e);
    if constexpr (ONE) {   // the last groups' weights take the registers that the input row came in
        __builtin_amdgcn_sched_barrier(0);
        #pragma unroll
        for (int i = 0; i < XV; i++) {
            const int n = 4 * (tid + 64 * kWaves * i);
            if (NE % (4 * kWaves) == 0 || n < NE * 64) *reinterpret_cast<float4*>(&xs[0][n]) = xfirst[i];
        }
        __builtin_amdgcn_sched_barrier(0);
        #pragma unroll
        for (int e = NG - XV; e < NG; e++) load_weights(e);
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!ONE) {
        #pragma unroll
        for (int k = 0; k < NX; k++)
            for (int n = CI + tid; n < NE * 64; n += 64 * kWaves) xs[k][n] = 0.f;
    }

    // The staged rows stay in LDS between the passes: keeps the compiler from holding what one pass read in registers for
    // the next, and (every few groups) from starting a whole pass's reads at once
    float zero = 0.f;   // (ONE: a value the compiler does not know, another one in every pass, so that no pass holds the maxima of the one before)
    auto pass_fence = [&]() { asm volatile("" : "+v"(zero) : : "memory"); };
    auto group_fence = [](int e) {
        if (NX == 2 ? e % 2 == 1 : OP == kStreamSort && NE >= 48 && e % 4 == 3) { asm volatile("" ::: "memory"); __builtin_amdgcn_sched_barrier(0); }
    };
    auto load4 = [&](const float* row, int e, float (&x)[4]) {
        if (VEC) {
            const float4 t = *reinterpret_cast<const float4*>(&row[4 * (64 * e + lane)]);
            x[0] = t.x; x[1] = t.y; x[2] = t.z; x[3] = t.w;
        } else {
            #pragma unroll
            for (int j = 0; j < 4; j++) x[j] = row[256 * e + 64 * j + lane];
        }
    };
    // terms of group e, and what bit 31 of a position says about each (only evaluated where it is used)
    auto terms = [&](int side, int e, float (&v)[4], bool (&flag)[4]) {
        if constexpr (ONE) {
            #pragma unroll
            for (int j = 0; j < 4; j++) { v[j] = w[e][j]; flag[j] = false; }
            return;
        }
        float x[4], u[4];
        load4(xs[0], e, x);
        if (NX == 2) load4(xs[NX - 1], e, u);
        #pragma unroll
        for (int j = 0; j < 4; j++) {
            if (NX == 1) { const float d = x[j] - w[e][j]; v[j] = fabsf(d); flag[j] = d < 0.f; }
            else {
                const float t1 = w[e][j] - x[j], t2 = u[j] - w[e][j];
                v[j] = side ? fmaxf(t1, t2) : -fminf(t1, t2);
                flag[j] = !(t1 <= t2);
            }
        }
    };

    const float sh = output_shift(a.shift, a.shift_sign, c);
    float coef = 1.f, rest = 1.f;                      // weight of the lane's term, what is left behind the K-th
    if (OP == kStreamSort) {
        for (int k = 0; k < K; k++) { coef = lane == k ? rest : coef; rest *= 1.f - a.q; }
    }

    // (the divisions behind the loads of the weights: in front of them 0.5 us of 17 at 1 x 5120 x 5120)
    const int r_lo = ONE ? (int)blockIdx.y : (int)((long long)blockIdx.y * a.R / gridDim.y);
    const int r_hi = ONE ? r_lo + 1 : (int)((long long)(blockIdx.y + 1) * a.R / gridDim.y);
    for (int r = r_lo; r < r_hi; r++) {
        const size_t xoff = (size_t)(r * a.G + g) * CI;
        const uint32_t* xkeep = MASKABLE && a.xmask ? a.xmask + (size_t)(r * a.G + g) * nchunks : nullptr;
        if (r > r_lo) __syncthreads();                 // every wavefront is done with the row before
        for (int n = VEC ? 4 * tid : tid; !ONE && n < CI; n += (VEC ? 4 : 1) * 64 * kWaves) {
            constexpr int W = VEC ? 4 : 1;
            float x[W], u[W];
            if (VEC) {
                const float4 t = *reinterpret_cast<const float4*>(a.x0 + xoff + n);
                x[0] = t.x; x[W / 2] = t.z; x[W > 1 ? 1 : 0] = W > 1 ? t.y : t.x; x[W - 1] = W > 1 ? t.w : t.x;
            } else x[0] = a.x0[xoff + n];
            if (NX == 2) {
                if (VEC) {
                    const float4 t = *reinterpret_cast<const float4*>(a.x1 + xoff + n);
                    u[0] = t.x; u[W / 2] = t.z; u[W > 1 ? 1 : 0] = W > 1 ? t.y : t.x; u[W - 1] = W > 1 ? t.w : t.x;
                } else u[0] = a.x1[xoff + n];
            }
            #pragma unroll
            for (int j = 0; j < W; j++) {
                if (NX == 2) { if (x[j] > u[j]) x[j] = u[j] = (x[j] + u[j]) * 0.5f; }
                if (xkeep) x[j] = masked(x[j], xkeep, n + j);
                xs[0][n + j] = x[j];
                if (NX == 2) xs[NX - 1][n + j] = u[j];
            }
        }
        __syncthreads();
        if constexpr (ONE) {
            #pragma unroll
            for (int e = 0; e < NG; e++) {
                float x[4];
                load4(xs[0], e, x);
                #pragma unroll
                for (int j = 0; j < 4; j++) {
                    w[e][j] = fabsf(x[j] - w[e][j]);
                    asm volatile("" : "+v"(w[e][j]));   // the magnitude itself, not the difference and a modifier at each use
                }
                if (e % 2 == 1) { asm volatile("" ::: "memory"); __builtin_amdgcn_sched_barrier(0); }
            }
        }

        const size_t o = (size_t)(r * a.G + g) * a.COg + m;
        if (OP == kStreamMax) {
            float top[NX];
            #pragma unroll
            for (int k = 0; k < NX; k++) top[k] = 0.f;
            #pragma unroll
            for (int e = 0; e < NG; e++) {
                #pragma unroll
                for (int k = 0; k < NX; k++) {
                    float v[4];
                    bool flag[4];
                    terms(k, e, v, flag);
                    top[k] = fmaxf(fmaxf(fmaxf(fmaxf(top[k], v[0]), v[1]), v[2]), v[3]);
                }
                group_fence(e);
            }
            #pragma unroll
            for (int k = 0; k < NX; k++) asm volatile("" : "+v"(top[k]));   // both maxima are formed in the one pass above
            #pragma unroll
            for (int k = 0; k < NX; k++) {
                top[k] = wave_max(top[k]);
                if (mine && lane == 0) (k ? a.y1 : a.y0)[o] = fmaxf(top[k], kEps) + sh;
            }
            continue;
        }
        #pragma unroll
        for (int side = 0; side < NX; side++) {
            float gm[ONE ? 1 : NG], top = 0.f;         // maxima per group and per lane (undefined terms never win)
            // (ONE forms the maximum of a group from its terms again: 20 registers less, of which a fifth wavefront is made)
            auto group_max = [&](int e) {
                if constexpr (ONE) return fmaxf(fmaxf(fmaxf(fmaxf(zero, w[e][0]), w[e][1]), w[e][2]), w[e][3]);
                else return gm[e];
            };
            #pragma unroll
            for (int e = 0; e < NG; e++) {
                float v[4];
                bool flag[4];
                terms(side, e, v, flag);
                const float most = fmaxf(fmaxf(fmaxf(v[0], v[1]), v[2]), v[3]);
                if constexpr (!ONE) gm[e] = most;
                top = fmaxf(top, most);
                group_fence(e);
            }
            pass_fence();
            if (OP == kStreamPos) {
                top = wave_max(top);
                int pos = NX == 2 && side == 0 ? (int)kNanId : 0;
                bool found = !(top > kEps);
                // groups in ascending order of their inputs; inside a group VEC: the lane decides before the element,
                // else the element before the lane
                #pragma unroll
                for (int e = 0; e < NG; e++) {
                    if (found || __builtin_amdgcn_ballot_w64(group_max(e) == top) == 0ull) continue;
                    found = true;
                    float v[4];
                    bool flag[4];
                    terms(side, e, v, flag);
                    if (VEC) {
                        int at = 0;
                        bool has = false;
                        #pragma unroll
                        for (int j = 3; j >= 0; j--)
                            if (v[j] == top) { at = (4 * (64 * e + lane) + j) | (flag[j] ? (int)kSign : 0); has = true; }
                        pos = __builtin_amdgcn_readlane(at, (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(has)));
                    } else {
                        #pragma unroll
                        for (int j = 3; j >= 0; j--) {
                            const unsigned long long hit = __builtin_amdgcn_ballot_w64(v[j] == top);
                            const unsigned long long second = __builtin_amdgcn_ballot_w64(flag[j]);
                            if (hit == 0ull) continue;
                            const int l = (int)__builtin_ctzll(hit);
                            pos = (256 * e + 64 * j + l) | ((second >> l) & 1ull ? (int)kSign : 0);
                        }
                    }
                }
                if (mine && lane == 0) {
                    (side ? a.y1 : a.y0)[o] = fmaxf(top, kEps);
                    (side ? a.p1 : a.p0)[o] = pos;
                }
                continue;
            }
            // lower bound of the K-th largest term: the largest bit pattern that K lane maxima reach (their order as
            // numbers is their order as integers), or a smaller one that exactly K reach
            uint32_t bits = 0u;
            int bit = 30;
            if (K <= 64) {                             // the bits that all lane maxima share
                const uint32_t hi = __float_as_uint(wave_max(top)), diff = hi ^ __float_as_uint(wave_min(top));
                bit = 31 - __builtin_clz(diff | 1u);
                bits = hi >> (bit + 1) << (bit + 1);
                if (diff == 0u) { bits = hi; bit = -1; }
            }
            for (; bit >= 0; bit--) {
                const uint32_t t = bits | (1u << bit);
                const int reach = __builtin_popcountll(__builtin_amdgcn_ballot_w64(__float_as_uint(top) >= t));
                if (reach < K) continue;
                bits = t;
                if (reach == K) break;
            }
            const float T = __uint_as_float(bits > 0u ? bits : 1u);   // fewer than K positive lane maxima: every positive term
            int groups = 0, count = 0;                 // groups that reach T, more than 16 of them: not all of them kept
            #pragma unroll
            for (int e = 0; e < NG; e++) {
                const unsigned long long any = __builtin_amdgcn_ballot_w64(group_max(e) >= T);
                if (any == 0ull) continue;
                const int at = groups;
                groups += __builtin_popcountll(any);
                if (groups <= 16 && group_max(e) >= T) {
                    float v[4];
                    bool flag[4];
                    terms(side, e, v, flag);
                    *reinterpret_cast<float4*>(&cand[wave][4 * (at + lanes_below(any))]) = make_float4(v[0], v[1], v[2], v[3]);
                }
            }
            if (groups <= 16) {
                wave_fence();
                // the terms that reach T move to the front
                const float v = lane < 4 * groups ? cand[wave][lane] : 0.f;
                const unsigned long long hit = __builtin_amdgcn_ballot_w64(v >= T);
                count = __builtin_popcountll(hit);
                wave_fence();
                if (v >= T) cand[wave][lanes_below(hit)] = v;
            } else {
                if constexpr (ONE) pass_fence();
                #pragma unroll
                for (int e = 0; e < NG; e++) {
                    if (__builtin_amdgcn_ballot_w64(group_max(e) >= T) == 0ull) continue;
                    float v[4];
                    bool flag[4];
                    terms(side, e, v, flag);
                    #pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const unsigned long long hit = __builtin_amdgcn_ballot_w64(v[j] >= T);
                        const int at = count + lanes_below(hit);
                        if (v[j] >= T && at < 64) cand[wave][at] = v[j];
                        count += __builtin_popcountll(hit);
                    }
                    group_fence(e);
                }
            }
            wave_fence();
            float sorted = 0.f;                        // lane k: the k-th largest term (0 when there are fewer)
            if (count <= 16) {
                // lane 16 q + i counts how many of the terms 4 q .. 4 q + 3 come before term i (as numbers, then as listed)
                if (lane >= count && lane < 16) cand[wave][lane] = 0.f;
                wave_fence();
                const uint32_t own = __float_as_uint(cand[wave][lane & 15]);
                const float4 four = *reinterpret_cast<const float4*>(&cand[wave][lane >> 4 << 2]);
                const int ahead = (lane & 15) - (lane >> 4 << 2);
                int rank = (__float_as_uint(four.x) + (ahead > 0 ? 1u : 0u) > own ? 1 : 0) + (__float_as_uint(four.y) + (ahead > 1 ? 1u : 0u) > own ? 1 : 0) +
                           (__float_as_uint(four.z) + (ahead > 2 ? 1u : 0u) > own ? 1 : 0) + (__float_as_uint(four.w) + (ahead > 3 ? 1u : 0u) > own ? 1 : 0);
                rank += __shfl_xor(rank, 16);
                rank += __shfl_xor(rank, 32);
                wave_fence();
                if (lane < count) cand[wave][rank] = __uint_as_float(own);
                wave_fence();
                sorted = lane < count ? cand[wave][lane] : 0.f;
                wave_fence();
            } else if (count <= 64) {
                const float own = lane < count ? cand[wave][lane] : 0.f;
                int rank = 0;
                for (int j = 0; j < count; j++) {
                    const float other = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(own), j));
                    rank += (other > own || (other == own && j < lane)) ? 1 : 0;
                }
                wave_fence();
                if (lane < count) cand[wave][rank] = own;   // ranks are the numbers 0 .. count - 1
                wave_fence();
                sorted = lane < count ? cand[wave][lane] : 0.f;
                wave_fence();
            } else {
                float below = __builtin_inff();
                bool first = true;
                for (int k = 0; k < K;) {
                    float best = 0.f;
                    #pragma unroll
                    for (int e = 0; e < NG; e++) {
                        float v[4];
                        bool flag[4];
                        terms(side, e, v, flag);
                        #pragma unroll
                        for (int j = 0; j < 4; j++) best = (v[j] < below || (first && v[j] == below)) && v[j] > best ? v[j] : best;
                        group_fence(e);
                    }
                    best = wave_max(best);
                    if (best == 0.f) break;
                    int same = 0;
                    #pragma unroll
                    for (int e = 0; e < NG; e++) {
                        float v[4];
                        bool flag[4];
                        terms(side, e, v, flag);
                        #pragma unroll
                        for (int j = 0; j < 4; j++) same += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v[j] == best));
                        group_fence(e);
                    }
                    if (lane >= k && lane < k + same) sorted = best;
                    k += same;
                    below = best;
                    first = false;
                }
            }
            // every lane weighs its own term; they are added up from the largest on
            const int weighed = __float_as_int(sorted * coef * a.q);
            float ans = kEps;
            for (int k = 0; k < K; k++) ans += __int_as_float(__builtin_amdgcn_readlane(weighed, k));
            if (mine && lane == 0) (side ? a.y1 : a.y0)[o] = ans / (1.f - rest) + sh;
        }
    }
}

template <int NE, int NX, StreamOp OP>
int launch(const FwdArgs& a, int K, hipStream_t stream) {
    // few weight rows: the batch rows are dealt to several workgroups, each of which loads the weight rows again; as many as
    // the device holds at once, so that none waits for another's end (512 x 5120 x 10, K = 10, with three wavefronts per SIMD:
    // 19 us; in 1.3 times as many 26 and, interval bounds, 42 and 55).  Rows of up to 1024 inputs, with twice as many workgroups as for longer ones: 54 x 730 x 730
    // 40 us instead of 50, intervals 75 and 99, l-inf with positions 11 and 14; 32 x 1024 x 1536 52 and 63.  (Three for two against rows
    // of 1025 to 3072 inputs, values of the l-inf distance: 54 x 1500 x 730 12.5 and 13.9, but 7 x 3072 x 2000 15.1 and 13.2.)
    constexpr int kWaves = stream_waves(OP), kPerCu = 4 * stream_resident(NE, NX, OP) / kWaves;
    const int tiles = (a.COg + kWaves - 1) / kWaves * a.G, most = (kPerCu > 1 ? kPerCu : 1) * num_cus();
    auto dealt = [&](int slices) { return slices < a.R ? (a.R + slices - 1) / slices : 1; };
    int rows = dealt(tiles >= most ? 1 : most / tiles);
    // Two to four times as many where that leaves a workgroup fewer rows in all (a selection of the K largest takes about four times as
    // long as loading the weight row): 256 x 10240 x 10, three times one row instead of four, 32 us instead of 37, intervals 66 and 80
    if constexpr (OP == kStreamSort) {
        for (int n = 2, best = 4 * rows + 1; tiles < most && n <= 4; n++) {
            const int r = dealt(n * most / tiles), cost = n * (4 * r + 1);
            if (cost < best) { best = cost; rows = r; }
        }
    }
    const dim3 grid(tiles, (a.R + rows - 1) / rows), block(64 * kWaves);
    note_forward_kernel("row_stream_kernel", kWaves, NE);
    forward_kernel_timer(stream, false);
    const bool vec = a.fast_x && a.fast_w;
    if constexpr (NX == 1 && OP == kStreamSort) {
        // (up to four rounds of workgroups: in many more the selection, which forms the maxima again, weighs more than the loads. 1 x 640 x
        // 20000 17.7 -> 15.4 us, x 200000 325 -> 333)
        if (rows == 1 && tiles <= 4 * most) {
            if (vec) hipLaunchKernelGGL((row_stream_kernel<NE, true, NX, OP, true>), grid, block, 0, stream, a, K);
            else hipLaunchKernelGGL((row_stream_kernel<NE, false, NX, OP, true>), grid, block, 0, stream, a, K);
            forward_kernel_timer(stream, true);
            return check_launch("row_stream_kernel");
        }
    }
    if (vec) hipLaunchKernelGGL((row_stream_kernel<NE, true, NX, OP, false>), grid, block, 0, stream, a, K);
    else hipLaunchKernelGGL((row_stream_kernel<NE, false, NX, OP, false>), grid, block, 0, stream, a, K);
    forward_kernel_timer(stream, true);
    return check_launch("row_stream_kernel");
}

template <int NX, StreamOp OP>
int dispatch(const FwdArgs& a, int K, hipStream_t stream) {
    if (a.CIg <= 16 * 64) return launch<16, NX, OP>(a, K, stream);
    if (a.CIg <= 48 * 64) return launch<48, NX, OP>(a, K, stream);
    if (a.CIg <= 80 * 64) return launch<80, NX, OP>(a, K, stream);
    return launch<160, NX, OP>(a, K, stream);
}

}  // namespace

bool row_stream_sizes_ok(const FwdArgs& a, long long limit) {
    return a.HW == 1 && !a.ci_idx && !a.co_idx && a.CIg <= 160 * 64 && (long long)a.R * a.G * a.COg * a.CIg <= limit;
}

bool row_stream_ok(const FwdArgs& a, long long limit) {
    return row_stream_sizes_ok(a, limit) &&
           (a.mask_mode < 0 || (a.mask_mode == SD_MASK_FACTORED && a.xmask && a.wmask));
}

bool row_stream_sort_ok(const FwdArgs& a) {
    const long long outputs = (long long)a.R * a.G * a.COg, per_input = a.x1 ? 56 : 80;
    long long most = a.x1 ? 3ll << 14 : 1ll << 16;
    // Rows that are loaded value by value meet the tables on their padded copies earlier (in us, streamed -> tables at spreads 0.05 / 0.3
    // / 3 of the inputs, K = 10): values 24 x 2199 x 2199 71 -> 40 / 56 / 67, 32 x 1067 x 1067 36 -> 28 / 42 / 36, 8 x 4443 x 4443 118 ->
    // 71 / 90 / 110, 4 x 4443 x 4443 64 -> 70 / 83 / 61; intervals 16 x 1067 x 1067 54 -> 33 / 46 / 49, 4 x 4443 x 4443 109 -> 75 / 93 /
    // 101, 2 x 4443 x 4443 60 -> 73 / 85 / 121.
    if (!a.fast_w) most = a.x1 ? 1ll << 14 : a.CIg > 48 * 64 ? 1ll << 15 : 3ll << 14;
    return outputs <= most && outputs <= per_input * a.CIg && row_stream_ok(a, 1ll << 62);
}

bool row_stream_sort_before_terms(const FwdArgs& a) {
    const bool longer = a.CIg > 48 * 64;   // (fewer wavefronts at a time)
    const long long outputs = (long long)a.R * a.G * a.COg, per_input = a.x1 ? 100 : 150;
    const long long most = a.x1 ? (longer ? 3ll << 14 : 1ll << 17) : (longer ? 1ll << 17 : 1ll << 18);
    return outputs <= most && outputs <= per_input * a.CIg && row_stream_ok(a, 1ll << 62);
}

int row_stream_linf(const FwdArgs& a, hipStream_t stream) {
    return a.p0 ? dispatch<1, kStreamPos>(a, 0, stream) : dispatch<1, kStreamMax>(a, 0, stream);
}
int row_stream_bound(const FwdArgs& a, hipStream_t stream) {
    return a.p0 ? dispatch<2, kStreamPos>(a, 0, stream) : dispatch<2, kStreamMax>(a, 0, stream);
}
int row_stream_sort(const FwdArgs& a, int K, hipStream_t stream) {
    return a.x1 ? dispatch<2, kStreamSort>(a, K, stream) : dispatch<1, kStreamSort>(a, K, stream);
}

}  // namespace sd
