// Candidate tables: which inputs of a row can matter to any row of a tile of the other operand (sort_cols.hip: weight rows
// against tiles of 128 batch rows; row_cands.hip: batch rows against tiles of 128 weight rows).
//
// Over a tile the terms of (row, input) are bracketed by the ranges of the tile's column.  K disjoint groups of inputs whose
// best lower bound is at least t hold K terms that are at least t in every row of the tile (fp32 subtraction is monotone, so
// the brackets hold for the rounded terms), which bounds the K-th largest term of every output from below; an input is marked
// when the largest its term can be reaches that bound and is positive (an undefined one is not: its term is left out).
//
// One kernel does both steps for a few rows: a lane owns four consecutive inputs of every 256, so a row is read 1 KB at a
// time, its 64 groups are the lanes, and the bound is selected with ballots.  Rows of up to 12288 inputs are read once and kept
// in registers from the bound to the marks (stream_tables), longer ones twice (build_tables).  512 x 5120 x 5120, K = 10: 42 us
// (105 MB of weights at 2.5 TB/s; about 12 us of vector work, 19 dependent steps of selection per two rows, 164 KB of ranges
// per compute unit to begin with), 64 with the rows read twice and the ranges staged in LDS for every four of them;
// interval bounds of 256 x 10240 x 10240 132 us instead of 238.
#pragma once
#include "common.h"

namespace sd {

constexpr int kTableBlock = 256;     // inputs of one block: four per lane
constexpr int kTableSlice = 512;     // inputs whose ranges are staged at a time
constexpr int kTableWaves = 4;       // wavefronts of a workgroup
constexpr int kStreamWaves = 16;     // most wavefronts of a workgroup of stream_tables

// words of a row's table: one bit per input in ascending order, whole blocks of 256 inputs
inline __host__ __device__ int table_row_words(int N) { return (N + kTableBlock - 1) / kTableBlock * 8; }

struct TableArgs {
    const float* v1;                // rows (R, N); PAIR: the upper of two values
    const float* v2;                // PAIR: the lower
    const uint32_t* keep;           // MASK: one word per (row, 32 inputs)
    const float* ranges;            // [tiles][N] of (min, max), TWO without PAIR: of (min l, max l, min u, max u)
    int R, Rp, N, tiles, K;
    float* low;                     // [tiles][TWO ? 2 : 1][Rp]
    uint32_t* bits;                 // [tiles][Rp][table_row_words(N)]
};

// Marks are collected without the scalar unit: the sign of (term - bound) moves into a register of the lane, four inputs of up to
// eight rows and tiles (units) to a word, and the eight lanes that hold the 32 inputs of a table word exchange their nibbles.
// (Ballots and two lane writes per 64 inputs took 6 vector and 3 scalar instructions instead of 5, and spilled scalars.)
// `d`: not negative where the input is marked; nor is it undefined.  Units and inputs go in descending order.
__device__ __forceinline__ void push_mark(uint32_t& not_marked, float d) {
    not_marked = __builtin_amdgcn_alignbit(not_marked, __float_as_uint(d), 31);
}
// lane 8 w + u: word w (32 inputs) of unit u, from the lanes 8 w + i that hold nibble u of every unit's inputs 4 i .. 4 i + 3
__device__ __forceinline__ uint32_t exchange_marks(uint32_t x, int lane) {
    int o = __builtin_amdgcn_update_dpp(0, (int)x, 0x104, 0xf, 0x5, false);   // row_shl:4 into the even banks
    o = __builtin_amdgcn_update_dpp(o, (int)x, 0x114, 0xf, 0xa, false);       // row_shr:4 into the odd ones
    x = __builtin_amdgcn_perm((uint32_t)o, x, lane & 4 ? 0x03020706u : 0x05040100u);
    o = __builtin_amdgcn_update_dpp(0, (int)x, 0x4e, 0xf, 0xf, false);        // lane ^ 2
    x = __builtin_amdgcn_perm((uint32_t)o, x, lane & 2 ? 0x03070105u : 0x06020400u);
    o = __builtin_amdgcn_update_dpp(0, (int)x, 0xb1, 0xf, 0xf, false);        // lane ^ 1
    const uint32_t turned = __builtin_amdgcn_alignbit((uint32_t)o, (uint32_t)o, lane & 1 ? 4 : 28);
    const uint32_t own = lane & 1 ? 0xf0f0f0f0u : 0x0f0f0f0fu;
    return (x & own) | (turned & ~own);
}
// what marks are compared with: a term only counts when it is positive, and the difference from the bound is to be defined
__device__ __forceinline__ float mark_bound(float kth) { return fminf(kth > 0.f ? kth : 1.401298464e-45f, 3.402823466e38f); }

// An inverted interval becomes its midpoint.  One bound for both results (TWO = false) rests on the term of the upper one being at
// least that of the lower one, which does not hold where an end is undefined (each result then takes the term of the other end):
// such an input is given no bound and is always marked.
template <bool TWO>
__device__ __forceinline__ void repair_row(float& l, float& u) {
    if (l > u) l = u = (l + u) * 0.5f;
    if constexpr (!TWO) { if (!(l <= u)) { l = -__builtin_inff(); u = __builtin_inff(); } }
}

// largest value over the wavefront of floats that are not negative
__device__ __forceinline__ float wave_max_nonneg(float f) {
    int v = __builtin_bit_cast(int, f);
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));   // row_shr:1
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));   // row_shr:2
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));   // row_shr:4
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));   // row_shr:8
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));   // row_bcast:15 into rows 1 and 3
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));   // row_bcast:31 into rows 2 and 3
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(v, 63));
}

// K-th largest over the wavefront of floats that are not negative: the bits of the result from the top, by counting; the last 11
// are left out, which lowers a bound by less than 0.05 %.  (19 dependent steps; ten of two bits each measured 3 us more per
// 512 x 5120 x 5120 layer, for their scalar instructions.)
__device__ __forceinline__ float wave_kth_nonneg(float f, int K) {
    const int v = __float_as_int(f);
    int kth = 0;
    #pragma unroll 1
    for (int bit = 30; bit > 11; bit--) {
        const int c = kth | (1 << bit);
        kth = __builtin_popcountll(__builtin_amdgcn_ballot_w64(v >= c)) >= K ? c : kth;
    }
    return __int_as_float(kth);
}

// Row values v1, v2 (equal unless PAIR) against ranges (lo, hi): lowest and largest a term max(v1 - x, x - v2) can be.
// TWO: a bound for each result of the intervals: marks for max(v1 - x, x - v2) and for max(v2 - x, x - v1) (PAIR), or ranges
// (min l, max l, min u, max u) of an interval [l, u] against one value v, marks for max(u - v, v - l) and for max(l - v, v - u).
// Returns the marks that the lane has stored.
template <int RW, int NT, bool PAIR, bool TWO, bool MASK>
__device__ __forceinline__ int build_tables(const TableArgs& a, int bx, int by, float* smem) {
    static_assert(RW * NT <= 4 && kTableSlice == 2 * kTableBlock, "");
    constexpr int NP = TWO && !PAIR ? 4 : 2, NL = TWO ? 2 : 1, T = 64 * kTableWaves, PER = NP * kTableSlice / T;
    typedef float Plane[NP][kTableSlice];
    Plane* rg = reinterpret_cast<Plane*>(smem);   // [NT]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int N = a.N, NB = (N + kTableBlock - 1) / kTableBlock, NCH = N / 32;
    const int r0 = (bx * kTableWaves + wave) * RW, t0 = by * NT;
    int row[RW];
    #pragma unroll
    for (int r = 0; r < RW; r++) row[r] = r0 + r < a.R ? r0 + r : a.R - 1;

    float4 u[RW][2], l[PAIR ? RW : 1][2];        // the slice after the one in use
    uint32_t kw[MASK ? RW : 1][2];
    float pr[NT][PER];
    auto fetch = [&](int n0) __attribute__((always_inline)) {
        #pragma unroll
        for (int b = 0; b < 2; b++) {
            int n = n0 + b * kTableBlock + 4 * lane;
            n = n < N ? n : N - 4;
            #pragma unroll
            for (int r = 0; r < RW; r++) {
                u[r][b] = *reinterpret_cast<const float4*>(a.v1 + (size_t)row[r] * N + n);
                if constexpr (PAIR) l[r][b] = *reinterpret_cast<const float4*>(a.v2 + (size_t)row[r] * N + n);
                if constexpr (MASK) kw[r][b] = a.keep[(size_t)row[r] * NCH + (n >> 5)] >> (n & 31);
            }
        }
        #pragma unroll
        for (int t = 0; t < NT; t++) {
            const int tt = t0 + t < a.tiles ? t0 + t : a.tiles - 1;
            const float* src = a.ranges + ((size_t)tt * N + n0) * NP;
            const int left = (N - n0) * NP;   // floats of the slice that exist; undefined behind them: no bound and no mark
            #pragma unroll
            for (int i = 0; i < PER; i++) {
                const float v = src[tid + T * i < left ? tid + T * i : left - 1];
                pr[t][i] = tid + T * i < left ? v : __builtin_nanf("");
            }
        }
    };
    auto stage = [&]() __attribute__((always_inline)) {
        #pragma unroll
        for (int t = 0; t < NT; t++) {
            #pragma unroll
            for (int i = 0; i < PER; i++) { const int e = tid + T * i; rg[t][e % NP][e / NP] = pr[t][i]; }
        }
    };
    // (u, l) of this lane's four inputs of block b
    auto values = [&](int b, int r, float (&vu)[4], float (&vl)[4]) __attribute__((always_inline)) {
        const float4 x = u[r][b];
        vu[0] = x.x; vu[1] = x.y; vu[2] = x.z; vu[3] = x.w;
        if constexpr (PAIR) {
            const float4 y = l[r][b];
            vl[0] = y.x; vl[1] = y.y; vl[2] = y.z; vl[3] = y.w;
        }
        #pragma unroll
        for (int e = 0; e < 4; e++) {
            if constexpr (PAIR) repair_row<TWO>(vl[e], vu[e]);
            if constexpr (MASK) {   // undefined where the row does not keep the input
                const bool k = (kw[r][b] >> e) & 1u;
                vu[e] = k ? vu[e] : __builtin_nanf("");
                if constexpr (PAIR) vl[e] = k ? vl[e] : __builtin_nanf("");
            }
            if constexpr (!PAIR) vl[e] = vu[e];
        }
    };
    // goes over the rows once: body(slice, values of the rows), with the ranges of the slice in LDS
    auto pass = [&](auto&& body) __attribute__((always_inline)) {
        fetch(0);
        for (int n0 = 0; n0 < N; n0 += kTableSlice) {
            float vu[2][RW][4], vl[2][RW][4];
            __syncthreads();
            stage();
            #pragma unroll
            for (int b = 0; b < 2; b++) {
                #pragma unroll
                for (int r = 0; r < RW; r++) values(b, r, vu[b][r], vl[b][r]);
            }
            if (n0 + kTableSlice < N) fetch(n0 + kTableSlice);
            __syncthreads();
            body(n0, vu, vl);
        }
    };
    auto range4 = [&](int t, int p, int b, float (&o)[4]) __attribute__((always_inline)) {
        const float4 x = *reinterpret_cast<const float4*>(&rg[t][p][b * kTableBlock + 4 * lane]);
        o[0] = x.x; o[1] = x.y; o[2] = x.z; o[3] = x.w;
    };

    float best[RW][NT][NL];
    #pragma unroll
    for (int r = 0; r < RW; r++) {
        #pragma unroll
        for (int t = 0; t < NT; t++) {
            #pragma unroll
            for (int k = 0; k < NL; k++) best[r][t][k] = 0.f;
        }
    }
    pass([&](int, const float (&vu)[2][RW][4], const float (&vl)[2][RW][4]) __attribute__((always_inline)) {
        #pragma unroll
        for (int b = 0; b < 2; b++) {
            #pragma unroll
            for (int t = 0; t < NT; t++) {
                float p0[4], p1[4], p2[4], p3[4];
                range4(t, 0, b, p0); range4(t, 1, b, p1);
                if constexpr (TWO && !PAIR) { range4(t, 2, b, p2); range4(t, 3, b, p3); }
                #pragma unroll
                for (int r = 0; r < RW; r++) {
                    #pragma unroll
                    for (int e = 0; e < 4; e++) {   // (fmaxf drops undefined differences)
                        if constexpr (TWO && PAIR) {
                            best[r][t][0] = fmaxf(fmaxf(best[r][t][0], vu[b][r][e] - p1[e]), p0[e] - vl[b][r][e]);
                            best[r][t][1] = fmaxf(fmaxf(best[r][t][1], vl[b][r][e] - p1[e]), p0[e] - vu[b][r][e]);
                        } else if constexpr (TWO) {
                            best[r][t][0] = fmaxf(fmaxf(best[r][t][0], vu[b][r][e] - p1[e]), p2[e] - vl[b][r][e]);
                            best[r][t][1] = fmaxf(fmaxf(best[r][t][1], p0[e] - vu[b][r][e]), vl[b][r][e] - p3[e]);
                        } else {
                            // (PAIR: the lower bound of the term max(l - x, x - u), which is what marks for either bound are taken against)
                            best[r][t][0] = fmaxf(fmaxf(best[r][t][0], vl[b][r][e] - p1[e]), p0[e] - vu[b][r][e]);
                        }
                    }
                }
            }
        }
    });
    // K-th largest over the lanes: the bits of the result from the top, by counting; the last 11 are left out, which lowers a
    // bound by less than 0.05 % (19 steps, those of all rows and tiles side by side)
    int kth[RW][NT][NL];
    #pragma unroll
    for (int r = 0; r < RW; r++) {
        #pragma unroll
        for (int t = 0; t < NT; t++) {
            #pragma unroll
            for (int k = 0; k < NL; k++) kth[r][t][k] = a.K == 1 ? __float_as_int(wave_max_nonneg(best[r][t][k])) : 0;
        }
    }
    if (a.K != 1) {
        #pragma unroll 1
        for (int bit = 30; bit > 11; bit--) {
            #pragma unroll
            for (int r = 0; r < RW; r++) {
                #pragma unroll
                for (int t = 0; t < NT; t++) {
                    #pragma unroll
                    for (int k = 0; k < NL; k++) {
                        const int c = kth[r][t][k] | (1 << bit);
                        const bool more = __builtin_popcountll(__builtin_amdgcn_ballot_w64(__float_as_int(best[r][t][k]) >= c)) >= a.K;
                        kth[r][t][k] = more ? c : kth[r][t][k];
                    }
                }
            }
        }
    }
    #pragma unroll
    for (int r = 0; r < RW; r++) {
        #pragma unroll
        for (int t = 0; t < NT; t++) {
            #pragma unroll
            for (int k = 0; k < NL; k++) {
                const float v = __int_as_float(kth[r][t][k]);
                if (lane == 0 && r0 + r < a.R && t0 + t < a.tiles) a.low[((size_t)(t0 + t) * NL + k) * a.Rp + r0 + r] = v;
                best[r][t][k] = mark_bound(v);
            }
        }
    }
    int marks = 0;
    // the (block of the slice, row, tile) whose words this lane stores
    const int unit = lane & 7, ub = unit / (RW * NT), ur = unit / NT % RW, ut = unit % NT;
    const bool mine = ub < 2 && r0 + ur < a.R && t0 + ut < a.tiles;
    uint32_t* dst = a.bits + ((size_t)(t0 + ut) * a.Rp + r0 + ur) * ((size_t)NB * 8) + ub * 8 + (lane >> 3);
    pass([&](int n0, const float (&vu)[2][RW][4], const float (&vl)[2][RW][4]) __attribute__((always_inline)) {
        uint32_t out = 0;
        #pragma unroll
        for (int b = 1; b >= 0; b--) {
            #pragma unroll
            for (int r = RW - 1; r >= 0; r--) {
                #pragma unroll
                for (int t = NT - 1; t >= 0; t--) {
                    float p0[4], p1[4], p2[4], p3[4];
                    range4(t, 0, b, p0); range4(t, 1, b, p1);
                    if constexpr (TWO && !PAIR) { range4(t, 2, b, p2); range4(t, 3, b, p3); }
                    #pragma unroll
                    for (int e = 3; e >= 0; e--) {
                        // (an undefined term is not marked)
                        float d;
                        if constexpr (TWO && PAIR) {
                            d = fmaxf(fmaxf(vu[b][r][e] - p0[e], p1[e] - vl[b][r][e]), 0.f) - best[r][t][0];
                            d = fmaxf(d, fmaxf(fmaxf(vl[b][r][e] - p0[e], p1[e] - vu[b][r][e]), 0.f) - best[r][t][1]);
                        } else if constexpr (TWO) {
                            d = fmaxf(fmaxf(vu[b][r][e] - p0[e], p3[e] - vl[b][r][e]), 0.f) - best[r][t][0];
                            d = fmaxf(d, fmaxf(fmaxf(p1[e] - vu[b][r][e], vl[b][r][e] - p2[e]), 0.f) - best[r][t][1]);
                        } else d = fmaxf(fmaxf(vu[b][r][e] - p0[e], p1[e] - vl[b][r][e]), 0.f) - best[r][t][0];
                        push_mark(out, d);
                    }
                }
            }
        }
        out = exchange_marks(~out, lane);
        if (mine && n0 / kTableBlock + ub < NB) {
            dst[(size_t)(n0 / kTableBlock) * 8] = out;
            marks += __builtin_popcount(out);
        }
    });
    return marks;
}

// The same for rows of at most 3 * 16 * 256 inputs, which pass once: the wavefronts of a workgroup share a row between them (up to
// J blocks of 256 inputs each), keep the ranges of their inputs against NT tiles in registers for as long as the workgroup lives,
// and the inputs of R rows from the bound to the marks, with the next R rows on their way.  A lane's groups are the same as above
// (the wavefronts' maxima meet in LDS), and so are the bounds and the words.
// smem: waves * U * 64 floats, then U floats, U = R * NT * (TWO ? 2 : 1).
template <int J, int R, int NT, bool PAIR, bool TWO, bool MASK>
__device__ __forceinline__ int stream_tables(const TableArgs& a, int bx, int nbx, int by, float* smem) {
    static_assert(R * NT <= 8, "a word of the table per lane and block");
    constexpr int NP = TWO && !PAIR ? 4 : 2, NL = TWO ? 2 : 1, U = R * NT * NL;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = (int)(blockDim.x >> 6);
    const int N = a.N, NB = (N + kTableBlock - 1) / kTableBlock, NCH = N / 32, t0 = by * NT;
    float* part = smem;
    float* bound = smem + waves * U * 64;

    int at[J];                      // the lane's inputs
    bool used[J];
    float rg[NT][NP][J][4];
    #pragma unroll
    for (int j = 0; j < J; j++) {
        const int n = (wave + j * waves) * kTableBlock + 4 * lane;
        used[j] = j == 0 || wave + j * waves < NB;   // (wave-uniform; each wavefront has a block)
        at[j] = n < N ? n : N - 4;
        #pragma unroll
        for (int t = 0; t < NT; t++) {
            const int tt = t0 + t < a.tiles ? t0 + t : a.tiles - 1;
            const float4* src = reinterpret_cast<const float4*>(a.ranges + ((size_t)tt * N + at[j]) * NP);
            float v[4 * NP];
            #pragma unroll
            for (int i = 0; i < NP; i++) {
                const float4 x = src[i];
                v[4 * i] = x.x; v[4 * i + 1] = x.y; v[4 * i + 2] = x.z; v[4 * i + 3] = x.w;
            }
            #pragma unroll
            for (int e = 0; e < 4; e++) {
                #pragma unroll
                for (int p = 0; p < NP; p++) rg[t][p][j][e] = n < N ? v[e * NP + p] : __builtin_nanf("");   // no bound, no mark
            }
        }
    }

    float4 u[R][J], l[PAIR ? R : 1][J];          // the rows after those in use
    uint32_t kw[MASK ? R : 1][J];
    auto fetch = [&](int r0) __attribute__((always_inline)) {
        #pragma unroll
        for (int r = 0; r < R; r++) {
            const size_t row = r0 + r < a.R ? r0 + r : a.R - 1;
            #pragma unroll
            for (int j = 0; j < J; j++) {
                if (!used[j]) continue;
                u[r][j] = *reinterpret_cast<const float4*>(a.v1 + row * N + at[j]);
                if constexpr (PAIR) l[r][j] = *reinterpret_cast<const float4*>(a.v2 + row * N + at[j]);
                if constexpr (MASK) kw[r][j] = a.keep[row * NCH + (at[j] >> 5)];
            }
        }
    };
    int marks = 0;
    const int unit = lane & 7, ur = unit / NT, ut = unit % NT;   // the (row, tile) whose words of a block this lane stores
    fetch(bx * R);
    for (int r0 = bx * R; r0 < a.R; r0 += nbx * R) {
        float vu[R][J][4], vl[PAIR ? R : 1][J][4];
        #pragma unroll
        for (int r = 0; r < R; r++) {
            #pragma unroll
            for (int j = 0; j < J; j++) {
                const float4 x = u[r][j];
                vu[r][j][0] = x.x; vu[r][j][1] = x.y; vu[r][j][2] = x.z; vu[r][j][3] = x.w;
                if constexpr (PAIR) {
                    const float4 y = l[r][j];
                    vl[r][j][0] = y.x; vl[r][j][1] = y.y; vl[r][j][2] = y.z; vl[r][j][3] = y.w;
                }
                #pragma unroll
                for (int e = 0; e < 4; e++) {
                    if constexpr (PAIR) repair_row<TWO>(vl[r][j][e], vu[r][j][e]);
                    if constexpr (MASK) {   // undefined where the row does not keep the input
                        const bool k = (kw[r][j] >> ((at[j] & 31) + e)) & 1u;
                        vu[r][j][e] = k ? vu[r][j][e] : __builtin_nanf("");
                        if constexpr (PAIR) vl[r][j][e] = k ? vl[r][j][e] : __builtin_nanf("");
                    }
                }
            }
        }
        if (r0 + nbx * R < a.R) fetch(r0 + nbx * R);
        float best[R][NT][NL];
        #pragma unroll
        for (int r = 0; r < R; r++) {
            #pragma unroll
            for (int t = 0; t < NT; t++) {
                #pragma unroll
                for (int k = 0; k < NL; k++) best[r][t][k] = 0.f;
                #pragma unroll
                for (int j = 0; j < J; j++) {
                    if (!used[j]) continue;
                    #pragma unroll
                    for (int e = 0; e < 4; e++) {   // (fmaxf drops undefined differences)
                        const float hi = vu[r][j][e], lo = PAIR ? vl[PAIR ? r : 0][j][e] : hi, p0 = rg[t][0][j][e], p1 = rg[t][1][j][e];
                        if constexpr (TWO && PAIR) {
                            best[r][t][0] = fmaxf(fmaxf(best[r][t][0], hi - p1), p0 - lo);
                            best[r][t][1] = fmaxf(fmaxf(best[r][t][1], lo - p1), p0 - hi);
                        } else if constexpr (TWO) {
                            best[r][t][0] = fmaxf(fmaxf(best[r][t][0], hi - p1), rg[t][2][j][e] - hi);
                            best[r][t][1] = fmaxf(fmaxf(best[r][t][1], p0 - hi), hi - rg[t][3][j][e]);
                        } else best[r][t][0] = fmaxf(fmaxf(best[r][t][0], lo - p1), p0 - hi);
                    }
                }
            }
        }
        #pragma unroll
        for (int r = 0; r < R; r++) {
            #pragma unroll
            for (int t = 0; t < NT; t++) {
                #pragma unroll
                for (int k = 0; k < NL; k++) part[(wave * U + (r * NT + t) * NL + k) * 64 + lane] = best[r][t][k];
            }
        }
        __syncthreads();
        for (int i = wave; i < U; i += waves) {
            float v = 0.f;   // (eight reads at a time: one after the other they took 1 us)
            #pragma unroll 1
            for (int k0 = 0; k0 < waves; k0 += 8) {
                float w[8];
                #pragma unroll
                for (int k = 0; k < 8; k++) w[k] = part[((k0 + k < waves ? k0 + k : 0) * U + i) * 64 + lane];
                #pragma unroll
                for (int k = 0; k < 8; k++) v = fmaxf(v, w[k]);
            }
            const float kth = a.K == 1 ? wave_max_nonneg(v) : wave_kth_nonneg(v, a.K);
            const int r = r0 + i / NL / NT, t = t0 + i / NL % NT;
            if (lane == 0) {
                if (r < a.R && t < a.tiles) a.low[((size_t)t * NL + i % NL) * a.Rp + r] = kth;
                bound[i] = mark_bound(kth);
            }
        }
        __syncthreads();
        uint32_t* dst = a.bits + ((size_t)(t0 + ut) * a.Rp + r0 + ur) * ((size_t)NB * 8) + (lane >> 3);
        const bool mine = unit < R * NT && r0 + ur < a.R && t0 + ut < a.tiles;
        #pragma unroll
        for (int j = 0; j < J; j++) {
            if (!used[j]) continue;
            uint32_t out = 0;
            #pragma unroll
            for (int r = R - 1; r >= 0; r--) {
                #pragma unroll
                for (int t = NT - 1; t >= 0; t--) {
                    const float b0 = bound[(r * NT + t) * NL], b1 = bound[(r * NT + t) * NL + NL - 1];
                    #pragma unroll
                    for (int e = 3; e >= 0; e--) {
                        const float hi = vu[r][j][e], lo = PAIR ? vl[PAIR ? r : 0][j][e] : hi, p0 = rg[t][0][j][e], p1 = rg[t][1][j][e];
                        float d;   // (an undefined term is not marked)
                        if constexpr (TWO && PAIR) {
                            d = fmaxf(fmaxf(hi - p0, p1 - lo), 0.f) - b0;
                            d = fmaxf(d, fmaxf(fmaxf(lo - p0, p1 - hi), 0.f) - b1);
                        } else if constexpr (TWO) {
                            d = fmaxf(fmaxf(hi - p0, rg[t][3][j][e] - hi), 0.f) - b0;
                            d = fmaxf(d, fmaxf(fmaxf(p1 - hi, hi - rg[t][2][j][e]), 0.f) - b1);
                        } else d = fmaxf(fmaxf(hi - p0, p1 - lo), 0.f) - b0;
                        push_mark(out, d);
                    }
                }
            }
            out = exchange_marks(~out, lane);
            if (mine) {
                dst[(size_t)(wave + j * waves) * 8] = out;
                marks += __builtin_popcount(out);
            }
        }
    }
    return marks;
}

// Workgroups of stream_tables: J for the row, the wavefronts that share it, and as many groups of rows as fill the device once
// (a workgroup's ranges are fetched once per group).
struct StreamShape { int waves, rows; };
inline int stream_blocks(int N) { return ((N + kTableBlock - 1) / kTableBlock + kStreamWaves - 1) / kStreamWaves; }
inline StreamShape stream_shape(int N, int R, int rows, int tile_groups) {
    const int NB = (N + kTableBlock - 1) / kTableBlock, waves = NB < kStreamWaves ? NB : kStreamWaves;
    const int batches = (rows + R - 1) / R, wgs = num_cus() * (kStreamWaves / waves);
    const int most = wgs / tile_groups > 1 ? wgs / tile_groups : 1, per = (batches + most - 1) / most;
    return {waves, (batches + per - 1) / per};
}
inline size_t stream_lds(int waves, int U) { return ((size_t)waves * 64 + 1) * U * 4; }

// sum over the wavefront
__device__ __forceinline__ int wave_total(int v) {
    #pragma unroll
    for (int o = 32; o; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Adds up the marks (one number per work-item) of all workgroups; true in one thread of the workgroup that was the last, with the
// sum in *total.  `sum` counts the workgroups in its upper 24 bits, so that one atomic does both and nothing has to be ordered
// (a fence of device scope writes the die's whole cache back: 800 workgroups with one each took 50 us longer).  The marks of a
// layer are below 2^40 and its workgroups below 2^24 while its operands can be indexed with 31 bits.
__device__ __forceinline__ bool add_marks(unsigned long long* sum, int marks, unsigned long long* total) {
    __shared__ int part[kStreamWaves];
    marks = wave_total(marks);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = marks;
    __syncthreads();
    if (threadIdx.x != 0) return false;
    unsigned long long s = 1ull << 40;
    for (int i = 0; i < (int)(blockDim.x >> 6); i++) s += (unsigned long long)part[i];
    const unsigned long long all = atomicAdd(sum, s) + s;
    *total = all & ((1ull << 40) - 1ull);
    return all >> 40 == (unsigned long long)gridDim.x * gridDim.y * gridDim.z;
}

// What a table per weight row leaves for the choice of kernel.
struct TableCount {
    unsigned long long marks;       // all ones when the table was not built
    unsigned long long above;       // 1 when the marks are above the limit
    float stat[2];                  // probe: widths of the input columns over all batch tiles; of the same columns over 16 weight rows
    unsigned long long sum;         // see add_marks
};

}  // namespace sd
