// Candidate tables: which inputs of a row can matter to any row of a tile of the other operand (sort_cols.hip: weight rows
// against tiles of 128 batch rows; row_cands.hip: batch rows against tiles of 128 weight rows).
//
// Over a tile the terms of (row, input) are bracketed by the ranges of the tile's column.  K disjoint groups of inputs whose
// best lower bound is at least t hold K terms that are at least t in every row of the tile (fp32 subtraction is monotone, so
// the brackets hold for the rounded terms), which bounds the K-th largest term of every output from below; an input is marked
// when the largest its term can be reaches that bound and is positive (an undefined one is not: its term is left out).
//
// One kernel does both steps for a few rows: a lane owns four consecutive inputs of every 256, so a row is read 1 KB at a
// time, its 64 groups are the lanes, the bound is selected with ballots, and a ballot over the second reading of the row is a
// table word.  A wavefront takes RW rows against NT tiles, with the ranges of the tiles staged in LDS for the workgroup.
// 63 us at 512 x 5120 x 5120 (K = 10), 44 us at 512 x 3072 x 5120 (K = 1): the two readings of the rows, 210 MB at 3.3 TB/s,
// beside about as much vector work.  (Four launches before, a lane to a row: lists of the K largest chunk maxima per slice
// 34, their merge 10, the words 32, the sum of the marks 5.  Two launches with the ranges as scalar operands: 34 + 43.)
#pragma once
#include "common.h"

namespace sd {

constexpr int kTableBlock = 256;     // inputs of one block: four per lane
constexpr int kTableSlice = 512;     // inputs whose ranges are staged at a time
constexpr int kTableWaves = 4;       // wavefronts of a workgroup

// words of a row's table: eight per block of 256 inputs, of which word 2 j + h holds, for its lanes 32 h .. 32 h + 31, the
// inputs 4 lane + j
inline __host__ __device__ int table_row_words(int N) { return (N + kTableBlock - 1) / kTableBlock * 8; }

// the marks of inputs 32 c .. 32 c + 31, one bit each in ascending order
__device__ __forceinline__ uint32_t table_word(const uint32_t* __restrict__ rowbits, int c) {
    const uint8_t* p = reinterpret_cast<const uint8_t*>(rowbits + (size_t)(c >> 3) * 8) + (c & 7);
    uint32_t word = 0;
    #pragma unroll
    for (int j = 0; j < 4; j++) {
        uint32_t x = p[8 * j];   // bit t: input 32 c + 4 t + j
        x = (x | (x << 12)) & 0x000f000fu;
        x = (x | (x << 6)) & 0x03030303u;
        x = (x | (x << 3)) & 0x11111111u;
        word |= x << j;
    }
    return word;
}

struct TableArgs {
    const float* v1;                // rows (R, N); PAIR: the upper of two values
    const float* v2;                // PAIR: the lower
    const uint32_t* keep;           // MASK: one word per (row, 32 inputs)
    const float* ranges;            // [tiles][N] of (min, max), TWO without PAIR: of (min l, max l, min u, max u)
    int R, Rp, N, tiles, K;
    float* low;                     // [tiles][TWO ? 2 : 1][Rp]
    uint32_t* bits;                 // [tiles][Rp][table_row_words(N)]
};

// `v` with lane `lane` replaced by a wave-uniform value (the instruction has no builtin in this compiler)
extern "C" __device__ int sd_writelane(int value, int lane, int v) __asm("llvm.amdgcn.writelane.i32");

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

// Row values v1, v2 (equal unless PAIR) against ranges (lo, hi): lowest and largest a term max(v1 - x, x - v2) can be.
// TWO: a bound for each result of the intervals: marks for max(v1 - x, x - v2) and for max(v2 - x, x - v1) (PAIR), or ranges
// (min l, max l, min u, max u) of an interval [l, u] against one value v, marks for max(u - v, v - l) and for max(l - v, v - u).
// Returns the marks of a wavefront's rows.
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
            if constexpr (PAIR) { if (vl[e] > vu[e]) vl[e] = vu[e] = (vl[e] + vu[e]) * 0.5f; }   // inverted interval: midpoint
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
                const bool there = r0 + r < a.R && t0 + t < a.tiles;
                if (lane == 0 && there) a.low[((size_t)(t0 + t) * NL + k) * a.Rp + r0 + r] = v;
                // only a positive term counts; rows and tiles past the last one have no marks
                best[r][t][k] = !there ? __builtin_nanf("") : v > 0.f ? v : 1.401298464e-45f;
            }
        }
    }
    int marks = 0;
    const int unit = lane >> 4, ur = unit / NT, ut = unit % NT;   // the (row, tile) whose words of a slice this lane stores
    const bool mine = unit < RW * NT && r0 + ur < a.R && t0 + ut < a.tiles;
    uint32_t* dst = a.bits + ((size_t)(t0 + ut) * a.Rp + r0 + ur) * ((size_t)NB * 8) + (lane & 15);
    pass([&](int n0, const float (&vu)[2][RW][4], const float (&vl)[2][RW][4]) __attribute__((always_inline)) {
        uint32_t out = 0;
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
                    for (int e = 0; e < 4; e++) {
                        bool mark;
                        if constexpr (TWO && PAIR) {
                            mark = fmaxf(vu[b][r][e] - p0[e], p1[e] - vl[b][r][e]) >= best[r][t][0];
                            mark = mark || fmaxf(vl[b][r][e] - p0[e], p1[e] - vu[b][r][e]) >= best[r][t][1];
                        } else if constexpr (TWO) {
                            mark = fmaxf(vu[b][r][e] - p0[e], p3[e] - vl[b][r][e]) >= best[r][t][0];
                            mark = mark || fmaxf(p1[e] - vu[b][r][e], vl[b][r][e] - p2[e]) >= best[r][t][1];
                        } else mark = fmaxf(vu[b][r][e] - p0[e], p1[e] - vl[b][r][e]) >= best[r][t][0];
                        const unsigned long long m = __builtin_amdgcn_ballot_w64(mark);
                        const int at = (r * NT + t) * 16 + b * 8 + 2 * e;
                        marks += __builtin_popcountll(m);
                        out = (uint32_t)sd_writelane((int)(uint32_t)m, at, (int)out);
                        out = (uint32_t)sd_writelane((int)(uint32_t)(m >> 32), at + 1, (int)out);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);   // (all ballots of a slice at once would not fit the scalar registers)
            }
        }
        if (mine && n0 / kTableBlock + ((lane >> 3) & 1) < NB) dst[(size_t)(n0 / kTableBlock) * 8] = out;
    });
    return marks;
}

// Adds up the marks (one number per wavefront) of all workgroups; true in one thread of the workgroup that was the last, with the
// sum in *total.  `sum` counts the workgroups in its upper 24 bits, so that one atomic does both and nothing has to be ordered
// (a fence of device scope writes the die's whole cache back: 800 workgroups with one each took 50 us longer).  The marks of a
// layer are below 2^40 and its workgroups below 2^24 while its operands can be indexed with 31 bits.
__device__ __forceinline__ bool add_marks(unsigned long long* sum, int marks, unsigned long long* total) {
    __shared__ int part[kTableWaves];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = marks;
    __syncthreads();
    if (threadIdx.x != 0) return false;
    unsigned long long s = 1ull << 40;
    #pragma unroll
    for (int i = 0; i < kTableWaves; i++) s += (unsigned long long)part[i];
    const unsigned long long all = atomicAdd(sum, s) + s;
    *total = all & ((1ull << 40) - 1ull);
    return all >> 40 == (unsigned long long)gridDim.x * gridDim.y * gridDim.z;
}

// What a table per weight row leaves for the choice of kernel.  All zero before the ranges are taken.
struct TableCount {
    unsigned long long marks;       // all ones when the table was not built
    unsigned long long above;       // 1 when the marks are above the limit
    float stat[2];                  // probe: widths of the input columns over all batch tiles; of the same columns over 16 weight rows
    unsigned long long sum;         // see add_marks
};

}  // namespace sd
