// Sort neuron, its interval bounds and the l-inf forward from candidate tables per batch row (see row_cands.h).
#include "row_cands.h"
#include <cstddef>
#include <type_traits>
#include "cand_tables.h"
#include "cand_walk.h"
#include "fwd_tile.h"

namespace sd {

namespace {

constexpr int kChunk = kRowCandsChunk;
constexpr int kTileW = 128;          // weight rows of a tile: 64 lanes x 2
constexpr int kBPad = 128;           // batch rows are padded to a multiple of this in the tables

inline size_t align256(size_t b) { return (b + 255) / 256 * 256; }
inline int tiles_w(int M) { return (M + kTileW - 1) / kTileW; }
inline int bpad_of(int B) { return (B + kBPad - 1) / kBPad * kBPad; }
// Counters.  Zeroed by rc_range_kernel, which is queued in front of the tables.
struct RowCount {
    unsigned long long marks;      // all ones when the table was not built
    unsigned long long every;      // 1: the every-term kernels run
    unsigned long long run;        // 1: this table's kernel runs
    unsigned long long col_marks;  // marks per weight row (copy)
    unsigned long long fixes;      // outputs to recompute
    unsigned long long sum;        // see add_marks
    unsigned long long idle;       // 1: it does not
};

struct Carve {
    RowCount* count;
    float* wr;        // [T][N]  per tile of weight rows and input: (min, max) of the weights over the rows that keep the input
    float* low;       // [T][Bp]  lower bounds of the K-th largest terms of a batch row (kRowsBound: [T][2][Bp], of the two results)
    uint32_t* bits;   // [T][Bp][table_row_words] the marks
    uint32_t* fix;    // [B * M] outputs of the masked l-inf form whose bound did not hold (recomputed from every input)
    float* wt;        // [T][N][128] the weights of a tile, one 512-byte row per input (dropped weights undefined)
};

size_t carve_sizes(int form, int B, int M, int N, size_t (&sz)[6]) {
    const size_t T = tiles_w(M), Bp = bpad_of(B);
    sz[0] = 256;
    sz[1] = align256(T * 2 * N * 4);
    sz[2] = align256((form == kRowsBound ? 2 : 1) * T * Bp * 4);
    sz[3] = align256(T * Bp * table_row_words(N) * 4);
    sz[4] = form == kRowsMax ? align256((size_t)B * M * 4) : 0;
    sz[5] = align256(T * N * kTileW * 4);
    size_t t = 0;
    for (size_t v : sz) t += v;
    return t;
}

Carve carve(void* ws, int form, int B, int M, int N) {
    size_t sz[6];
    carve_sizes(form, B, M, N, sz);
    char* p = static_cast<char*>(ws);
    Carve c;
    c.count = reinterpret_cast<RowCount*>(p); p += sz[0];
    c.wr = reinterpret_cast<float*>(p); p += sz[1];
    c.low = reinterpret_cast<float*>(p); p += sz[2];
    c.bits = reinterpret_cast<uint32_t*>(p); p += sz[3];
    c.fix = reinterpret_cast<uint32_t*>(p); p += sz[4];
    c.wt = reinterpret_cast<float*>(p);
    return c;
}

// inverted intervals become their midpoint (core/cuda/sort_neuron.cu:262)
__device__ __forceinline__ void repair(float& l, float& u) {
    if (l > u) l = u = (l + u) * 0.5f;
}

// The probe of sort_cols.hip (same constant): the batch rows of a tile differ by more than 2.5 times what 16 entries
// of a weight column do.  stat[0] = widths of the input columns over all batch tiles, stat[1] = widths of the same
// columns over 16 weight rows.
// `ratio` is kProbeRatio for the sort-neuron forms.  The l-inf form asks for more (kProbeRatioMax): its kernel only pays
// below about 25 % of marks, and on inputs spread evenly over their range the marked share is about 1 / (that ratio), so
// its tables are not even built unless the probe promises that few.  Without a probe (null) they are built.
constexpr float kProbeRatio = 2.5f, kProbeRatioMax = 5.f;
__device__ __forceinline__ bool rows_decide(const float* stat, int S, float ratio) {
    return stat == nullptr || stat[0] > ratio * (float)S * stat[1];
}

// ---- tables ----------------------------------------------------------------------------------
// Column ranges of the weights over a tile of 128 weight rows (WMASK: over the rows that keep the input; a column
// that no row keeps, or that holds an undefined or infinite weight, becomes (-inf, +inf): no lower bound, always a
// candidate), and the transposed copy of the tile.  64 inputs x 4 groups of 32 rows per workgroup.
// Under the mask a lane fetches the keep bits of one of the wavefront's rows, 64 inputs wide, and hands them to the others:
// 59 us at 5120 x 5120 (92 with a word fetched per row and lane), held to 64 registers: with the 104 it takes otherwise half the
// wavefronts are in flight, 66 us.
template <bool WMASK>
__global__ void __launch_bounds__(256, WMASK ? 8 : 1) rc_range_kernel(const float* __restrict__ w, const uint32_t* __restrict__ wkeep,
                                                       int M, int N, int S, float* __restrict__ wr, float* __restrict__ wt,
                                                       RowCount* __restrict__ count, const float* __restrict__ stat, float ratio) {
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) count->sum = count->fixes = 0ull;
    if (!rows_decide(stat, S, ratio)) return;
    __shared__ float part[4][3][64];
    const int nl = threadIdx.x & 63, grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = blockIdx.x * 64 + nl, t = blockIdx.y;
    const int r0 = t * kTileW + grp * (kTileW / 4);
    float lo = __builtin_inff(), hi = -__builtin_inff(), odd = 0.f;
    if (n < N) {
        float v[kTileW / 4];
        #pragma unroll
        for (int i = 0; i < kTileW / 4; i++) v[i] = r0 + i < M ? w[(size_t)(r0 + i) * N + n] : 0.f;
        // keep bits of the wavefront's 64 inputs: row i's words in lane i
        uint32_t k0 = ~0u, k1 = ~0u;
        if constexpr (WMASK) {
            const int c0 = blockIdx.x * 2, c1 = c0 + 1 < N / kChunk ? c0 + 1 : c0, row = r0 + (nl & 31) < M ? r0 + (nl & 31) : M - 1;
            k0 = wkeep[(size_t)row * (N / kChunk) + c0];
            k1 = wkeep[(size_t)row * (N / kChunk) + c1];
        }
        #pragma unroll
        for (int i = 0; i < kTileW / 4; i++) {
            bool kept = r0 + i < M;
            if constexpr (WMASK) {
                const uint32_t a = __builtin_amdgcn_readlane(k0, i), b = __builtin_amdgcn_readlane(k1, i);
                kept = kept && __builtin_amdgcn_inverse_ballot_w64((unsigned long long)a | ((unsigned long long)b << 32));
                if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);   // (all rows' bits at once would not fit the scalar registers)
            }
            if (kept) { lo = fminf(lo, v[i]); hi = fmaxf(hi, v[i]); odd += v[i] - v[i]; }
            else if (WMASK) v[i] = __builtin_nanf("");
        }
        float4* dst = reinterpret_cast<float4*>(wt + ((size_t)t * N + n) * kTileW + grp * (kTileW / 4));
        #pragma unroll
        for (int i = 0; i < kTileW / 16; i++) dst[i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
    }
    part[grp][0][nl] = lo; part[grp][1][nl] = hi; part[grp][2][nl] = odd;
    __syncthreads();
    if (grp == 0 && n < N) {
        #pragma unroll
        for (int g = 1; g < 4; g++) { lo = fminf(lo, part[g][0][nl]); hi = fmaxf(hi, part[g][1][nl]); odd += part[g][2][nl]; }
        if (!(odd == 0.f) || lo > hi) { lo = -__builtin_inff(); hi = __builtin_inff(); }
        reinterpret_cast<float2*>(wr)[(size_t)t * N + n] = make_float2(lo, hi);
    }
}

// Bounds and marks (cand_tables.h); J = 0: rows of any length
template <int J, int R, int NT, bool PAIR, bool TWO, bool MASK>
__global__ void __launch_bounds__(64 * (J ? kStreamWaves : kTableWaves))
rc_tables_kernel(TableArgs a, RowCount* __restrict__ c, const unsigned long long* __restrict__ col_count,
                 const float* __restrict__ stat, int S, unsigned long long limit, float ratio) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    unsigned long long marks = ~0ull;
    if (rows_decide(stat, S, ratio)) {
        int part;
        if constexpr (J == 0) part = build_tables<R, NT, PAIR, TWO, MASK>(a, blockIdx.x, blockIdx.y, smem);
        else part = stream_tables<J, R, NT, PAIR, TWO, MASK>(a, blockIdx.x, gridDim.x, blockIdx.y, smem);
        if (!add_marks(&c->sum, part, &marks)) return;
    } else if (blockIdx.x != 0 || blockIdx.y != 0 || threadIdx.x != 0) return;
    const bool run = marks <= limit;   // (the limit is a share of the (tile, row, input) triples: never all ones)
    c->marks = marks;
    c->every = ((col_count == nullptr || col_count[1] != 0ull) && !run) ? 1ull : 0ull;
    c->run = run ? 1ull : 0ull;
    c->idle = run ? 0ull : 1ull;
    c->col_marks = col_count == nullptr ? ~0ull : col_count[0];
}

// ---- main kernel -------------------------------------------------------------------------------
// A wavefront takes one batch row against the tile's 128 weight rows (lane l holds the rows l and l + 64): it lists the
// row's marked inputs in LDS, cuts the list by what a few strong marks say (cand_walk.h) and walks what is left: per mark
// the row's value(s) (scalar operands) and the lane's two weights from the transposed copy (two coalesced 256-byte loads).
// No tile is staged and no barrier is met, so a wavefront with many marks holds nobody up; a workgroup is eight wavefronts
// = eight batch rows, and the workgroups of a tile are dealt to one die, so that the tile's transposed weights (2.6 MB at
// 5120 inputs) stay in that die's cache while its 64 resident workgroups walk them.
// Forms: top-K lists of values (branch-free median insertion, left out where it would change no lane's list), of both
// interval bounds, of values with the input numbers (the reference's ordered insertion: the marks go by in ascending input
// order), the interval bounds of the l-inf distance, and the l-inf distance (the difference of largest magnitude and, optionally, its input; under the factored mask the
// dropped weights of the transposed copy are undefined, the table holds no input the batch row drops, and an output that
// ends below the bound its marks were taken against is listed for rc_fix_kernel).
constexpr int kRtWaves = 8;          // wavefronts of a workgroup

struct RtArgs {
    const float* xl; const float* xu; const float* wt; const float* wr;
    const uint32_t* bits; const float* low;
    RowCount* count;
    uint32_t* fix;
    int B, Bp, M, N;
    float q;
    float* outL; float* outU; int* pos; int* posL;
    const float* shift;   // kRowsSortValues, kRowsSortInterval: see FwdArgs
    float shift_sign;
};

template <int FORM, int K, bool POS, bool MASKED>
__global__ void __launch_bounds__(64 * kRtWaves) rt_main_kernel(RtArgs a) {
    if (a.count->run == 0ull) return;
    constexpr bool IV = FORM == kRowsSortInterval || FORM == kRowsBound;
    constexpr bool LISTS = FORM != kRowsMax && FORM != kRowsBound;
    constexpr bool ORDERED = FORM == kRowsSortPos || (!LISTS && POS);   // the input a term sits at is wanted
    __shared__ uint16_t lists[kRtWaves][kWalkListCap];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int B = a.B, M = a.M, N = a.N, NCH = N / kChunk;
    const int BG = (B + kRtWaves - 1) / kRtWaves;
    // consecutive (tile, batch rows) pairs are dealt out so that the workgroups of a tile share a die and its cache
    int item = blockIdx.x;
    if (gridDim.x % 8 == 0) item = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const int bg = item % BG, t = item / BG;
    const int b = bg * kRtWaves + wave;
    if (b >= B) return;   // wave-uniform
    const float* __restrict__ wcol = a.wt + (size_t)t * N * kTileW + lane;
    uint16_t* list = lists[wave];
    const size_t plane = (size_t)B * M;
    const bool in0 = t * kTileW + lane < M, in1 = t * kTileW + lane + 64 < M;   // the lane's weight rows exist

    // state of the row x the lane's two weight rows: top-K lists (ascending; as bit patterns where only values are wanted), or
    // the difference of largest magnitude
    using Entry = typename std::conditional<FORM == kRowsSortValues || FORM == kRowsSortInterval, int, float>::type;
    Entry hi[2][LISTS ? K : 1], lo[IV ? 2 : 1][IV ? K : 1];
    int idx[ORDERED ? 2 : 1][FORM == kRowsSortPos ? K : 1], idxL[2];
    auto clear = [&]() __attribute__((always_inline)) {
        #pragma unroll
        for (int j = 0; j < 2; j++) {
            if constexpr (LISTS) {
                #pragma unroll
                for (int k = 0; k < K; k++) {
                    hi[j][k] = 0;
                    if constexpr (IV) lo[j][k] = 0;
                    if constexpr (FORM == kRowsSortPos) idx[j][k] = 0;
                }
            } else {
                hi[j][0] = kEps;
                if constexpr (POS) idx[j][0] = 0;
                if constexpr (FORM == kRowsBound) { lo[j][0] = kEps; idxL[j] = (int)kNanId; }
            }
        }
    };
    clear();
    const uint32_t* __restrict__ rowbits = a.bits + ((size_t)t * a.Bp + b) * table_row_words(N);
    const float* __restrict__ xlrow = a.xl + (size_t)b * N;
    const float* __restrict__ xurow = IV ? a.xu + (size_t)b * N : xlrow;
    const float2* __restrict__ ranges = reinterpret_cast<const float2*>(a.wr) + (size_t)t * N;
    float wa[2][4], wb[2][4];
    float least[2] = {0.f, 0.f};   // kRowsSortPos: lower bounds of the K-th largest terms
    auto load = [&](int buf, int i, int n) __attribute__((always_inline)) {
        wa[buf][i] = wcol[(size_t)n * kTileW];
        wb[buf][i] = wcol[(size_t)n * kTileW + 64];
    };
    // VALUES: a strong mark of kRowsSortPos, whose value alone is wanted
    auto term = [&](auto values, int buf, int i, int k, int n, const Own& o) __attribute__((always_inline)) {
        const float xi = lane_value(o.a, k);
        if constexpr (IV) {
            const float ui = lane_value(o.b, k);
            const float a1 = wa[buf][i] - xi, a2 = ui - wa[buf][i];
            const float b1 = wb[buf][i] - xi, b2 = ui - wb[buf][i];
            if constexpr (FORM == kRowsBound) {
                // an undefined operand leaves the other's term; only a strictly better term replaces a bound, so with
                // positions the first of equal terms keeps it
                const float L0 = -fminf(a1, a2), U0 = fmaxf(a1, a2), L1 = -fminf(b1, b2), U1 = fmaxf(b1, b2);
                if constexpr (POS) {
                    const int p0 = a1 <= a2 ? n : n | (int)kSign, p1 = b1 <= b2 ? n : n | (int)kSign;
                    const bool l0 = L0 > lo[0][0], l1 = L1 > lo[1][0], u0 = U0 > hi[0][0], u1 = U1 > hi[1][0];
                    lo[0][0] = l0 ? L0 : lo[0][0]; idxL[0] = l0 ? p0 : idxL[0];
                    lo[1][0] = l1 ? L1 : lo[1][0]; idxL[1] = l1 ? p1 : idxL[1];
                    hi[0][0] = u0 ? U0 : hi[0][0]; idx[0][0] = u0 ? p0 : idx[0][0];
                    hi[1][0] = u1 ? U1 : hi[1][0]; idx[1][0] = u1 ? p1 : idx[1][0];
                } else {
                    lo[0][0] = fmaxf(lo[0][0], L0); lo[1][0] = fmaxf(lo[1][0], L1);
                    hi[0][0] = fmaxf(hi[0][0], U0); hi[1][0] = fmaxf(hi[1][0], U1);
                }
                return;
            } else {
            // (the maximum with -1 turns a term that is undefined altogether into a negative one, which the lists ignore)
            insert_pair<K>(lo[0], fmaxf(fmaxf(-a1, -a2), -1.f), lo[1], fmaxf(fmaxf(-b1, -b2), -1.f));
            insert_pair<K>(hi[0], fmaxf(fmaxf(a1, a2), -1.f), hi[1], fmaxf(fmaxf(b1, b2), -1.f));
            }
        } else {
            const float d0 = xi - wa[buf][i], d1 = xi - wb[buf][i];
            if constexpr (FORM == kRowsSortValues) {
                insert_pair<K>(hi[0], fmaxf(fabsf(d0), -1.f), hi[1], fmaxf(fabsf(d1), -1.f));
            } else if constexpr (decltype(values)::value) {
                topk_insert_values<K>(hi[0], fabsf(d0));
                topk_insert_values<K>(hi[1], fabsf(d1));
            } else if constexpr (FORM == kRowsSortPos) {
                // the marks of a row go by in ascending input order: the ordered insertion of the scan
                // over all inputs (core/cuda/sort_neuron.cu:108-113, 176-185), ties included
                if (fabsf(d0) > hi[0][0] && fabsf(d0) >= least[0]) topk_insert<K>(hi[0], idx[0], fabsf(d0), n | (d0 >= 0.f ? 0 : (int)kSign));
                if (fabsf(d1) > hi[1][0] && fabsf(d1) >= least[1]) topk_insert<K>(hi[1], idx[1], fabsf(d1), n | (d1 >= 0.f ? 0 : (int)kSign));
            } else {
                // running maximum; only a larger term replaces it, so the first of equal terms keeps the
                // position (core/cuda/inf_dist_cuda.cu:176-190); an undefined term (a weight the row of
                // the mask drops) never compares greater
                // (the difference itself is kept: its magnitude is the maximum, its sign the flag of
                // the position)
                const bool g0 = fabsf(d0) > fabsf(hi[0][0]), g1 = fabsf(d1) > fabsf(hi[1][0]);
                hi[0][0] = g0 ? d0 : hi[0][0];
                hi[1][0] = g1 ? d1 : hi[1][0];
                if constexpr (POS) {
                    idx[0][0] = g0 ? n : idx[0][0];
                    idx[1][0] = g1 ? n : idx[1][0];
                }
            }
        }
    };
    auto value = [&](int buf, int i, int k, int n, const Own& o) __attribute__((always_inline)) { term(std::bool_constant<FORM == kRowsSortPos>{}, buf, i, k, n, o); };
    auto use = [&](int buf, int i, int k, int n, const Own& o) __attribute__((always_inline)) { term(std::false_type{}, buf, i, k, n, o); };
    // smallest results of the lane's rows over the wavefront (weight rows past the last one do not count)
    float thU = 0.f, thL = 0.f;
    // (never below what it was: an ordered walk forgets the strong marks' results, but they are terms of these rows)
    auto smallest = [&](float was, float v0, float v1) __attribute__((always_inline)) {
        return fmaxf(was, wave_min_nonneg(fminf(in0 ? v0 : __builtin_inff(), in1 ? v1 : __builtin_inff())));
    };
    // In kRowsSortPos the strong marks give each row a lower bound of its K-th largest term.  A term below it is never among
    // the K largest, and whether one at or above it enters depends only on entries at least that large, so the walk in input
    // order may leave the others out.
    for_marks(list, NCH, lane, [&](int c) __attribute__((always_inline)) { return rowbits[c]; },
              [&](int total, bool first) __attribute__((always_inline)) {
        walk_marks<ORDERED, IV, 128, LISTS && !ORDERED ? walk_short(K) : 0>(list, total, first, lane,
            [&](int n) __attribute__((always_inline)) {
                Own o{xlrow[n], 0.f};
                if constexpr (IV) { o.b = xurow[n]; repair(o.a, o.b); }
                return o;
            },
            [&](int n, const Own& o) __attribute__((always_inline)) {
                const float2 r = ranges[n];
                return fmaxf(r.y - o.a, (IV ? o.b : o.a) - r.x);
            },
            load, value, use,
            [&](bool strong) __attribute__((always_inline)) {
                if (FORM == kRowsSortPos && strong) { least[0] = hi[0][0]; least[1] = hi[1][0]; }
                if constexpr (FORM == kRowsSortValues || FORM == kRowsSortInterval) thU = smallest(thU, __int_as_float(hi[0][0]), __int_as_float(hi[1][0]));
                else thU = smallest(thU, fmaxf(fabsf(hi[0][0]), least[0]), fmaxf(fabsf(hi[1][0]), least[1]));
                if constexpr (FORM == kRowsSortInterval) thL = smallest(thL, __int_as_float(lo[0][0]), __int_as_float(lo[1][0]));
                else if constexpr (IV) thL = smallest(thL, lo[0][0], lo[1][0]);
            },
            [&](int n, const Own& o) __attribute__((always_inline)) {
                const float2 r = ranges[n];
                bool keep = !(fmaxf(r.y - o.a, (IV ? o.b : o.a) - r.x) < thU);
                if constexpr (IV) keep = keep || !(fmaxf(o.a - r.x, r.y - o.b) < thL);
                return keep;
            },
            clear);
    });
    #pragma unroll
    for (int j = 0; j < 2; j++) {
        const int col = t * kTileW + lane + 64 * j;
        if (col < M) {
            const size_t o = (size_t)b * M + col;
            if constexpr (LISTS) {
                if constexpr (FORM == kRowsSortPos) a.outU[o] = geo_sum<K>(hi[j], a.q);
                else {
                    const float add = output_shift(a.shift, a.shift_sign, col);
                    a.outU[o] = geo_sum_bits<K>(hi[j], a.q) + add;
                    if constexpr (IV) a.outL[o] = geo_sum_bits<K>(lo[j], a.q) + add;
                }
                if constexpr (FORM == kRowsSortPos) {
                    #pragma unroll
                    for (int k = 0; k < K; k++) a.pos[(size_t)(K - 1 - k) * plane + o] = idx[j][k];   // plane 0 = largest
                }
            } else {
                a.outU[o] = fabsf(hi[j][0]);
                if constexpr (FORM == kRowsBound) {
                    a.outL[o] = lo[j][0];
                    if constexpr (POS) { a.pos[o] = idx[j][0]; a.posL[o] = idxL[j]; }
                } else if constexpr (POS) a.pos[o] = idx[j][0] | (hi[j][0] >= 0.f ? 0 : (int)kSign);
                if constexpr (MASKED) {
                    // The bound rests on K inputs that the batch row keeps; a weight row that keeps none of them
                    // may have its maximum at an unmarked input: such an output is recomputed from every input.
                    if (!(fabsf(hi[j][0]) >= a.low[(size_t)t * a.Bp + b])) a.fix[atomicAdd(&a.count->fixes, 1ull)] = (uint32_t)o;
                }
            }
        }
    }
}

struct FixArgs {
    const float* xl; const float* w;
    const uint32_t* xkeep; const uint32_t* wkeep;
    const RowCount* count;
    const uint32_t* fix;
    int M, N;
    float* outU; int* pos;
};

// Outputs of the masked l-inf form whose maximum stayed below the bound their marks were taken against: one
// wavefront per output over every input that both rows keep, lowest input first among equal terms.
template <bool POS>
__global__ void __launch_bounds__(256) rc_fix_kernel(FixArgs a) {
    if (a.count->run == 0ull) return;
    const unsigned long long total = a.count->fixes;
    const int lane = threadIdx.x & 63;
    const int N = a.N, NCH = N / kChunk;
    for (unsigned long long e = (unsigned long long)blockIdx.x * 4 + (threadIdx.x >> 6); e < total; e += (unsigned long long)gridDim.x * 4) {
        const uint32_t o = a.fix[e];
        const int b = (int)(o / (uint32_t)a.M), m = (int)(o % (uint32_t)a.M);
        const float* xr = a.xl + (size_t)b * N;
        const float* wrow = a.w + (size_t)m * N;
        float best = kEps;
        int where = 0;
        for (int n = lane; n < N; n += 64) {
            const uint32_t keep = a.xkeep[(size_t)b * NCH + (n >> 5)] & a.wkeep[(size_t)m * NCH + (n >> 5)];
            const float d = xr[n] - wrow[n];
            if (((keep >> (n & 31)) & 1u) && fabsf(d) > best) { best = fabsf(d); where = n | (d >= 0.f ? 0 : (int)kSign); }
        }
        #pragma unroll
        for (int s = 32; s; s >>= 1) {
            const float ob = __shfl_xor(best, s);
            const int ow = __shfl_xor(where, s);
            // a lane that found nothing keeps (1e-10, 0) and loses to any term; equal terms: the lower input
            const bool take = ob > best || (ob == best && ob > kEps && (ow & 0x7fffffff) < (where & 0x7fffffff));
            best = take ? ob : best;
            where = take ? ow : where;
        }
        if (lane == 0) {
            a.outU[o] = best;
            if constexpr (POS) a.pos[o] = where;
        }
    }
}

template <int FORM, int K, bool POS, bool MASKED>
int launch_rt(const RtArgs& a, hipStream_t st) {
    const int T = tiles_w(a.M), BG = (a.B + kRtWaves - 1) / kRtWaves;
    hipLaunchKernelGGL((rt_main_kernel<FORM, K, POS, MASKED>), dim3((unsigned)(T * BG)), dim3(64 * kRtWaves), 0, st, a);
    return check_launch("rt_main_kernel");
}

// ranges, transposed weights, tables
template <bool PAIR, bool TWO, bool MASK>
int run_tables(const float* xl, const float* xu, const float* w, const uint32_t* xkeep, const uint32_t* wkeep, int B, int M,
               int N, int K, const Carve& c, unsigned long long limit, const float* col_stat, const unsigned long long* col_count,
               float ratio, hipStream_t st) {
    const int T = tiles_w(M), S = (B + 127) / 128;
    int rc;
    hipLaunchKernelGGL((rc_range_kernel<MASK>), dim3((N + 63) / 64, T), dim3(256), 0, st, w, wkeep, M, N, S, c.wr, c.wt, c.count, col_stat, ratio);
    if ((rc = check_launch("rc_range_kernel"))) return rc;
    const TableArgs t{PAIR ? xu : xl, xl, xkeep, c.wr, B, bpad_of(B), N, T, K, c.low, c.bits};
    auto tables = [&](auto j, auto rows, auto nt) {
        constexpr int J = decltype(j)::value, R = decltype(rows)::value, NT = decltype(nt)::value;
        const int groups = (T + NT - 1) / NT;
        dim3 grid((B + R * kTableWaves - 1) / (R * kTableWaves), groups), block(64 * kTableWaves);
        size_t lds = (size_t)NT * 2 * kTableSlice * 4;
        if (J) {
            const StreamShape s = stream_shape(N, R, B, groups);
            grid.x = s.rows;
            block.x = 64 * s.waves;
            lds = stream_lds(s.waves, R * NT * (TWO ? 2 : 1));
        }
        hipLaunchKernelGGL((rc_tables_kernel<J, R, NT, PAIR, TWO, MASK>), grid, block, lds, st, t, c.count, col_count, col_stat, S, limit, ratio);
        return check_launch("rc_tables_kernel");
    };
    using std::integral_constant;
    constexpr integral_constant<int, 4> four{};
    constexpr integral_constant<int, 2> two{};
    constexpr integral_constant<int, 1> one{};
    // four tiles of weight rows at a time, two where the registers hold no more ranges
    switch (stream_blocks(N)) {
        case 1: return tables(one, two, four);
        case 2: return tables(two, integral_constant<int, PAIR ? 1 : 2>{}, integral_constant<int, MASK ? 3 : 4>{});
        case 3: return tables(integral_constant<int, 3>{}, one, two);
    }
    return tables(integral_constant<int, 0>{}, one, four);
}

template <int FORM, int K>
int run(const float* xl, const float* xu, const float* w, int B, int M, int N, float q, float* outL, float* outU, int* pos,
        const Carve& c, unsigned long long limit, const float* col_stat, const unsigned long long* col_count, const float* shift,
        float shift_sign, hipStream_t st) {
    constexpr bool IV = FORM == kRowsSortInterval;
    const int rc = run_tables<IV, false, false>(xl, xu, w, nullptr, nullptr, B, M, N, K, c, limit, col_stat, col_count, kProbeRatio, st);
    if (rc) return rc;
    RtArgs a{xl, xu, c.wt, c.wr, c.bits, c.low, c.count, c.fix, B, bpad_of(B), M, N, q, outL, outU, pos, nullptr, shift, shift_sign};
    return launch_rt<FORM, K, false, false>(a, st);
}

template <bool MASKED>
int run_max(const float* x, const float* w, const uint32_t* xkeep, const uint32_t* wkeep, int B, int M, int N, int K, float* y,
            int* pos, const Carve& c, unsigned long long limit, const float* col_stat, const unsigned long long* col_count,
            float ratio, hipStream_t st) {
    int rc = run_tables<false, false, MASKED>(x, nullptr, w, xkeep, wkeep, B, M, N, K, c, limit, col_stat, col_count, ratio, st);
    if (rc) return rc;
    RtArgs a{x, nullptr, c.wt, c.wr, c.bits, c.low, c.count, c.fix, B, bpad_of(B), M, N, 0.f, nullptr, y, pos, nullptr, nullptr, 0.f};
    if (pos) rc = launch_rt<kRowsMax, 1, true, MASKED>(a, st);
    else rc = launch_rt<kRowsMax, 1, false, MASKED>(a, st);
    if (rc || !MASKED) return rc;
    const FixArgs f{x, w, xkeep, wkeep, c.count, c.fix, M, N, y, pos};
    if (pos) hipLaunchKernelGGL((rc_fix_kernel<true>), dim3(256), dim3(256), 0, st, f);
    else hipLaunchKernelGGL((rc_fix_kernel<false>), dim3(256), dim3(256), 0, st, f);
    return check_launch("rc_fix_kernel");
}

int run_bound(const float* xl, const float* xu, const float* w, int B, int M, int N, float* outL, float* outU, int* posL, int* posU,
              const Carve& c, unsigned long long limit, const float* col_stat, const unsigned long long* col_count, hipStream_t st) {
    const int rc = run_tables<true, true, false>(xl, xu, w, nullptr, nullptr, B, M, N, 1, c, limit, col_stat, col_count, kProbeRatio, st);
    if (rc) return rc;
    RtArgs a{xl, xu, c.wt, c.wr, c.bits, c.low, c.count, c.fix, B, bpad_of(B), M, N, 0.f, outL, outU, posU, posL, nullptr, 0.f};
    return posU ? launch_rt<kRowsBound, 1, true, false>(a, st) : launch_rt<kRowsBound, 1, false, false>(a, st);
}

}  // namespace

size_t row_cands_workspace(int form, int B, int CO, int CI) {
    size_t sz[6];
    return carve_sizes(form, B, CO, CI, sz);
}

bool row_cands_supported(int form, int K) {
    switch (form) {
        case kRowsSortValues: return K >= 2 && K <= 25;
        case kRowsSortInterval: return K >= 2 && K <= 25;
        case kRowsSortPos: return K >= 2 && K <= 25;
        case kRowsBound: return K == 1;
        case kRowsMax: return K == 1 || K == 8 || K == 12 || K == 16 || K == 20 || K == 24;
    }
    return false;
}

#define SD_ROWS_K12(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)
#define SD_ROWS_K18(X) SD_ROWS_K12(X) X(13) X(14) X(15) X(16) X(17) X(18)
#define SD_ROWS_K25(X) SD_ROWS_K18(X) X(19) X(20) X(21) X(22) X(23) X(24) X(25)

const unsigned long long* row_cands_idle(const unsigned long long* every) {
    return every + (offsetof(RowCount, idle) - offsetof(RowCount, every)) / sizeof(unsigned long long);
}

int row_cands_forward(int form, const float* xl, const float* xu, const float* w, const uint32_t* xkeep,
                      const uint32_t* wkeep, int B, int CO, int CI, float q, int K, float* outL, float* outU, int* pos,
                      void* ws, float density, bool forced, const float* col_stat, const unsigned long long* col_count,
                      const unsigned long long** every, hipStream_t st, int* pos_lower, const float* shift, float shift_sign) {
    const float ratio_max = forced ? kProbeRatio : kProbeRatioMax;
    if (CI % kChunk != 0 || B < 1 || CO < 1 || !row_cands_supported(form, K) || (xkeep == nullptr) != (wkeep == nullptr) ||
        (long long)B * CO >= (1ll << 32)) {
        set_error("row_cands_forward: shape or form not supported");
        return SD_ERR_ARG;
    }
    if (CI > 65536) {   // (16-bit input numbers in the lists of marks)
        set_error("row_cands_forward: rows of more than 65536 inputs");
        return SD_ERR_ARG;
    }
    const Carve c = carve(ws, form, B, CO, CI);
    const float d = density < 0.f ? 0.f : density > 1.f ? 1.f : density;
    const unsigned long long limit = (unsigned long long)((double)tiles_w(CO) * B * CI * d);
    *every = &c.count->every;
    switch (form) {
        case kRowsSortValues:
            switch (K) {
#define X(k) case k: return run<kRowsSortValues, k>(xl, nullptr, w, B, CO, CI, q, outL, outU, nullptr, c, limit, col_stat, col_count, shift, shift_sign, st);
                SD_ROWS_K25(X)
#undef X
            }
            break;
        case kRowsSortInterval:
            switch (K) {
#define X(k) case k: return run<kRowsSortInterval, k>(xl, xu, w, B, CO, CI, q, outL, outU, nullptr, c, limit, col_stat, col_count, shift, shift_sign, st);
                SD_ROWS_K25(X)
#undef X
            }
            break;
        case kRowsSortPos:
            switch (K) {
#define X(k) case k: return run<kRowsSortPos, k>(xl, nullptr, w, B, CO, CI, q, outL, outU, pos, c, limit, col_stat, col_count, shift, shift_sign, st);
                SD_ROWS_K25(X)
#undef X
            }
            break;
        case kRowsBound:
            return run_bound(xl, xu, w, B, CO, CI, outL, outU, pos_lower, pos, c, limit, col_stat, col_count, st);
        case kRowsMax:
            return xkeep ? run_max<true>(xl, w, xkeep, wkeep, B, CO, CI, K, outU, pos, c, limit, col_stat, col_count, ratio_max, st)
                         : run_max<false>(xl, w, nullptr, nullptr, B, CO, CI, K, outU, pos, c, limit, col_stat, col_count, ratio_max, st);
    }
    set_error("row_cands_forward: K=%d not supported for form %d", K, form);
    return SD_ERR_ARG;
}

}  // namespace sd
