// Sort neuron and its interval bounds from per-weight-row candidate tables (see sort_cols.h).
#include "sort_cols.h"
#include <type_traits>
#include <utility>
#include "cand_tables.h"
#include "cand_walk.h"
#include "fwd_tile.h"

namespace sd {

namespace {

constexpr int kChunk = kSortColsChunk;
constexpr int kTileB = 128;          // batch rows of a tile: 64 lanes x 2
constexpr int kRowPad = 128;         // weight rows are padded to a multiple of this in the tables
constexpr int kMainWaves = 4;        // wavefronts of a workgroup of the main kernels
constexpr int kMainTile = kMainWaves;   // weight rows of a workgroup, one per wavefront
constexpr int kSample = 640;         // see walk_marks

inline size_t align256(size_t b) { return (b + 255) / 256 * 256; }
inline int tiles_b(int B) { return (B + kTileB - 1) / kTileB; }
inline int mpad_of(int M) { return (M + kRowPad - 1) / kRowPad * kRowPad; }
struct Carve {
    TableCount* count;
    float* xr;        // [S][N] per batch tile and input: (min, max) over the tile's rows, of the hull of l and u in the interval form; K = 1 there: (min l, max l, min u, max u)
    float* xT;        // [N][Bp] the inputs transposed ((l, u) pairs in the interval form), intervals repaired
    float* low;       // [S][2][Mp] lower bounds of the K-th largest terms of a weight row (K = 1 in the interval form: for either bound)
    uint32_t* bits;   // [S][Mp][table_row_words] the marks
    float2* widths;   // [S][N / 32] what the probe adds up, see sc_range_kernel
};

size_t carve_sizes(int B, int M, int N, size_t (&sz)[6]) {
    const size_t S = tiles_b(B), Bp = S * kTileB, Mp = mpad_of(M);
    sz[0] = 256;
    sz[1] = align256(S * N * 16);
    sz[2] = align256((size_t)N * Bp * 8);
    sz[3] = align256(S * 2 * Mp * 4);
    sz[4] = align256(S * Mp * table_row_words(N) * 4);
    sz[5] = align256(S * (N / kChunk) * 8);
    size_t t = 0;
    for (size_t v : sz) t += v;
    return t;
}

Carve carve(void* ws, int B, int M, int N) {
    size_t sz[6];
    carve_sizes(B, M, N, sz);
    char* p = static_cast<char*>(ws);
    Carve c;
    c.count = reinterpret_cast<TableCount*>(p); p += sz[0];
    c.xr = reinterpret_cast<float*>(p); p += sz[1];
    c.xT = reinterpret_cast<float*>(p); p += sz[2];
    c.low = reinterpret_cast<float*>(p); p += sz[3];
    c.bits = reinterpret_cast<uint32_t*>(p); p += sz[4];
    c.widths = reinterpret_cast<float2*>(p);
    return c;
}

// inverted intervals become their midpoint (core/cuda/sort_neuron.cu:262)
__device__ __forceinline__ void repair(float& l, float& u) {
    if (l > u) l = u = (l + u) * 0.5f;
}

// ---- tables ----------------------------------------------------------------------------------
// Column ranges of a tile of 128 batch rows, and the transposed copy of the tile the main kernel reads (one row of 128
// values per input).  Value form: l = u = x.  A workgroup takes 32 inputs, a work-item 16 of the rows at one of them, all
// its loads in flight.
// Also answers whether the table is worth building: it can only prune when the rows of a batch tile are alike
// compared with the entries of a weight row.  A workgroup leaves the widths of its columns' ranges and, in tile 0, the
// ranges of the same columns over the first 16 weight rows; sc_tables_kernel adds them up (the launch that cleared a sum for
// atomics took 4.7 us, adding up 640 pairs 1).
// MASKED (value form only): xkeep holds one word per (batch row, 32 inputs); an input a row does not keep takes no
// part in the ranges and is undefined in the transposed copy, so that its term never wins a comparison.  A column no
// row of the tile keeps has neither a lower bound nor a candidate.
// TWO: the ranges of l and of u apart.  BOX: intervals with the inputs x beside them, one range over all three; xT2: x transposed.
// SPARE: see sc_tables_kernel (the test alone is 0.3 of 5.6 us).
template <bool IV, bool TWO, bool MASKED, bool BOX = false, bool SPARE = false>
__global__ void __launch_bounds__(256) sc_range_kernel(const float* __restrict__ xl, const float* __restrict__ xu,
                                                       const float* __restrict__ w, const uint32_t* __restrict__ xkeep,
                                                       int B, int M, int N, int Bp, float* __restrict__ xr,
                                                       float* __restrict__ xT, float2* __restrict__ widths,
                                                       TableCount* __restrict__ count, const unsigned long long* __restrict__ unless,
                                                       const float* __restrict__ x, float* __restrict__ xT2) {
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) count->sum = 0ull;
    if (SPARE && unless[1] == 0ull) return;
    static_assert(!BOX || (IV && !TWO), "");
    static_assert(!(IV && MASKED) && (IV || !TWO), "the factored mask belongs to the value form, two ranges to the interval form");
    constexpr int kCols = kChunk, kGroups = 256 / kCols, kRows = kTileB / kGroups;
    __shared__ float part[kGroups][5][kCols];
    __shared__ float wpart[kGroups][2][kCols];
    __shared__ float tl[kCols][kTileB + 1];
    __shared__ float tu[IV ? kCols : 1][kTileB + 1];
    __shared__ float tx[BOX ? kCols : 1][kTileB + 1];
    const int tid = threadIdx.x, nl = tid % kCols, grp = tid / kCols;
    const int n0 = blockIdx.x * kCols, n = n0 + nl, s = blockIdx.y;   // (N is a multiple of 32)
    float l[kRows], u[IV ? kRows : 1], v[BOX ? kRows : 1];
    uint32_t kept = ~0u;
    #pragma unroll
    for (int r = 0; r < kRows; r++) {
        const int row = s * kTileB + grp * kRows + r, rr = row < B ? row : B - 1;
        l[r] = xl[(size_t)rr * N + n];
        if constexpr (IV) u[r] = xu[(size_t)rr * N + n];
        if constexpr (BOX) v[r] = x[(size_t)rr * N + n];
        if constexpr (MASKED) { if (!((xkeep[(size_t)rr * (N / kChunk) + blockIdx.x] >> nl) & 1u)) kept &= ~(1u << r); }
    }
    // the probe: ranges of the same columns over the first 16 weight rows (tile 0 only)
    float wlo = __builtin_inff(), whi = -__builtin_inff();
    if (s == 0) {
        #pragma unroll
        for (int k = 0; k < 16 / kGroups; k++) {
            const int m = grp * (16 / kGroups) + k;
            if (m < M) { const float v = w[(size_t)m * N + n]; wlo = fminf(wlo, v); whi = fmaxf(whi, v); }
        }
    }
    float lmin = __builtin_inff(), lmax = -__builtin_inff(), umin = __builtin_inff(), umax = -__builtin_inff();
    float odd = 0.f;   // stays 0 while every value of the column is finite
    #pragma unroll
    for (int r = 0; r < kRows; r++) {
        const int col = grp * kRows + r;
        float a = l[r], b = IV ? u[IV ? r : 0] : a, m = BOX ? v[BOX ? r : 0] : a;
        if (s * kTileB + col >= B) a = b = m = 0.f;
        else if ((kept >> r) & 1u) {
            odd += (a - a) + (b - b);
            if (IV) repair(a, b);
            lmin = fminf(lmin, a); lmax = fmaxf(lmax, a);
            umin = fminf(umin, b); umax = fmaxf(umax, b);
            if (BOX) { odd += m - m; lmin = fminf(lmin, m); umax = fmaxf(umax, m); }
        } else a = b = __builtin_nanf("");
        tl[nl][col] = a;
        if (IV) tu[nl][col] = b;
        if (BOX) tx[nl][col] = m;
    }
    part[grp][0][nl] = lmin; part[grp][1][nl] = lmax; part[grp][2][nl] = umin; part[grp][3][nl] = umax;
    part[grp][4][nl] = odd;
    wpart[grp][0][nl] = wlo; wpart[grp][1][nl] = whi;
    __syncthreads();
    if (grp == 0) {
        float ww = 0.f;
        #pragma unroll
        for (int g = 1; g < kGroups; g++) {
            lmin = fminf(lmin, part[g][0][nl]); lmax = fmaxf(lmax, part[g][1][nl]);
            umin = fminf(umin, part[g][2][nl]); umax = fmaxf(umax, part[g][3][nl]);
            wlo = fminf(wlo, wpart[g][0][nl]); whi = fmaxf(whi, wpart[g][1][nl]);
            odd += part[g][4][nl];
        }
        // A row whose value is undefined or infinite at this input drops terms the other rows keep, so nothing
        // may be concluded from the column: its range becomes everything (no lower bound, always a candidate).
        if (!(odd == 0.f)) { lmin = umin = -__builtin_inff(); lmax = umax = __builtin_inff(); }
        const bool empty = lmin > lmax;   // no row of the tile keeps this input
        float bw = empty ? 0.f : fmaxf(lmax - lmin, umax - umin);
        // empty: w - max l = -inf and min u - w = -inf (no lower bound); w - min l = -inf and max u - w = -inf (no candidate)
        if (TWO) reinterpret_cast<float4*>(xr)[(size_t)s * N + n] = make_float4(lmin, lmax, umin, umax);
        else if (empty) reinterpret_cast<float2*>(xr)[(size_t)s * N + n] = make_float2(__builtin_nanf(""), __builtin_nanf(""));
        else reinterpret_cast<float2*>(xr)[(size_t)s * N + n] = make_float2(lmin, umax);
        if (s == 0) ww = whi - wlo;
        if (!(bw < 3.0e38f)) bw = 3.0e38f;   // infinite or undefined widths count as very wide
        #pragma unroll
        for (int o = kCols / 2; o; o >>= 1) { bw += __shfl_xor(bw, o); ww += __shfl_xor(ww, o); }
        if (nl == 0) widths[(size_t)s * gridDim.x + blockIdx.x] = make_float2(bw, ww);
    }
    for (int e = tid; e < kCols * kTileB; e += 256) {
        const int nn = e >> 7, col = e & (kTileB - 1);
        const size_t o = (size_t)(n0 + nn) * Bp + s * kTileB + col;
        if (IV) reinterpret_cast<float2*>(xT)[o] = make_float2(tl[nn][col], tu[nn][col]);
        else xT[o] = tl[nn][col];
        if (BOX) xT2[o] = tx[nn][col];
    }
}

// The batch rows of a tile differ by more than kProbeRatio times what 16 entries of a weight column do (images
// against small weights): the table would mark nearly every input, so it is not built and reported as full.
// stat[0]: widths of the column ranges over all tiles and columns, stat[1]: those of the weights.  Every workgroup adds them
// up for itself, in the same order; the first leaves them for the tables per batch row.
constexpr float kProbeRatio = 2.5f;
__device__ __forceinline__ bool table_pointless(const float2* __restrict__ widths, int n, int S, float* __restrict__ stat) {
    __shared__ float2 part[kStreamWaves];
    float bw = 0.f, ww = 0.f;
    for (int i = threadIdx.x; i < n; i += (int)blockDim.x) { const float2 v = widths[i]; bw += v.x; ww += v.y; }
    #pragma unroll
    for (int o = 32; o; o >>= 1) { bw += __shfl_xor(bw, o); ww += __shfl_xor(ww, o); }
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = make_float2(bw, ww);
    __syncthreads();
    bw = ww = 0.f;
    for (int i = 0; i < (int)(blockDim.x >> 6); i++) { bw += part[i].x; ww += part[i].y; }
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) { stat[0] = bw; stat[1] = ww; }
    // (wave-uniform: a scalar comparison, so that no lane mask is held)
    return __builtin_amdgcn_readfirstlane(bw > kProbeRatio * (float)S * ww ? 1 : 0) != 0;
}

// Bounds and marks (cand_tables.h); J = 0: rows of any length.  SPARE: tables that may not be needed, see `unless` (a form of its own: the
// test alone took the others from 28.2 to 29.3 us at 128 x 5120 x 5120)
template <int J, int R, int NT, bool TWO, bool MASK, bool SPARE>
__global__ void __launch_bounds__(64 * (J ? kStreamWaves : kTableWaves))
sc_tables_kernel(TableArgs a, const float2* __restrict__ widths, TableCount* __restrict__ c, unsigned long long limit,
                 const unsigned long long* __restrict__ unless) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    if (SPARE && unless[1] == 0ull) {   // not needed: no kernel of this table, none that forms every term, and none of the other orientation
        if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) { c->marks = ~0ull; c->above = 0ull; c->stat[0] = c->stat[1] = 0.f; }
        return;
    }
    if (table_pointless(widths, a.tiles * (a.N / kChunk), a.tiles, c->stat)) {
        if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) { c->marks = ~0ull; c->above = 1ull; }
        return;
    }
    int marks;
    if constexpr (J == 0) marks = build_tables<R, NT, false, TWO, MASK>(a, blockIdx.x, blockIdx.y, smem);
    else marks = stream_tables<J, R, NT, false, TWO, MASK>(a, blockIdx.x, gridDim.x, blockIdx.y, smem);
    unsigned long long total;
    if (add_marks(&c->sum, marks, &total)) { c->marks = total; c->above = total > limit ? 1ull : 0ull; }
}

template <int J, int R, int NT, bool TWO, bool MASK>
int launch_tables(const TableArgs& t, const Carve& c, unsigned long long limit, const unsigned long long* unless, hipStream_t st) {
    const int groups = (t.tiles + NT - 1) / NT;
    dim3 grid((t.R + R * kTableWaves - 1) / (R * kTableWaves), groups), block(64 * kTableWaves);
    size_t lds = (size_t)NT * (TWO ? 4 : 2) * kTableSlice * 4;
    if (J) {
        const StreamShape s = stream_shape(t.N, R, t.R, groups);
        grid.x = s.rows;
        block.x = 64 * s.waves;
        lds = stream_lds(s.waves, R * NT * (TWO ? 2 : 1));
    }
    if (!MASK && unless != nullptr) hipLaunchKernelGGL((sc_tables_kernel<J, R, NT, TWO, MASK, !MASK>), grid, block, lds, st, t, c.widths, c.count, limit, unless);
    else hipLaunchKernelGGL((sc_tables_kernel<J, R, NT, TWO, MASK, false>), grid, block, lds, st, t, c.widths, c.count, limit, nullptr);
    return check_launch("sc_tables_kernel");
}
// As many batch tiles at a time as there are, up to four, and as the registers hold ranges of (64 per lane).
template <bool TWO, bool MASK>
int run_tables(const float* w, const uint32_t* wkeep, int S, int M, int Mp, int N, int K, const Carve& c,
               unsigned long long limit, const unsigned long long* unless, hipStream_t st) {
    const TableArgs t{w, w, wkeep, c.xr, M, Mp, N, S, K, c.low, c.bits};
    switch (stream_blocks(N)) {
        case 1:
            if (S == 1) return launch_tables<1, 4, 1, TWO, MASK>(t, c, limit, unless, st);
            if (S == 2) return launch_tables<1, 2, 2, TWO, MASK>(t, c, limit, unless, st);
            return launch_tables<1, 2, 4, TWO, MASK>(t, c, limit, unless, st);
        case 2:
            if (S == 1) return launch_tables<2, 2, 1, TWO, MASK>(t, c, limit, unless, st);
            if (TWO || S == 2) return launch_tables<2, TWO ? 1 : 2, 2, TWO, MASK>(t, c, limit, unless, st);
            return launch_tables<2, MASK ? 1 : 2, TWO ? 2 : 4, TWO, MASK>(t, c, limit, unless, st);
        case 3:
            if (TWO || S == 1) return launch_tables<3, 2, 1, TWO, MASK>(t, c, limit, unless, st);
            return launch_tables<3, 1, TWO ? 1 : 2, TWO, MASK>(t, c, limit, unless, st);
    }
    return launch_tables<0, 1, 4, TWO, MASK>(t, c, limit, unless, st);
}

// ---- main kernels ------------------------------------------------------------------------------
// A workgroup takes four weight rows (kMainTile) and one batch tile; each of its wavefronts one of the rows, with lane l holding the
// batch rows l and l + 64 of the tile.  For its row the wavefront lists the marked inputs in LDS, cuts the list by what a
// few strong marks say (cand_walk.h) and walks what is left: per mark one weight (a scalar operand), one transposed row of
// inputs (two coalesced loads) and the terms.  The results of the workgroup leave through LDS, 16 bytes wide.
// Workgroups go to the chip's eight dies in turn, each with a cache of its own: consecutive (tile, rows) pairs are dealt out
// so that a die sees few batch tiles, whose transposed inputs it re-reads.
__device__ __forceinline__ int main_item() {
    return gridDim.x % 8 == 0 ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3) : blockIdx.x;
}

// Largest a term of one weight row can be over the rows of a batch tile: the value (or the upper bound), the lower bound.
// Without ranges of l and u apart the first stands for both (it is the larger).
template <bool TWO>
struct Caps {
    const float* __restrict__ ranges;   // of the tile's inputs
    __device__ __forceinline__ float2 operator()(int n, float w) const {
        if constexpr (TWO) {
            const float4 r = reinterpret_cast<const float4*>(ranges)[n];
            return make_float2(fmaxf(w - r.x, r.w - w), fmaxf(r.y - w, w - r.z));
        } else {
            const float2 r = reinterpret_cast<const float2*>(ranges)[n];
            const float c = fmaxf(w - r.x, r.y - w);
            return make_float2(c, c);
        }
    }
};

// Sums over the K largest terms, values only: the insertions into the top-K lists are the single-pass kernel's
// (branch-free medians; same terms, same lists).
// MAXFORM (K = 1, interval form): the lists are the running maxima of the interval bounds of the l-inf distance
// (core/cuda/bound_inf_dist_cuda.cu:15-118), which leave as max(1e-10, .) instead of through the geometric sum.
// BOX (with IV): values and bounds in one walk, which meets no more marks than the bounds' alone (an input in its interval has the K-th
// largest term between theirs): 512 x 5120 x 5120, K = 10,
// 192 us, 133 and 78 for the two by themselves.  Four wavefronts per SIMD of 128 registers (five of 96 for the bounds alone).
template <int K, bool IV, bool MAXFORM = false, bool BOX = false>
__global__ void __launch_bounds__(64 * kMainWaves, BOX ? 4 : 1)
sc_main_kernel(const float* __restrict__ xT, const float* __restrict__ w, const uint32_t* __restrict__ bits,
               const float* __restrict__ xr, const float* __restrict__ low, const unsigned long long* __restrict__ count,
               unsigned long long limit, int B, int Bp, int M, int Mp, int N, float q, float* __restrict__ yL,
               float* __restrict__ yU, const float* __restrict__ shift, float shift_sign, const float* __restrict__ xT2,
               float* __restrict__ y) {
    if (gate_closed(count, limit, 0)) return;
    static_assert(!MAXFORM || (K == 1 && IV), "the maximum form is the interval form with one entry");
    union Shared {
        uint16_t list[kMainWaves][kWalkListCap];
        float stage[BOX ? 3 : IV ? 2 : 1][kTileB][kMainTile + 1];
    };
    __shared__ Shared sh;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int MB = Mp / kMainTile, NCH = N / kChunk, item = main_item();
    const int mb = item % MB, s = item / MB, m = mb * kMainTile + wave;
    using X = typename std::conditional<IV, float2, float>::type;
    const X* __restrict__ xcol = reinterpret_cast<const X*>(xT) + (size_t)s * kTileB + lane;
    const float* __restrict__ vcol = BOX ? xT2 + (size_t)s * kTileB + lane : nullptr;
    int hi[2][K], lo[IV ? 2 : 1][IV ? K : 1], val[BOX ? 2 : 1][BOX ? K : 1];
    #pragma unroll
    for (int k = 0; k < K; k++) {
        hi[0][k] = hi[1][k] = 0;
        if constexpr (BOX) val[0][k] = val[1][k] = 0;
        if constexpr (IV) lo[0][k] = lo[1][k] = 0;
    }
    if (m < M) {   // wave-uniform
        const uint32_t* __restrict__ rowbits = bits + ((size_t)s * Mp + m) * table_row_words(N);
        const float* __restrict__ wrow = w + (size_t)m * N;
        const Caps<MAXFORM> caps{xr + (size_t)s * N * (MAXFORM ? 4 : 2)};
        const float LU = low[(size_t)s * (MAXFORM ? 2 : 1) * Mp + m], LL = MAXFORM ? low[(size_t)(s * 2 + 1) * Mp + m] : LU;
        const bool in0 = s * kTileB + lane < B, in1 = s * kTileB + lane + 64 < B;   // the lane's batch rows exist
        X xa[2][4], xb[2][4];
        float va[BOX ? 2 : 1][BOX ? 4 : 1], vb[BOX ? 2 : 1][BOX ? 4 : 1];
        auto load = [&](int buf, int i, int n) __attribute__((always_inline)) {
            xa[buf][i] = xcol[(size_t)n * Bp];
            xb[buf][i] = xcol[(size_t)n * Bp + 64];
            if constexpr (BOX) { va[buf][i] = vcol[(size_t)n * Bp]; vb[buf][i] = vcol[(size_t)n * Bp + 64]; }
        };
        auto use = [&](int buf, int i, int k, int, const Own& o) __attribute__((always_inline)) {
            const float wi = lane_value(o.a, k);
            if constexpr (BOX) insert_pair<K>(val[0], fmaxf(fabsf(va[buf][i] - wi), -1.f), val[1], fmaxf(fabsf(vb[buf][i] - wi), -1.f));
            if constexpr (IV && MAXFORM) {
                // a term with an undefined operand is dropped (min / max keep the defined one, as the reference's do;
                // the final max with 0 drops a term that is undefined altogether)
                const float a1 = wi - xa[buf][i].x, a2 = xa[buf][i].y - wi;
                const float b1 = wi - xb[buf][i].x, b2 = xb[buf][i].y - wi;
                insert_bits<K>(lo[0], fmaxf(-fminf(a1, a2), 0.f));
                insert_bits<K>(hi[0], fmaxf(fmaxf(a1, a2), 0.f));
                insert_bits<K>(lo[1], fmaxf(-fminf(b1, b2), 0.f));
                insert_bits<K>(hi[1], fmaxf(fmaxf(b1, b2), 0.f));
            } else if constexpr (IV) {
                const float a1 = wi - xa[buf][i].x, a2 = xa[buf][i].y - wi;
                const float b1 = wi - xb[buf][i].x, b2 = xb[buf][i].y - wi;
                // (the maximum with -1 turns a term that is undefined altogether, whose bit pattern would order above
                // every number, into a negative one, which the lists ignore; three-operand maxima, so it costs no
                // instruction)
                insert_pair<K>(lo[0], fmaxf(fmaxf(-a1, -a2), -1.f), lo[1], fmaxf(fmaxf(-b1, -b2), -1.f));
                insert_pair<K>(hi[0], fmaxf(fmaxf(a1, a2), -1.f), hi[1], fmaxf(fmaxf(b1, b2), -1.f));
            } else {
                // (the same for the value form: the maximum stands where the absolute value's own instruction stood)
                insert_pair<K>(hi[0], fmaxf(fabsf(xa[buf][i] - wi), -1.f), hi[1], fmaxf(fabsf(xb[buf][i] - wi), -1.f));
            }
        };
        uint16_t* list = sh.list[wave];
        float thU = 0.f, thL = 0.f;   // smallest entries of the lists over the tile's rows (rows past the last one do not count)
        auto smallest = [&](int v0, int v1) __attribute__((always_inline)) {
            const int none = 0x7f800000;
            return wave_min_nonneg(__builtin_bit_cast(float, min(in0 ? v0 : none, in1 ? v1 : none)));
        };
        for_marks(list, NCH, lane, [&](int c) __attribute__((always_inline)) { return rowbits[c]; },
                  [&](int total, bool first) __attribute__((always_inline)) {
            walk_marks<false, false, kSample, walk_short(K)>(list, total, first, lane,
                [&](int n) __attribute__((always_inline)) { return Own{wrow[n], 0.f}; },
                [&](int n, const Own& o) __attribute__((always_inline)) { const float2 v = caps(n, o.a); return fmaxf(v.x - LU, v.y - LL); },
                load, use, use,
                [&](bool) __attribute__((always_inline)) {
                    // (one cap stands for every result of the forms without ranges of l and u apart)
                    if constexpr (BOX) thU = thL = smallest(min(min(hi[0][0], lo[0][0]), val[0][0]), min(min(hi[1][0], lo[1][0]), val[1][0]));
                    else if constexpr (IV && !MAXFORM) thU = thL = smallest(min(hi[0][0], lo[0][0]), min(hi[1][0], lo[1][0]));
                    else {
                        thU = smallest(hi[0][0], hi[1][0]);
                        if constexpr (IV) thL = smallest(lo[0][0], lo[1][0]);
                        else thL = thU;
                    }
                },
                [&](int n, const Own& o) __attribute__((always_inline)) { const float2 v = caps(n, o.a); return !(v.x < thU) || !(v.y < thL); },
                [] {});
        });
    }
    __syncthreads();
    #pragma unroll
    for (int j = 0; j < 2; j++) {
        if constexpr (MAXFORM) {
            sh.stage[0][lane + 64 * j][wave] = fmaxf(__builtin_bit_cast(float, hi[j][0]), kEps);
            sh.stage[1][lane + 64 * j][wave] = fmaxf(__builtin_bit_cast(float, lo[j][0]), kEps);
        } else {
            sh.stage[0][lane + 64 * j][wave] = geo_sum_bits<K>(hi[j], q);
            if constexpr (IV) sh.stage[1][lane + 64 * j][wave] = geo_sum_bits<K>(lo[j], q);
            if constexpr (BOX) sh.stage[2][lane + 64 * j][wave] = geo_sum_bits<K>(val[j], q);
        }
    }
    __syncthreads();
    for (int e = tid; e < kTileB * kMainTile; e += 64 * kMainWaves) {
        const int bl = e / kMainTile, mloc = e % kMainTile;
        const int b = s * kTileB + bl, mm = mb * kMainTile + mloc;
        if (b < B && mm < M) {
            const float add = output_shift(shift, shift_sign, mm);
            yU[(size_t)b * M + mm] = sh.stage[0][bl][mloc] + add;
            if constexpr (IV) yL[(size_t)b * M + mm] = sh.stage[1][bl][mloc] + add;
            if constexpr (BOX) y[(size_t)b * M + mm] = sh.stage[2][bl][mloc] + add;
        }
    }
}

// l-inf distance (maximum and where it sits) from the same tables, value form, optionally under the factored mask.
// As sc_main_kernel, with the running maximum and its position (input number, bit 31 = the difference is negative;
// the marks are walked in ascending input order and only a larger term replaces the maximum, so the first of
// equal terms wins as in core/cuda/inf_dist_cuda.cu:176-190) instead of the top-K lists.  `low` holds the bound the
// marks were taken against: every unmarked input's term is below it in every row, so a maximum that reaches it is
// the maximum over all inputs.  Under the mask a row may keep none of the inputs the bound rests on; if any row of
// the wavefront ends below the bound, the wavefront walks the weight row again over every input it keeps (`wkeep`
// words; all inputs without a mask).
template <bool POS>
__global__ void __launch_bounds__(64 * kMainWaves)
mc_main_kernel(const float* __restrict__ xT, const float* __restrict__ w, const uint32_t* __restrict__ bits,
               const uint32_t* __restrict__ wkeep, const float* __restrict__ xr, const float* __restrict__ low,
               const unsigned long long* __restrict__ count, unsigned long long limit, int B, int Bp, int M, int Mp,
               int N, float* __restrict__ y, int* __restrict__ pos) {
    if (gate_closed(count, limit, 0)) return;
    union Shared {
        uint16_t list[kMainWaves][kWalkListCap];
        struct { float y[kTileB][kMainTile + 1]; int p[POS ? kTileB : 1][kMainTile + 1]; } stage;
    };
    __shared__ Shared sh;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int MB = Mp / kMainTile, NCH = N / kChunk, item = main_item();
    const int mb = item % MB, s = item / MB, m = mb * kMainTile + wave;
    const float* __restrict__ xcol = xT + (size_t)s * kTileB + lane;
    // per batch row of the lane: the difference of largest magnitude so far (its sign is the position's flag)
    // and the input it sits at; without positions only the magnitude
    float best[2] = {kEps, kEps};
    int where[2] = {0, 0};
    if (m < M) {   // wave-uniform
        const float* __restrict__ wrow = w + (size_t)m * N;
        const Caps<false> caps{xr + (size_t)s * N * 2};
        const bool in0 = s * kTileB + lane < B, in1 = s * kTileB + lane + 64 < B;   // the lane's batch rows exist
        uint16_t* list = sh.list[wave];
        float xa[2][4], xb[2][4];
        auto load = [&](int buf, int i, int n) __attribute__((always_inline)) {
            xa[buf][i] = xcol[(size_t)n * Bp];
            xb[buf][i] = xcol[(size_t)n * Bp + 64];
        };
        auto use = [&](int buf, int i, int k, int n, const Own& o) __attribute__((always_inline)) {
            const float wi = lane_value(o.a, k);
            const float d0 = xa[buf][i] - wi, d1 = xb[buf][i] - wi;
            // an undefined difference (an input the row does not keep) never compares greater
            if constexpr (POS) {
                const bool g0 = fabsf(d0) > fabsf(best[0]), g1 = fabsf(d1) > fabsf(best[1]);
                best[0] = g0 ? d0 : best[0]; where[0] = g0 ? n : where[0];
                best[1] = g1 ? d1 : best[1]; where[1] = g1 ? n : where[1];
            } else {
                best[0] = fmaxf(best[0], fabsf(d0));
                best[1] = fmaxf(best[1], fabsf(d1));
            }
        };
        float th = 0.f;   // smallest maximum of the tile's rows so far (rows past the last one do not count)
        // first pass: the table's words; second pass: the inputs that the row keeps
        const uint32_t* __restrict__ rowbits = bits + ((size_t)s * Mp + m) * table_row_words(N);
        for (int pass = 0; pass < 2; pass++) {
            for_marks(list, NCH, lane, [&](int c) __attribute__((always_inline)) {
                          return pass == 0 ? rowbits[c] : wkeep ? wkeep[(size_t)m * NCH + c] : ~0u;
                      },
                      [&](int total, bool first) __attribute__((always_inline)) {
                walk_marks<POS, false, kSample, 0>(list, total, first, lane,
                    [&](int n) __attribute__((always_inline)) { return Own{wrow[n], 0.f}; },
                    [&](int n, const Own& o) __attribute__((always_inline)) { return caps(n, o.a).x; },
                    load, use, use,
                    [&](bool) __attribute__((always_inline)) {   // (never below what the strong marks showed, which an ordered walk forgets)
                        th = fmaxf(th, wave_min_nonneg(fminf(in0 ? fabsf(best[0]) : __builtin_inff(), in1 ? fabsf(best[1]) : __builtin_inff())));
                    },
                    [&](int n, const Own& o) __attribute__((always_inline)) { return !(caps(n, o.a).x < th); },
                    [&]() __attribute__((always_inline)) { best[0] = best[1] = kEps; where[0] = where[1] = 0; });
            });
            const float bound = low[(size_t)s * Mp + m];
            if (__builtin_amdgcn_ballot_w64((in0 && fabsf(best[0]) < bound) || (in1 && fabsf(best[1]) < bound)) == 0ull) break;
            if (pass == 0) {
                best[0] = best[1] = kEps;
                where[0] = where[1] = 0;
            }
        }
    }
    __syncthreads();
    #pragma unroll
    for (int j = 0; j < 2; j++) {
        sh.stage.y[lane + 64 * j][wave] = fabsf(best[j]);
        if (POS) sh.stage.p[lane + 64 * j][wave] = where[j] | (best[j] >= 0.f ? 0 : (int)kSign);
    }
    __syncthreads();
    for (int e = tid; e < kTileB * kMainTile; e += 64 * kMainWaves) {
        const int bl = e / kMainTile, mloc = e % kMainTile;
        const int b = s * kTileB + bl, mm = mb * kMainTile + mloc;
        if (b < B && mm < M) {
            y[(size_t)b * M + mm] = sh.stage.y[bl][mloc];
            if (POS) pos[(size_t)b * M + mm] = sh.stage.p[bl][mloc];
        }
    }
}

template <bool MASK>
int run_max(const float* x, const float* w, const uint32_t* xkeep, const uint32_t* wkeep, int B, int M, int N, int K, float* y,
            int* pos, const Carve& c, unsigned long long limit, hipStream_t st) {
    const int S = tiles_b(B), Bp = S * kTileB, Mp = mpad_of(M);
    int rc;
    hipLaunchKernelGGL((sc_range_kernel<false, false, MASK>), dim3(N / kChunk, S), dim3(256), 0, st, x, nullptr, w, xkeep, B, M, N, Bp, c.xr, c.xT, c.widths, c.count, nullptr, nullptr, nullptr);
    if ((rc = check_launch("sc_range_kernel"))) return rc;
    if ((rc = run_tables<false, MASK>(w, wkeep, S, M, Mp, N, K, c, limit, nullptr, st))) return rc;
    const dim3 grid((unsigned)(S * (Mp / kMainTile)));
    if (pos) hipLaunchKernelGGL((mc_main_kernel<true>), grid, dim3(64 * kMainWaves), 0, st, c.xT, w, c.bits, wkeep, c.xr, c.low, &c.count->marks, limit, B, Bp, M, Mp, N, y, pos);
    else hipLaunchKernelGGL((mc_main_kernel<false>), grid, dim3(64 * kMainWaves), 0, st, c.xT, w, c.bits, wkeep, c.xr, c.low, &c.count->marks, limit, B, Bp, M, Mp, N, y, pos);
    return check_launch("mc_main_kernel");
}

template <class F, int... R>
__device__ __forceinline__ void static_for(F&& f, std::integer_sequence<int, R...>) {
    (f(std::integral_constant<int, R>{}), ...);
}

// Value form with positions (core/cuda/sort_neuron.cu:111-214), in two walks.  The first is that of sc_main_kernel and gives
// each output its K-th largest term.  A smaller term is never among the K largest, and whether one at or above it enters depends
// only on entries at least that large; so the second walk, in ascending input order, takes the terms that reach it, K and
// their ties per output, and only these meet the ordered insertion that carries the input numbers: same values and positions
// as the scan over all inputs, ties included.  They differ from lane to lane, so the second walk only notes their inputs in
// LDS, and the lists are formed at the end, all lanes at work (an insertion at every mark that any of 128 outputs takes is four
// times the instructions of the value alone).  Outputs with more than two ties too many: their row is walked with an
// insertion at every mark.
// pos is (K, B, M) with slot 0 = largest; the K planes leave through LDS one after the other.
// 128 x 5120 x 5120, K = 10, 12 % marked: 149 us, 234 with the insertion at every mark.
template <int K>
__global__ void __launch_bounds__(64 * kMainWaves)
sp_main_kernel(const float* __restrict__ xT, const float* __restrict__ w, const uint32_t* __restrict__ bits,
               const float* __restrict__ xr, const unsigned long long* __restrict__ count, unsigned long long limit, int B,
               int Bp, int M, int Mp, int N, float q, float* __restrict__ y, int* __restrict__ pos) {
    if (gate_closed(count, limit, 0)) return;
    constexpr int kSlots = K + 2;
    union Shared {
        uint16_t list[kMainWaves][kWalkListCap];
        int stage[kTileB][kMainTile + 1];
    };
    __shared__ Shared sh;
    __shared__ uint16_t noted[kMainWaves][kSlots][kTileB];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int MB = Mp / kMainTile, NCH = N / kChunk, item = main_item();
    const int mb = item % MB, s = item / MB, m = mb * kMainTile + wave;
    const float* __restrict__ xcol = xT + (size_t)s * kTileB + lane;
    float res[2][K];
    int idx[2][K];
    #pragma unroll
    for (int k = 0; k < K; k++) { res[0][k] = res[1][k] = 0.f; idx[0][k] = idx[1][k] = 0; }
    if (m < M) {   // wave-uniform
        const uint32_t* __restrict__ rowbits = bits + ((size_t)s * Mp + m) * table_row_words(N);
        const float* __restrict__ wrow = w + (size_t)m * N;
        const Caps<false> caps{xr + (size_t)s * N * 2};
        const bool in0 = s * kTileB + lane < B, in1 = s * kTileB + lane + 64 < B;   // the lane's batch rows exist
        uint16_t* list = sh.list[wave];
        float xa[2][4], xb[2][4];
        auto load = [&](int buf, int i, int n) __attribute__((always_inline)) {
            xa[buf][i] = xcol[(size_t)n * Bp];
            xb[buf][i] = xcol[(size_t)n * Bp + 64];
        };
        auto word = [&](int c) __attribute__((always_inline)) { return rowbits[c]; };
        auto own = [&](int n) __attribute__((always_inline)) { return Own{wrow[n], 0.f}; };
        auto cap = [&](int n, const Own& o) __attribute__((always_inline)) { return caps(n, o.a).x; };
        float th = 0.f;   // smallest K-th largest term over the tile's rows so far (rows past the last one do not count)
        auto keep = [&](int n, const Own& o) __attribute__((always_inline)) { return !(caps(n, o.a).x < th); };
        float least[2];
        int listed;
        {
            int top[2][K];
            #pragma unroll
            for (int k = 0; k < K; k++) top[0][k] = top[1][k] = 0;
            auto value = [&](int buf, int i, int k, int, const Own& o) __attribute__((always_inline)) {
                const float wi = lane_value(o.a, k);   // (the maximum with -1: see sc_main_kernel)
                insert_pair<K>(top[0], fmaxf(fabsf(xa[buf][i] - wi), -1.f), top[1], fmaxf(fabsf(xb[buf][i] - wi), -1.f));
            };
            auto smallest = [&]() __attribute__((always_inline)) {
                const int none = 0x7f800000;
                th = wave_min_nonneg(__builtin_bit_cast(float, min(in0 ? top[0][0] : none, in1 ? top[1][0] : none)));
            };
            listed = for_marks(list, NCH, lane, word, [&](int total, bool first) __attribute__((always_inline)) {
                walk_marks<false, false, kSample, 0>(list, total, first, lane, own, cap, load, value, value,
                                         [&](bool) __attribute__((always_inline)) { smallest(); }, keep, [] {});
            });
            smallest();
            // only a positive term counts
            #pragma unroll
            for (int j = 0; j < 2; j++) least[j] = __builtin_bit_cast(float, max(top[j][0], 1));
        }
        int cnt[2] = {0, 0};
        auto note = [&](int buf, int i, int k, int n, const Own& o) __attribute__((always_inline)) {
            const float wi = lane_value(o.a, k);
            if (fabsf(xa[buf][i] - wi) >= least[0]) { noted[wave][min(cnt[0], kSlots - 1)][lane] = (uint16_t)n; cnt[0]++; }
            if (fabsf(xb[buf][i] - wi) >= least[1]) { noted[wave][min(cnt[1], kSlots - 1)][lane + 64] = (uint16_t)n; cnt[1]++; }
        };
        for_marks(list, NCH, lane, word, [&](int total, bool) __attribute__((always_inline)) {
            walk_marks<true, false, kSample, 0>(list, total, false, lane, own, cap, load, note, note, [](bool) {}, keep, [] {});
        }, listed);
        auto enter = [&](int j, float d, int n) __attribute__((always_inline)) {
            if (fabsf(d) > res[j][0] && fabsf(d) >= least[j]) topk_insert<K>(res[j], idx[j], fabsf(d), n | (d >= 0.f ? 0 : (int)kSign));
        };
        __builtin_amdgcn_wave_barrier();
        if (__builtin_amdgcn_ballot_w64(max(cnt[0], cnt[1]) > kSlots) == 0ull) {
            float d[2][2];
            int n[2][2];
            auto fetch = [&](int e) __attribute__((always_inline)) {
                #pragma unroll
                for (int j = 0; j < 2; j++) {
                    n[e & 1][j] = e < cnt[j] ? (int)noted[wave][e][lane + 64 * j] : 0;
                    d[e & 1][j] = xcol[(size_t)n[e & 1][j] * Bp + 64 * j] - wrow[n[e & 1][j]];
                }
            };
            fetch(0);
            #pragma unroll
            for (int e = 0; e < kSlots; e++) {
                if (e + 1 < kSlots) fetch(e + 1);
                #pragma unroll
                for (int j = 0; j < 2; j++) if (e < cnt[j]) enter(j, d[e & 1][j], n[e & 1][j]);
            }
        } else {
            auto ordered = [&](int buf, int i, int k, int n, const Own& o) __attribute__((always_inline)) {
                const float wi = lane_value(o.a, k);
                enter(0, xa[buf][i] - wi, n);
                enter(1, xb[buf][i] - wi, n);
            };
            for_marks(list, NCH, lane, word, [&](int total, bool) __attribute__((always_inline)) {
                walk_marks<true, false, kSample, 0>(list, total, false, lane, own, cap, load, ordered, ordered, [](bool) {}, keep, [] {});
            }, listed);
        }
    }
    __syncthreads();
    const size_t plane = (size_t)B * M;
    // the values, then the K planes of positions (slot 0 = largest = res[K-1]); the rounds are expanded at compile
    // time so that the lists are only ever indexed with constants and stay in registers
    static_for([&](auto R) __attribute__((always_inline)) {
        constexpr int round = decltype(R)::value;
        if (m < M) {
            #pragma unroll
            for (int j = 0; j < 2; j++) {
                if constexpr (round == 0) sh.stage[lane + 64 * j][wave] = __builtin_bit_cast(int, geo_sum<K>(res[j], q));
                else sh.stage[lane + 64 * j][wave] = idx[j][K - round];
            }
        }
        __syncthreads();
        for (int e = tid; e < kTileB * kMainTile; e += 64 * kMainWaves) {
            const int bl = e / kMainTile, mloc = e % kMainTile;
            const int b = s * kTileB + bl, mm = mb * kMainTile + mloc;
            if (b < B && mm < M) {
                const size_t o = (size_t)b * M + mm;
                if constexpr (round == 0) y[o] = __builtin_bit_cast(float, sh.stage[bl][mloc]);
                else pos[(size_t)(round - 1) * plane + o] = sh.stage[bl][mloc];
            }
        }
        __syncthreads();
    }, std::make_integer_sequence<int, K + 1>{});
}

template <int K, bool IV, bool MAXFORM = false>
int run(const float* xl, const float* xu, const float* w, int B, int M, int N, float q, float* outL, float* outU,
        int* pos, const Carve& c, unsigned long long limit, const float* shift, float shift_sign, const unsigned long long* unless, hipStream_t st) {
    const int S = tiles_b(B), Bp = S * kTileB, Mp = mpad_of(M);
    int rc;
    const dim3 grid(N / kChunk, S), block(256);
    if (unless != nullptr) hipLaunchKernelGGL((sc_range_kernel<IV, MAXFORM, false, false, true>), grid, block, 0, st, xl, xu, w, nullptr, B, M, N, Bp, c.xr, c.xT, c.widths, c.count, unless, nullptr, nullptr);
    else hipLaunchKernelGGL((sc_range_kernel<IV, MAXFORM, false>), grid, block, 0, st, xl, xu, w, nullptr, B, M, N, Bp, c.xr, c.xT, c.widths, c.count, nullptr, nullptr, nullptr);
    if ((rc = check_launch("sc_range_kernel"))) return rc;
    if ((rc = run_tables<MAXFORM, false>(w, nullptr, S, M, Mp, N, K, c, limit, unless, st))) return rc;
    if constexpr (!IV) {
        if (pos) {
            hipLaunchKernelGGL((sp_main_kernel<K>), dim3((unsigned)(S * (Mp / kMainTile))), dim3(64 * kMainWaves), 0, st,
                               c.xT, w, c.bits, c.xr, &c.count->marks, limit, B, Bp, M, Mp, N, q, outU, pos);
            return check_launch("sp_main_kernel");
        }
    }
    hipLaunchKernelGGL((sc_main_kernel<K, IV, MAXFORM>), dim3((unsigned)(S * (Mp / kMainTile))), dim3(64 * kMainWaves), 0, st,
                       c.xT, w, c.bits, c.xr, c.low, &c.count->marks, limit, B, Bp, M, Mp, N, q, outL, outU, shift, shift_sign, nullptr, nullptr);
    return check_launch("sc_main_kernel");
}

}  // namespace

size_t sort_cols_workspace(int B, int CO, int CI) {
    size_t sz[6];
    return carve_sizes(B, CO, CI, sz);
}

#define SD_SORT_COLS_K(X) \
    X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) X(17) \
    X(18) X(19) X(20) X(21) X(22) X(23) X(24) X(25)

int sort_cols_forward(const float* xl, const float* xu, const float* w, int B, int CO, int CI, float q, int K,
                      float* outL, float* outU, int* pos, void* ws, float density, const unsigned long long** gate,
                      unsigned long long* gate_limit, hipStream_t st, const float* shift, float shift_sign, const unsigned long long* unless) {
    if (CI % kChunk != 0 || CI > 65536 || B < 1 || CO < 1) {
        set_error("sort_cols_forward: shape not supported");
        return SD_ERR_ARG;
    }
    const Carve c = carve(ws, B, CO, CI);
    const float d = density < 0.f ? 0.f : density > 1.f ? 1.f : density;
    const unsigned long long limit = (unsigned long long)((double)tiles_b(B) * CO * CI * d);
    *gate = &c.count->marks;
    *gate_limit = limit;
    note_term_counts(&c.count->marks, 1, (double)tiles_b(B) * CO * CI, 1.0);
    if (K == 1 && xu) return run<1, true, true>(xl, xu, w, B, CO, CI, q, outL, outU, nullptr, c, limit, shift, shift_sign, unless, st);
    switch (K) {
#define X(k) case k: return xu ? run<k, true>(xl, xu, w, B, CO, CI, q, outL, outU, nullptr, c, limit, shift, shift_sign, unless, st) \
                               : run<k, false>(xl, nullptr, w, B, CO, CI, q, outL, outU, pos, c, limit, shift, shift_sign, unless, st);
        SD_SORT_COLS_K(X)
#undef X
    }
    set_error("sort_cols_forward: K=%d outside 2..25", K);
    return SD_ERR_ARG;
}


namespace {
float* box_inputs(void* ws, int B, int M, int N) { return reinterpret_cast<float*>(static_cast<char*>(ws) + align256(sort_cols_workspace(B, M, N))); }
}

size_t sort_cols_box_workspace(int B, int CO, int CI) {
    return align256(sort_cols_workspace(B, CO, CI)) + align256((size_t)CI * tiles_b(B) * kTileB * 4);
}

int sort_cols_box_tables(const float* x, const float* xl, const float* xu, const float* w, int B, int CO, int CI, void* ws,
                         float density, const unsigned long long** gate, unsigned long long* gate_limit, hipStream_t st) {
    if (CI % kChunk != 0 || CI > 65536 || B < 1 || CO < 1) {
        set_error("sort_cols_box_tables: shape not supported");
        return SD_ERR_ARG;
    }
    const Carve c = carve(ws, B, CO, CI);
    const float d = density < 0.f ? 0.f : density > 1.f ? 1.f : density;
    const int S = tiles_b(B), Bp = S * kTileB;
    *gate = &c.count->marks;
    *gate_limit = (unsigned long long)((double)S * CO * CI * d);
    note_term_counts(&c.count->marks, 1, (double)S * CO * CI, 1.0);
    hipLaunchKernelGGL((sc_range_kernel<true, false, false, true>), dim3(CI / kChunk, S), dim3(256), 0, st, xl, xu, w, nullptr, B, CO, CI, Bp, c.xr, c.xT,
                       c.widths, c.count, nullptr, x, box_inputs(ws, B, CO, CI));
    const int rc = check_launch("sc_range_kernel");
    return rc ? rc : run_tables<false, false>(w, nullptr, S, CO, mpad_of(CO), CI, kBoxK, c, *gate_limit, nullptr, st);
}

int sort_cols_box_main(const float* w, int B, int CO, int CI, float q, float* out, float* outL, float* outU, void* ws,
                       unsigned long long gate_limit, const float* shift, float shift_sign, hipStream_t st) {
    const Carve c = carve(ws, B, CO, CI);
    const int S = tiles_b(B), Bp = S * kTileB, Mp = mpad_of(CO);
    const dim3 grid((unsigned)(S * (Mp / kMainTile))), block(64 * kMainWaves);
    const float* xT2 = box_inputs(ws, B, CO, CI);
    hipLaunchKernelGGL((sc_main_kernel<kBoxK, true, false, true>), grid, block, 0, st, c.xT, w, c.bits, c.xr, c.low, &c.count->marks, gate_limit, B, Bp,
                       CO, Mp, CI, q, outL, outU, shift, shift_sign, xT2, out);
    return check_launch("sc_main_kernel");
}

int max_cols_depth(float keep_x) {
    if (keep_x >= 1.f) return 1;
    // inputs the bound rests on such that a row keeps none of them less often than once in 10^4 outputs (such an
    // output costs its wavefront a second pass over every input; more inputs lower the bound and mark more)
    const int need = (int)ceilf(logf(1e-4f) / logf(1.f - keep_x));
    for (int k : {8, 12, 16, 20, 24}) if (need <= k) return k;
    return 0;
}

int max_cols_forward(const float* x, const float* w, const uint32_t* xkeep, const uint32_t* wkeep, int B, int CO, int CI,
                     int K, float* y, int* pos, void* ws, float density, const unsigned long long** gate,
                     unsigned long long* gate_limit, hipStream_t st) {
    if (CI % kChunk != 0 || CI > 65536 || B < 1 || CO < 1 || (xkeep == nullptr) != (wkeep == nullptr)) {
        set_error("max_cols_forward: shape not supported");
        return SD_ERR_ARG;
    }
    const Carve c = carve(ws, B, CO, CI);
    const float d = density < 0.f ? 0.f : density > 1.f ? 1.f : density;
    const unsigned long long limit = (unsigned long long)((double)tiles_b(B) * CO * CI * d);
    *gate = &c.count->marks;
    *gate_limit = limit;
    note_term_counts(&c.count->marks, 1, (double)tiles_b(B) * CO * CI, 1.0);
    if (K < 1 || K > 64 || (!xkeep && K != 1)) { set_error("max_cols_forward: depth %d not supported", K); return SD_ERR_ARG; }
    return xkeep ? run_max<true>(x, w, xkeep, wkeep, B, CO, CI, K, y, pos, c, limit, st)
                 : run_max<false>(x, w, nullptr, nullptr, B, CO, CI, K, y, pos, c, limit, st);
}

}  // namespace sd
