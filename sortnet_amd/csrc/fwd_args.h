// Host-side validation and FwdArgs construction shared by the forward entry points.
#pragma once
#include <cmath>
#include "common.h"

namespace sd {

inline bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// Validates the common shape arguments and fills the shape part of FwdArgs.
// Returns SD_OK or SD_ERR_ARG (message set).
inline int make_fwd_args(FwdArgs& a, const char* who, const float* x0, const float* x1, const float* w,
                         int B, int CO, int CI, int G, int HW,
                         const int* ci_idx, const int* co_idx, int W_CO, int W_CI) {
    SD_REQUIRE(x0 && w, "%s: null input or weight pointer", who);
    SD_REQUIRE(B > 0 && CO > 0 && CI > 0 && G > 0 && HW > 0, "%s: sizes must be positive (B=%d CO=%d CI=%d G=%d HW=%d)",
               who, B, CO, CI, G, HW);
    SD_REQUIRE(CO % G == 0 && CI % G == 0, "%s: CO=%d and CI=%d must be multiples of G=%d", who, CO, CI, G);
    SD_REQUIRE((long long)B * HW < (1ll << 31) && (long long)B * CO * HW < (1ll << 31) &&
               (long long)B * CI * HW < (1ll << 31), "%s: tensor too large for 32-bit indexing", who);
    a = FwdArgs{};
    note_term_counts(nullptr, 0, 1.0, 1.0);   // until a table kernel is queued for this call
    a.x0 = x0; a.x1 = x1; a.w = w;
    a.ci_idx = ci_idx; a.co_idx = co_idx;
    a.B = B; a.R = B * HW; a.HW = HW; a.G = G;
    a.COg = CO / G; a.CIg = CI / G;
    if (co_idx) {
        SD_REQUIRE(W_CO > 0 && W_CO % G == 0, "%s: W_CO=%d must be a positive multiple of G", who, W_CO);
        a.W_COg = W_CO / G;
    } else a.W_COg = a.COg;
    if (ci_idx) {
        SD_REQUIRE(W_CI > 0 && W_CI % G == 0, "%s: W_CI=%d must be a positive multiple of G", who, W_CI);
        a.W_CIg = W_CI / G;
    } else a.W_CIg = a.CIg;
    SD_REQUIRE((long long)G * a.W_COg * a.W_CIg < (1ll << 31), "%s: weight too large for 32-bit indexing", who);
    a.nsplit = 1;
    a.mask_mode = -1;
    bool vec = HW == 1 && a.CIg % 4 == 0;
    a.fast_x = vec && aligned16(x0) && (!x1 || aligned16(x1));
    a.fast_w = !ci_idx && a.CIg % 4 == 0 && a.W_CIg % 4 == 0 && aligned16(w);
    return SD_OK;
}

// how many slices to cut the reduction range in.  A compute unit holds two to four of these
// workgroups at a time and a workgroup runs about as long alone as with neighbours, so the last,
// partly filled round of workgroups costs a full round: eight workgroups per compute unit keep that
// tail below a fifth of the run.  A slice keeps at least four LDS chunks (128 inputs).  The index-list
// kernels are bound by their gather loads, not by the tail, and pay for every slice with merge traffic: they
// ask for one workgroup per compute unit (per_cu).
inline int pick_nsplit(const FwdArgs& a, int BB, int BM, int per_cu = 8) {
    long long tiles = (long long)((a.R + BB - 1) / BB) * ((a.COg + BM - 1) / BM) * a.G;
    int chunks = (a.CIg + 31) / 32;
    long long want = (long long)per_cu * num_cus();
    int max_ns = chunks / 4;
    if (max_ns > 16) max_ns = 16;
    int ns = 1;
    while (ns * 2 <= max_ns && tiles * ns < want) ns *= 2;
    // Where that leaves compute units idle the slices go down to one chunk, until every unit has two workgroups (one
    // for the gather kernels): a workgroup of so small a problem waits on its chunks, one after the other, and the
    // merge of the slices is a few microseconds at most.  In us, four-chunk slices -> this, with narrow tiles below:
    // l-p at p = 8 on 32 x 784 x 256 40 -> 15, on 90 x 1600 x 230 41 -> 18; l-inf with positions 26 -> 10, 26 -> 17;
    // interval bounds on 256 x 10240 x 200 103 -> 68.  Four workgroups per unit were slower from 128 x 3072 x 1024 on
    // (l-inf 27 -> 33), one per unit below (p = 8 on 90 x 1600 x 230 18 -> 27).
    const long long fill = (per_cu > 1 ? 2ll : 1ll) * num_cus();
    if (!a.coarse && tiles * ns < fill && aligned16(a.y0) && aligned16(a.y1)) {   // (a merge by maximum starts from filled outputs)
        long long more = (fill + tiles - 1) / tiles;
        if (more > chunks) more = chunks;
        if (more > 64) more = 64;
        if (more > ns) ns = (int)more;
    }
    return ns;
}

// Whether the forward runs on tiles of 32 x 32 outputs (2 x 2 per work-item) instead of 32 or 64 x 64 or 128: up to as
// many chunks of 32 x 128 outputs as 32 per compute unit.  The narrow tile reads more LDS per term but pads less, fills
// the device with fewer slices and keeps more wavefronts in flight; larger layers keep the wide tiles, whose LDS traffic per
// term decides there.  Time on narrow over time on wide tiles, vector loads:
//   chunks per unit             4     24 (250 x 3072 x 1021)  24 (256 x 3072 x 1024)  32 (512 x 2048 x 1024)  48     72
//   l-inf                       0.78  0.89                    1.03                    1.08                    1.19   1.30
//   l-inf with positions        0.91  0.80                    0.84                    0.85                    1.02   1.05
//   interval / with positions   0.81  0.97 / 0.77             1.07 / 0.96             1.08 / 0.98             1.14   1.16
//   l-p, p = 8 / p = 24         0.85  0.98 / 0.96             0.99                    1.04 / 1.02             1.06   1.05
//   masked / with positions     -     0.88 / 0.81             -                       1.03 / 0.84             1.13   1.17
// The scalar-load kernels (index lists, several positions per sample, rows that are no multiple of 16 bytes) hold fewer wavefronts
// with their wide tile and go narrow up to twice that size.  Between 32 and 64 chunks per unit: lists p = inf 0.71 to 0.81,
// p = 8 0.95 to 0.99, p = 24 0.94 to 0.98; l-inf 0.50 to 0.87, with positions 0.80 to 0.86, p = 8 0.55 to 1.00; interval
// with positions 0.78 to 0.94, without 0.44 to 0.99 and, on four of nine shapes, 1.04 to 1.11; mask per term 0.94 to 0.98.
// (Above 64: lists at p = 8 1.04 to 1.07, l-p 1.06 to 1.11, interval 1.07 to 1.29.)  Under the factored mask, whose keep
// bits are drawn as a tile is staged, and a narrow one is staged more often, they keep the first limit: there 0.93 to 1.20.
inline bool narrow_tiles(const FwdArgs& a) {
    const long long tiles = (long long)((a.R + 31) / 32) * ((a.COg + 127) / 128) * a.G;
    const bool vector = a.fast_x && a.fast_w;
    return tiles * ((a.CIg + 31) / 32) < (vector || a.mask_mode == SD_MASK_FACTORED ? 32ll : 64ll) * num_cus();
}

// rows per work-item (batch tile = 16 * TB rows): the largest candidate whose tiles, after split-N,
// still give the device about four workgroups per compute unit; small problems fall to the smallest
inline int pick_tb(const FwdArgs& a, const int* candidates, int n, int BM) {
    for (int k = 0; k < n; k++) {
        int BB = 16 * candidates[k];
        if (a.R <= BB / 2 && k + 1 < n) continue;   // tile mostly padding
        long long tiles = (long long)((a.R + BB - 1) / BB) * ((a.COg + BM - 1) / BM) * a.G;
        if (tiles * pick_nsplit(a, BB, BM) >= 4ll * num_cus()) return candidates[k];
    }
    return candidates[n - 1];
}

}  // namespace sd
