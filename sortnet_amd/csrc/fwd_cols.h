// Forward of layers with several positions per sample (convolutions), dense in both channels; see fwd_cols.hip.
#pragma once
#include "common.h"

namespace sd {

// Whether the kernels serve the call: no index lists, no mask, one input tensor, and at least so many positions per sample and
// terms.  Fewer positions leave a wavefront's loads in pieces (in us, tiles -> this: 128 x 2700 x 1024 x 4 98 -> 118 with
// positions, 72 -> 95 without; 64 x 288 x 256 x 9 28 -> 27, 12 -> 21; x 16 36 -> 24, 14.4 -> 15.0; x 25 54 -> 30, 20.5 -> 19.1, at p = 8
// 25.2 -> 25.0); small layers do not make up for the launch that lays the weights out (16 x 144 x 64 x 16, 2.4 M terms, with positions
// 12 -> 14, x 64 18 -> 15; without, 16 x 144 x 64 x 64 9.5 -> 11.2, x 256 11.9 -> 11.5; p = 8, 16 x 800 x 64 x 256, 210 M terms,
// 32.5 -> 33.8, 64 x 288 x 256 x 64, 302 M, 40.1 -> 40.1).
// Images of up to 64 x 64 positions, what the figures cover; above them the kernels that stage tiles stay, as with index lists.
constexpr int kColsHW = 25, kColsPosHW = 16, kColsMostHW = 4096;
constexpr long long kColsTerms = 1ll << 26, kColsPosTerms = 1ll << 22, kColsLpTerms = 1ll << 28;
bool cols_ok(const FwdArgs& a, int hw, long long terms);
// slices of the reduction range
int cols_nsplit(const FwdArgs& a);
// bytes of the weights as the kernels read them
size_t cols_workspace(const FwdArgs& a);

// l-inf distance, with positions where a.p0 is set (then a.packed0, cleared, takes the slices' results where a.nsplit > 1);
// without them and a.nsplit > 1 the outputs have been cleared
int cols_linf(const FwdArgs& a, void* ws, hipStream_t stream);
// l-p distance of a whole p, 1 to 8; partial sums as LpPlain leaves them
int cols_lp(int ip, const FwdArgs& a, void* ws, hipStream_t stream);

}  // namespace sd
