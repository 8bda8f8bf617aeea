// Forward of layers that meet few batch rows: weights streamed once, a wavefront per weight row (row_stream.hip).
#pragma once
#include "common.h"

namespace sd {

// Size up to which a call is streamed, set where the time meets that of the tile kernels (with their fill and resolve
// launches) and, for the sort neuron, of its tables: terms (batch rows x weight rows x inputs) for the maxima, whose
// time follows the terms; outputs for the sort neuron, whose selection takes about 1 ns per output whatever the row's
// length (half of that where six wavefronts fit a SIMD), against kernels that take about 0.1 us per input of a row.  Measured, us, streamed / before
// (rows x inputs x outputs):
//   l-inf           32 x 3072 x 1024 (101 M) 13 / 22, 64 x (201 M) 23 / 24, 128 x 1024 x 1024 (134 M) 23 / 18,
//                   256 x 10240 x 10 (26 M) 14 / 60
//   with positions  64 x 1024 x 1024 (67 M) 18 / 23, 512 x 784 x 256 (103 M) 33 / 27, 256 x 10240 x 10 17 / 48
//   masked          32 x 1024 x 1024 (34 M) 17 / 28, 32 x 10240 x 200 (66 M) 79 / 56
//   interval        64 x 1024 x 1024 (67 M) 22 / 26 (with positions 35 / 34), 128 x 784 x 256 (26 M) 12 / 37 (20 / 39)
//   sort neuron     64 x 1024 x 1024 (66 k outputs) 41 / 114, 128 x 1024 x 1024 78 / 40 from tables, 512 x 5120 x 10 15 / 205
//   its interval    32 x 1024 x 1024 (33 k outputs) 41 / 154, 64 x 81 / 46 from tables
// Without tables, streamed / every term (row_stream_sort_before_terms):
//   sort neuron     100 x 1658 x 1658 (166 k outputs) 167 / 200, 150 x 1001 x 1001 96 / 130, 200 x 500 x 500 (200 per input) 60 / 52,
//                   36 x 3333 x 3333 (120 k) 233 / 440, 24 x 10239 x 10240 (246 k) 1685 / 1408, 512 x 5121 x 500 (256 k) 1152 / 649
//   its interval    78 x 1658 x 1658 (129 k) 285 / 301, 100 x 640 x 640 (100 per input) 75 / 90, 128 x 103 / 90, 24 x 3072 x 3072 162 / 308,
//                   30 x 3333 x 3333 (100 k) 630 / 547
constexpr long long kStreamMaxTerms = 3ll << 25, kStreamPosTerms = 5ll << 24, kStreamMaskTerms = 3ll << 24;
constexpr long long kStreamBoundTerms = 5ll << 24, kStreamBoundPosTerms = 7ll << 23;

// whether the streaming kernels serve a call of at most `limit` terms by its sizes: dense, rows short enough for the registers
bool row_stream_sizes_ok(const FwdArgs& a, long long limit);
// the same with what they read at hand: no mask, or a factored one with its keep bits built
bool row_stream_ok(const FwdArgs& a, long long limit);
// the same for the sort neuron (a.x1: its interval form)
bool row_stream_sort_ok(const FwdArgs& a);
// the same for a layer without tables (no room for them in its shape, or none that served it lately), against the kernels
// that form every term
bool row_stream_sort_before_terms(const FwdArgs& a);
// y = max(1e-10, max_n |x - w|), with the position of the maximum when a.p0 is set
int row_stream_linf(const FwdArgs& a, hipStream_t stream);
// interval bounds of the l-inf layer, with positions when a.p0 is set
int row_stream_bound(const FwdArgs& a, hipStream_t stream);
// sort neuron, values: the K largest terms with geometric weights (a.q); interval bounds of it when a.x1 is set
int row_stream_sort(const FwdArgs& a, int K, hipStream_t stream);

}  // namespace sd
