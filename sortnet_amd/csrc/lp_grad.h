// Gradients of the l-p distance with the batch side of every term in scalar registers (lp_grad.hip).
#pragma once
#include "common.h"

namespace sd {

struct LpGradArgs {
    const float* gy; const float* x; const float* w; const float* y;
    float* gx; float* gw;             // gw null: the gradient of the inputs alone
    const int* ci_idx; const int* co_idx;
    int R, HW, G, COg, CIg, W_COg, W_CIg;
};

// bytes of workspace (what the kernel reads the batch side from, and planes of partial sums) that lp_grad needs
size_t lp_grad_workspace(const LpGradArgs& a);

// both gradients (or that of the inputs) for p - 1 = ip, a whole number in 0..8, or any pm1 = p - 1 > 0 (ip < 0)
int lp_grad(int ip, float pm1, const LpGradArgs& a, void* ws, hipStream_t st);

// slices of the output channels that the general kernel (lp.hip) cuts `blocks` workgroups of 256 inputs and 32 rows into
int lp_even_slices(long long blocks, int slots, int channels);

// out[o] = the sum of `planes` partial sums, `plane` floats apart, in plane order (lp.hip)
int lp_merge_planes(const float* part, float* out, size_t total, size_t plane, int planes, hipStream_t st);

}  // namespace sd
