// Patches of a convolutional distance layer (core/models/norm_dist.py:148-155 uses torch's unfold): the gather of every
// window into a column, and its transpose, the sum of a column gradient back into the image.
//
// Both are copies bound by memory, with one work-item per element of the larger side and neighbouring work-items on
// neighbouring output addresses.  torch's unfold launches one kernel per image whose work-items each walk a whole
// window: 128 images of 3 x 32 x 32 through a 30 x 30 window (four positions) took 128 launches of 114 us; here it is
// one launch over all images (5.5 MB written).
#include "common.h"

namespace sd {

struct Window {
    int C, H, W, KH, KW, stride, pad, dil, OH, OW;
};

// out[b, (c, i, j), (oy, ox)] = x[b, c, oy * stride - pad + i * dil, ox * stride - pad + j * dil], 0 outside the image
__global__ void __launch_bounds__(256) unfold_kernel(const float* __restrict__ x, Window g, uint32_t total, float* __restrict__ out) {
    const uint32_t o = blockIdx.x * 256u + threadIdx.x;
    if (o >= total) return;
    const uint32_t L = (uint32_t)(g.OH * g.OW);
    uint32_t t = o / L;
    const uint32_t pos = o - t * L, oy = pos / (uint32_t)g.OW, ox = pos - oy * (uint32_t)g.OW;
    const uint32_t u = t / (uint32_t)g.KW, j = t - u * (uint32_t)g.KW;
    const uint32_t bc = u / (uint32_t)g.KH, i = u - bc * (uint32_t)g.KH;      // bc = b * C + c
    const int y = (int)oy * g.stride - g.pad + (int)i * g.dil, xx = (int)ox * g.stride - g.pad + (int)j * g.dil;
    const bool in = y >= 0 && y < g.H && xx >= 0 && xx < g.W;
    out[o] = in ? x[((size_t)bc * g.H + y) * g.W + xx] : 0.f;
}

// gx[b, c, y, x] = sum over the windows that hold the pixel of gcol[b, (c, i, j), (oy, ox)], in window order.  Only the
// window positions that reach the pixel are visited (at most ceil(KH / stride) x ceil(KW / stride) when dil = 1).
__global__ void __launch_bounds__(256) fold_kernel(const float* __restrict__ gcol, Window g, uint32_t total, float* __restrict__ gx) {
    const uint32_t o = blockIdx.x * 256u + threadIdx.x;
    if (o >= total) return;
    const uint32_t row = o / (uint32_t)g.W;
    const int xx = (int)(o - row * (uint32_t)g.W);
    const uint32_t bc = row / (uint32_t)g.H;
    const int y = (int)(row - bc * (uint32_t)g.H);
    const int L = g.OH * g.OW;
    auto first = [&](int v, int k) {               // smallest window number whose last tap is not left of v
        const int t = v + g.pad - (k - 1) * g.dil;
        return t <= 0 ? 0 : (t + g.stride - 1) / g.stride;
    };
    auto last = [&](int v, int n) { const int t = (v + g.pad) / g.stride; return t < n ? t : n - 1; };
    const int oy1 = last(y, g.OH), ox0 = first(xx, g.KW), ox1 = last(xx, g.OW);
    float s = 0.f;
    for (int oy = first(y, g.KH); oy <= oy1; oy++) {
        const int ti = y + g.pad - oy * g.stride, i = ti / g.dil;
        if (i * g.dil != ti) continue;
        for (int ox = ox0; ox <= ox1; ox++) {
            const int tj = xx + g.pad - ox * g.stride, j = tj / g.dil;
            if (j * g.dil != tj) continue;
            s += gcol[(((size_t)bc * g.KH + i) * g.KW + j) * L + oy * g.OW + ox];
        }
    }
    gx[o] = s;
}

static int make_window(Window& g, const char* who, int B, int C, int H, int W, int KH, int KW, int stride, int pad, int dil) {
    SD_REQUIRE(B > 0 && C > 0 && H > 0 && W > 0 && KH > 0 && KW > 0, "%s: sizes must be positive", who);
    SD_REQUIRE(stride > 0 && pad >= 0 && dil > 0, "%s: stride=%d, padding=%d or dilation=%d out of range", who, stride, pad, dil);
    g = Window{C, H, W, KH, KW, stride, pad, dil, 0, 0};
    const long long sy = (long long)H + 2ll * pad - (long long)dil * (KH - 1) - 1, sx = (long long)W + 2ll * pad - (long long)dil * (KW - 1) - 1;
    SD_REQUIRE(sy >= 0 && sx >= 0, "%s: a %d x %d window does not fit into %d x %d (padding %d, dilation %d)", who, KH, KW, H, W, pad, dil);
    g.OH = (int)(sy / stride) + 1; g.OW = (int)(sx / stride) + 1;
    SD_REQUIRE((long long)B * C * H * W < (1ll << 31) && (double)B * C * KH * KW * g.OH * g.OW < 2147483648.0,
               "%s: tensor too large for 32-bit indexing", who);
    return SD_OK;
}

}  // namespace sd

using namespace sd;

extern "C" int sd_unfold(const float* input, int B, int C, int H, int W, int KH, int KW, int stride, int padding, int dilation,
                         float* output, sd_stream_t stream) {
    Window g;
    int rc = make_window(g, "unfold", B, C, H, W, KH, KW, stride, padding, dilation);
    if (rc) return rc;
    SD_REQUIRE(input && output, "unfold: null pointer");
    const uint32_t total = (uint32_t)B * C * KH * KW * g.OH * g.OW;
    hipLaunchKernelGGL(unfold_kernel, dim3((total + 255u) / 256u), dim3(256), 0, static_cast<hipStream_t>(stream), input, g, total, output);
    return check_launch("unfold_kernel");
}

extern "C" int sd_fold(const float* columns, int B, int C, int H, int W, int KH, int KW, int stride, int padding, int dilation,
                       float* output, sd_stream_t stream) {
    Window g;
    int rc = make_window(g, "fold", B, C, H, W, KH, KW, stride, padding, dilation);
    if (rc) return rc;
    SD_REQUIRE(columns && output, "fold: null pointer");
    const uint32_t total = (uint32_t)B * C * H * W;
    hipLaunchKernelGGL(fold_kernel, dim3((total + 255u) / 256u), dim3(256), 0, static_cast<hipStream_t>(stream), columns, g, total, output);
    return check_launch("fold_kernel");
}
