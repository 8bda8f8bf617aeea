// Mean shift over batch and spatial positions, the step that follows every distance layer
// (core/models/bound_basic_module.py:106-157, training form without index list):
//   mean[c] = mean_{b,hw} x[b,c,hw];  running = (1 - momentum) running + momentum mean;  y = x - mean[c]
// the plain per-channel shift y = x - shift[c] used in evaluation mode and for a bias, and the training form
// with a kept-channel index list per 32-sample sub-batch.
#include "common.h"

namespace sd {

// One workgroup owns 64 channels (HW == 1) or one channel (HW > 1); 16 groups of 64 work-items walk
// the batch in parallel, partial sums meet in LDS, the sum order is fixed (deterministic result).  Few workgroups, so
// what counts is the loads each keeps in flight: eight rows at a time (512 x 5120 13.7 -> 4.9 us) and, with positions, the LDS
// reads of the last sum, which has few groups to add where the batch is small (128 x 1024 x 4 10.9 -> 7.8 us).
__global__ void __launch_bounds__(1024) channel_mean_kernel(const float* __restrict__ x, int B, int C, int HW,
                                                            float* __restrict__ mean, float* __restrict__ running,
                                                            float momentum) {
    __shared__ float part[16][64];
    const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
    float s = 0.f;
    if (HW == 1) {
        const int c = blockIdx.x * 64 + lane;
        if (c < C) {
            #pragma unroll 8
            for (int b = grp; b < B; b += 16) s += x[(size_t)b * C + c];
        }
        part[grp][lane] = s;
        __syncthreads();
        if (grp == 0 && c < C) {
            float t = 0.f;
            #pragma unroll
            for (int k = 0; k < 16; k++) t += part[k][lane];
            float m = t / (float)B;
            mean[c] = m;
            if (running) running[c] = (1.f - momentum) * running[c] + momentum * m;
        }
    } else {
        const int c = blockIdx.x;
        const uint32_t n = (uint32_t)B * (uint32_t)HW;      // (the tensor has fewer than 2^31 elements)
        #pragma unroll 4
        for (uint32_t i = threadIdx.x; i < n; i += 1024) {
            const uint32_t b = i / (uint32_t)HW, hw = i - b * (uint32_t)HW;
            s += x[((size_t)b * C + c) * HW + hw];
        }
        part[grp][lane] = s;
        __syncthreads();
        if (threadIdx.x == 0) {
            float t = 0.f;
            const int live = n < 1024u ? (int)((n + 63) / 64) : 16;      // the other groups hold zeros
            for (int k = 0; k < live; k++) {
                #pragma unroll
                for (int l = 0; l < 64; l++) t += part[k][l];
            }
            float m = t / (float)n;
            mean[c] = m;
            if (running) running[c] = (1.f - momentum) * running[c] + momentum * m;
        }
    }
}

// Both in one launch for up to 512 samples and 1, 4, 8 .. 64 positions: a workgroup owns 64 neighbouring values of a sample (64 / HW channels),
// its wavefronts keep every 16th sample in registers, and the values leave again with the mean subtracted.  Two launches were bound
// by the launches and, with positions, by reading one channel at a time (16 bytes of a cache line at HW = 4).  The order of the sums is
// that of the kernel above, so the bits are: with positions, where its 1024 work-items took every 1024th value of a channel and one added
// their sums up, the sums of `span` = 1024 / HW samples lie in LDS for one lane per channel to add.  Two launches -> one, us of the device (the
// host has a launch of 3 us less): 512 x 5120 9.3 -> 6.3, 128 x 1024 8.1 -> 4.7, with 4 positions 10.0 -> 7.7, 512 x 5120 x 4 72.6 -> 31.5.
constexpr int kShiftRows = 32;   // samples of a wavefront
template <int ROWS, bool POSITIONS>
__global__ void __launch_bounds__(1024) channel_mean_shift_kernel(const float* x, int B, int cols, int HW, float* __restrict__ mean,
                                                                  float* __restrict__ running, float momentum, float* y) {   // (y may be x)
    extern __shared__ __attribute__((aligned(16))) float part[];   // [16 or min(B, span)][64]
    __shared__ float shift[64];
    const int lane = threadIdx.x & 63, grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = blockIdx.x * 64 + lane, span = POSITIONS ? 1024 / HW : 16;
    const bool ok = col < cols;
    const float* src = x + (ok ? col : 0);
    float v[ROWS];
    #pragma unroll
    for (int k = 0; k < ROWS; k++) {
        const int b = grp + 16 * k;
        v[k] = src[(size_t)(b < B ? b : B - 1) * cols];
    }
    if constexpr (POSITIONS) {   // (the samples of a sum are all this wavefront's: span is a multiple of 16)
        #pragma unroll
        for (int k = 0; k < ROWS; k++) {
            const int b = grp + 16 * k;
            if (b < B) {
                float* sum = part + (b & (span - 1)) * 64 + lane;
                *sum = (b < span ? 0.f : *sum) + v[k];
            }
        }
    } else {
        float s = 0.f;
        #pragma unroll
        for (int k = 0; k < ROWS; k++) s += grp + 16 * k < B ? v[k] : 0.f;
        part[grp * 64 + lane] = s;
    }
    __syncthreads();
    if (grp == 0) {
        float t = 0.f;
        const int c = POSITIONS ? (int)(blockIdx.x * 64) / HW + lane : col;
        const bool mine = POSITIONS ? lane < 64 / HW && c * HW < cols : ok;
        if constexpr (POSITIONS) {
            if (mine) {
                const int rows = B < span ? B : span;
                const float* own = part + lane * HW;
                const int steps = __builtin_ctz(HW) - 2;   // of four positions: 2^steps to a sample
                #pragma unroll 8
                for (int i = 0; i < rows << steps; i++) {
                    const float4 e = *reinterpret_cast<const float4*>(own + (i >> steps) * 64 + 4 * (i & ((1 << steps) - 1)));
                    t += e.x; t += e.y; t += e.z; t += e.w;
                }
            }
        } else {
            #pragma unroll
            for (int k = 0; k < 16; k++) t += part[k * 64 + lane];
        }
        const float m = t / (float)((uint32_t)B * (uint32_t)HW);
        if constexpr (POSITIONS) { if (mine) for (int h = 0; h < HW; h++) shift[lane * HW + h] = m; }
        else shift[lane] = m;
        if (mine) {
            mean[c] = m;
            if (running) running[c] = (1.f - momentum) * running[c] + momentum * m;
        }
    }
    __syncthreads();
    if (!ok) return;
    const float m = shift[lane];
    #pragma unroll
    for (int k = 0; k < ROWS; k++) {
        const int b = grp + 16 * k;
        if (b < B) y[(size_t)b * cols + col] = v[k] - m;
    }
}

__global__ void __launch_bounds__(256) channel_shift_kernel(const float* x, const float* __restrict__ shift,
                                                            long long total, int C, int HW, float sign,
                                                            float* y, float* both) {   // (y may be x; grid.y = 2: `both` in place, too)
    if (blockIdx.y) x = y = both;
    long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= total) return;
    if (HW == 1 && C % 4 == 0 && i + 3 < total) {
        float4 v = *reinterpret_cast<const float4*>(x + i);
        float4 sh = *reinterpret_cast<const float4*>(shift + (i % C));
        v.x += sign * sh.x; v.y += sign * sh.y; v.z += sign * sh.z; v.w += sign * sh.w;
        *reinterpret_cast<float4*>(y + i) = v;
    } else {
        for (int k = 0; k < 4 && i + k < total; k++) {
            long long j = i + k;
            int c = (int)((j / HW) % C);
            y[j] = x[j] + sign * shift[c];
        }
    }
}

// ---- index-list form: the input holds, for every 32-sample sub-batch s, only the channels index[s, g, :] ----

// column sums of one sub-batch: work-item = one kept channel j of (s, g); the sum lands in the slot of the
// full channel it stands for.  A sub-batch lists a channel at most once, so slots are written at most once.
__global__ void __launch_bounds__(256) index_colsum_kernel(const float* __restrict__ x, const int* __restrict__ index,
                                                           int B, int G, int cnt, int Cg, int HW,
                                                           float* __restrict__ part, float* __restrict__ rows) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    const int sg = blockIdx.y, s = sg / G, g = sg - s * G;
    if (j >= cnt) return;
    const int b0 = s * kSubBatch, b1 = b0 + kSubBatch < B ? b0 + kSubBatch : B;
    float t = 0.f;
    if (HW == 1) {
        const float* src = x + (size_t)g * cnt + j;
        const size_t stride = (size_t)G * cnt;
        #pragma unroll 8
        for (int b = b0; b < b1; b++) t += src[b * stride];      // independent loads, added in sample order
    } else {
        for (int b = b0; b < b1; b++) {
            const float* src = x + ((size_t)(b * G + g) * cnt + j) * HW;
            for (int hw = 0; hw < HW; hw++) t += src[hw];
        }
    }
    const size_t slot = (size_t)s * G * Cg + (size_t)g * Cg + index[(size_t)sg * cnt + j];
    part[slot] = t;
    rows[slot] = (float)(b1 - b0);
}

// mean of every full channel over the sub-batches that kept it, in sub-batch order (deterministic)
__global__ void __launch_bounds__(256) index_mean_kernel(const float* __restrict__ part, const float* __restrict__ rows,
                                                         int S, int C, int HW, float* __restrict__ mean,
                                                         float* __restrict__ running, float momentum) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    float total = 0.f, seen = 1e-10f;
    for (int s = 0; s < S; s++) { total += part[(size_t)s * C + c]; seen += rows[(size_t)s * C + c]; }
    const float m = total / (seen * (float)HW);
    mean[c] = m;
    if (running) running[c] = (1.f - momentum) * running[c] + momentum * m;
}

__global__ void __launch_bounds__(256) index_shift_kernel(const float* __restrict__ x, const int* __restrict__ index,
                                                          const float* __restrict__ mean, long long total,
                                                          int G, int cnt, int Cg, int HW, float* __restrict__ y) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const long long t = i / HW;
    const int j = (int)(t % cnt);
    const long long bg = t / cnt;
    const int g = (int)(bg % G), b = (int)(bg / G);
    const int s = b / kSubBatch;
    y[i] = x[i] - mean[g * Cg + index[(size_t)(s * G + g) * cnt + j]];
}

// The three kernels above and the fill of their sums in one launch, for one position per sample.  A workgroup owns 64 full
// channels of a group; its wavefronts take a sub-batch each (up to 16 at a time).  A wavefront reads its list once and
// notes in LDS where each of the 64 channels stands in it (lists in any order), a lane then sums its channel's rows in
// sample order and the sub-batches are added in order: the same bits as above.  The rows are read a second time, from
// cache, for the shift.  A list that names a channel more than once (no list of a sampler does) has one of its columns in the
// mean, as above, and all of them shifted.  Four launches of 4 to 7 us each were bound by their launches: 32 x 192 of 256 channels
// 24 -> 6 us, 128 x 3840 of 5120 24 -> 12 us, 512 x 3840 of 5120 23 both ways.
constexpr int kFuseWaves = 16, kFuseSubs = 128;   // sub-batches at a time / at most (their positions are held in LDS)
__global__ void __launch_bounds__(64 * kFuseWaves) index_mean_shift_kernel(
    const float* __restrict__ x, const int* __restrict__ index, int B, int G, int cnt, int Cg, int S,
    float* __restrict__ mean, float* __restrict__ running, float momentum, float* __restrict__ y) {
    extern __shared__ int at[];                       // [S][64]: position of the channel in the sub-batch's list, or -1
    __shared__ float sums[kFuseWaves][64];
    __shared__ float shift[64];
    __shared__ int repeated;                          // a list names one of the channels more than once
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int g = blockIdx.y, c0 = blockIdx.x * 64, c = c0 + lane;
    const size_t stride = (size_t)G * cnt;
    // what a lane reads next may have been written by another lane of its wavefront
    auto posted = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    if (threadIdx.x == 0) repeated = 0;
    __syncthreads();
    float total = 0.f, seen = 1e-10f;                 // of wavefront 0
    for (int s0 = 0; s0 < S; s0 += waves) {
        const int s = s0 + wave;
        float t = 0.f;
        if (s < S) {
            int* slot = at + s * 64;
            slot[lane] = -1;
            posted();
            const int* list = index + (size_t)(s * G + g) * cnt;
            #pragma unroll 8
            for (int j = lane; j < cnt; j += 64) {
                const int k = list[j] - c0;
                if (k >= 0 && k < 64 && atomicExch(&slot[k], j) >= 0) repeated = 1;
            }
            posted();
            const int j = slot[lane];
            if (j >= 0) {
                const int b0 = s * kSubBatch, b1 = b0 + kSubBatch < B ? b0 + kSubBatch : B;
                const float* src = x + (size_t)g * cnt + j;
                #pragma unroll 8
                for (int b = b0; b < b1; b++) t += src[b * stride];
            }
        }
        sums[wave][lane] = t;
        __syncthreads();
        if (wave == 0) {
            for (int k = 0; k < waves && s0 + k < S; k++) {
                const int b0 = (s0 + k) * kSubBatch, b1 = b0 + kSubBatch < B ? b0 + kSubBatch : B;
                total += sums[k][lane];
                seen += at[(s0 + k) * 64 + lane] >= 0 ? (float)(b1 - b0) : 0.f;
            }
        }
        __syncthreads();
    }
    if (wave == 0) {
        const float m = total / seen;
        shift[lane] = m;
        if (c < Cg) {
            mean[g * Cg + c] = m;
            if (running) running[g * Cg + c] = (1.f - momentum) * running[g * Cg + c] + momentum * m;
        }
    }
    __syncthreads();
    if (repeated) {
        for (int s = wave; s < S; s += waves) {
            const int* list = index + (size_t)(s * G + g) * cnt;
            const int b0 = s * kSubBatch, b1 = b0 + kSubBatch < B ? b0 + kSubBatch : B;
            for (int j = lane; j < cnt; j += 64) {
                const int k = list[j] - c0;
                if (k < 0 || k >= 64) continue;
                const size_t o = (size_t)g * cnt + j;
                for (int b = b0; b < b1; b++) y[o + b * stride] = x[o + b * stride] - shift[k];
            }
        }
        return;
    }
    const float m = shift[lane];
    for (int s = wave; s < S; s += waves) {
        const int j = at[s * 64 + lane];
        if (j < 0) continue;
        const int b0 = s * kSubBatch, b1 = b0 + kSubBatch < B ? b0 + kSubBatch : B;
        const size_t o = (size_t)g * cnt + j;
        #pragma unroll 8
        for (int b = b0; b < b1; b++) y[o + b * stride] = x[o + b * stride] - m;
    }
}

int channel_shift(const float* x, const float* shift, int B, int C, int HW, float sign, float* y, hipStream_t stream) {
    const long long total = (long long)B * C * HW;
    hipLaunchKernelGGL(channel_shift_kernel, dim3((unsigned)((total / 4 + 255) / 256 + 1)), dim3(256), 0, stream, x, shift, total, C, HW, sign, y, nullptr);
    return check_launch("channel_shift_kernel");
}

int channel_shift_both(float* a, float* b, const float* shift, int B, int C, int HW, float sign, hipStream_t stream) {
    const long long total = (long long)B * C * HW;
    hipLaunchKernelGGL(channel_shift_kernel, dim3((unsigned)((total / 4 + 255) / 256 + 1), 2), dim3(256), 0, stream, a, shift, total, C, HW, sign, a, b);
    return check_launch("channel_shift_kernel");
}

static int check_dims(const char* who, int B, int C, int HW) {
    SD_REQUIRE(B > 0 && C > 0 && HW > 0, "%s: sizes must be positive", who);
    SD_REQUIRE((long long)B * C * HW < (1ll << 31), "%s: tensor too large for 32-bit indexing", who);
    return SD_OK;
}

}  // namespace sd

using namespace sd;

extern "C" int sd_mean_shift_forward(const float* input, int B, int C, int HW, float* mean, float* running_mean,
                                     float momentum, float* output, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    int rc = check_dims("mean_shift_forward", B, C, HW);
    if (rc) return rc;
    SD_REQUIRE(input && mean && output, "mean_shift_forward: null pointer");
    SD_REQUIRE(reinterpret_cast<uintptr_t>(input) % 16 == 0 && reinterpret_cast<uintptr_t>(output) % 16 == 0 &&
               reinterpret_cast<uintptr_t>(mean) % 16 == 0, "mean_shift_forward: buffers must be 16-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    // With positions the chain of one lane's additions bounds small layers (256 x 512 x 4 11.6 us in two launches, 12.8 in one; 129 x 64 x 16 10.5,
    // 12.1): up to 512 values of a channel, or tensors whose second reading costs more (512 x 1000 x 4 21.9 -> 15.3)
    const bool positions = HW >= 4 && HW <= 64 && (HW & (HW - 1)) == 0 && (B * HW <= 512 || (long long)B * C * HW >= 1ll << 20);
    if (B <= 16 * kShiftRows && (HW == 1 || positions)) {
        const int cols = C * HW, span = 1024 / HW;
        const dim3 blocks((cols + 63) / 64), threads(1024);
        const size_t lds = (size_t)(HW == 1 ? 16 : B < span ? B : span) * 64 * sizeof(float);
        if (HW == 1 && B <= 128) hipLaunchKernelGGL((channel_mean_shift_kernel<8, false>), blocks, threads, lds, st, input, B, cols, HW, mean, running_mean, momentum, output);
        else if (HW == 1) hipLaunchKernelGGL((channel_mean_shift_kernel<kShiftRows, false>), blocks, threads, lds, st, input, B, cols, HW, mean, running_mean, momentum, output);
        else if (B <= 128) hipLaunchKernelGGL((channel_mean_shift_kernel<8, true>), blocks, threads, lds, st, input, B, cols, HW, mean, running_mean, momentum, output);
        else hipLaunchKernelGGL((channel_mean_shift_kernel<kShiftRows, true>), blocks, threads, lds, st, input, B, cols, HW, mean, running_mean, momentum, output);
        return check_launch("channel_mean_shift_kernel");
    }
    dim3 grid(HW == 1 ? (C + 63) / 64 : C);
    hipLaunchKernelGGL(channel_mean_kernel, grid, dim3(1024), 0, st, input, B, C, HW, mean, running_mean, momentum);
    if ((rc = check_launch("channel_mean_kernel"))) return rc;
    return channel_shift(input, mean, B, C, HW, -1.f, output, st);
}

extern "C" int sd_channel_shift(const float* input, const float* shift, int B, int C, int HW, float sign,
                                float* output, sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    int rc = check_dims("channel_shift", B, C, HW);
    if (rc) return rc;
    SD_REQUIRE(input && shift && output, "channel_shift: null pointer");
    SD_REQUIRE(reinterpret_cast<uintptr_t>(input) % 16 == 0 && reinterpret_cast<uintptr_t>(output) % 16 == 0 &&
               reinterpret_cast<uintptr_t>(shift) % 16 == 0, "channel_shift: buffers must be 16-byte aligned");
    return channel_shift(input, shift, B, C, HW, sign, output, static_cast<hipStream_t>(stream));
}

extern "C" int sd_mean_shift_index_forward(const float* input, const int* index, int B, int G, int cnt, int Cg, int HW,
                                           float* mean, float* running_mean, float momentum, float* output,
                                           sd_stream_t stream) {
    sd::CallGuard call_guard;   // calls of several host threads reach a stream one after the other, whole
    SD_REQUIRE(G > 0 && cnt > 0 && Cg >= cnt, "mean_shift_index_forward: need G > 0 and 0 < cnt <= Cg (cnt=%d Cg=%d)", cnt, Cg);
    SD_REQUIRE((long long)G * cnt < (1ll << 31) && (long long)G * Cg < (1ll << 31), "mean_shift_index_forward: too many channels");
    int rc = check_dims("mean_shift_index_forward", B, G * cnt, HW);
    if (rc) return rc;
    SD_REQUIRE(input && index && mean && output, "mean_shift_index_forward: null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int S = (B + kSubBatch - 1) / kSubBatch, C = G * Cg;
    if (HW == 1 && S <= kFuseSubs && G < 65536) {
        const int waves = S < kFuseWaves ? S : kFuseWaves;
        hipLaunchKernelGGL(index_mean_shift_kernel, dim3((Cg + 63) / 64, G), dim3(64 * waves), (size_t)S * 64 * sizeof(int), st,
                           input, index, B, G, cnt, Cg, S, mean, running_mean, momentum, output);
        return check_launch("index_mean_shift_kernel");
    }
    float* part = static_cast<float*>(workspace((size_t)2 * S * C * sizeof(float), st));
    if (!part) return SD_ERR_HIP;
    float* rows = part + (size_t)S * C;
    if ((rc = fill_zero(part, (size_t)2 * S * C, st))) return rc;
    hipLaunchKernelGGL(index_colsum_kernel, dim3((cnt + 255) / 256, S * G), dim3(256), 0, st,
                       input, index, B, G, cnt, Cg, HW, part, rows);
    if ((rc = check_launch("index_colsum_kernel"))) return rc;
    hipLaunchKernelGGL(index_mean_kernel, dim3((C + 255) / 256), dim3(256), 0, st, part, rows, S, C, HW, mean,
                       running_mean, momentum);
    if ((rc = check_launch("index_mean_kernel"))) return rc;
    const long long total = (long long)B * G * cnt * HW;
    hipLaunchKernelGGL(index_shift_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                       input, index, mean, total, G, cnt, Cg, HW, output);
    return check_launch("index_shift_kernel");
}
