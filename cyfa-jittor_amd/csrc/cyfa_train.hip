// cyfa_train.hip -- the layer-side adjoints of a training step for gfx950: the
// gradients of the causal depthwise short convolution (ShortConvolution,
// layers/cyfa.py:138-233). Streaming kernels: each input is read once, sums
// over tokens accumulate in fp32 and partial sums are added in a fixed order,
// so that two backward passes give the same bits.
#include "cyfa_device.h"
#include "cyfa_internal.h"

namespace cyfa {

namespace {

// Four consecutive elements of bf16 or fp32 rows, widened to fp32.
template <class E>
struct Vec4 {
    typedef E type __attribute__((ext_vector_type(4)));
};

template <class E>
__device__ __forceinline__ f32x4 load4(const E* p) {
    const typename Vec4<E>::type v = *reinterpret_cast<const typename Vec4<E>::type*>(p);
    return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

template <class E>
__device__ __forceinline__ void store4(E* p, f32x4 v) {
    *reinterpret_cast<typename Vec4<E>::type*>(p) = typename Vec4<E>::type{(E)v[0], (E)v[1], (E)v[2], (E)v[3]};
}

// Adjoint of y[b, t, c] = bias[c] + sum_{w < W} weight[c, w] X[b, t + w - (W - 1), c]
// (X = x, before the start the cache or zero):
//   dx[b, i, c]   = sum_w weight[c, w] dy[b, i + W - 1 - w, c]   (i < 0: the cache's rows)
//   dweight[c, w] = sum_{b, t} dy[b, t, c] X[b, t + w - (W - 1), c],  dbias[c] = sum dy
// A lane takes four channels, a wave a run of CG_RUN tokens, sliding the last
// W - 1 rows of X and the next W - 1 rows of dy through registers, the next
// eight rows of both in flight; the workgroup's four waves take neighbouring
// runs of the same 256 channels and add their parts of dweight and dbias in
// LDS, in wave order, into one partial per workgroup (conv_grad_reduce_kernel
// adds the partials). x and dy are read once, dx written once (the partials
// are W + 1 floats per channel and 64 tokens), so a large call is bound by HBM;
// 2 x 1500 tokens of 1024 bf16 channels (18 MB) take 11.2 + 3.9 us on MI355X,
// latency of a few waves per SIMD. The library's depthwise convolution, as
// F.conv1d reaches it, took about 320 us forward and backward for such a
// tensor: transposes to channel-major, im2col, a GEMM per direction.
constexpr int CG_RUN = 16, CG_TOKENS = 4 * CG_RUN, CG_CHANNELS = 256;

template <class E, int W>
__global__ __launch_bounds__(256) void conv_grad_kernel(ConvGradParams p) {
    __shared__ __align__(16) float red[4][W + 1][CG_CHANNELS];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, b = blockIdx.y;
    const int c = blockIdx.x * CG_CHANNELS + 4 * lane, t0 = blockIdx.z * CG_TOKENS + wv * CG_RUN;
    const int T = p.T, D = p.D;
    const E* x = static_cast<const E*>(p.x) + (size_t)b * T * p.x_row;
    const E* dy = static_cast<const E*>(p.dy) + (size_t)b * T * D;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 dw[W + 1];  // dw[W]: the bias
#pragma unroll
    for (int w = 0; w <= W; w++) dw[w] = zero;
    if (c < D && t0 < T) {
        f32x4 wt[W];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int w = 0; w < W; w++) wt[w][i] = (float)static_cast<const E*>(p.weight)[(size_t)(c + i) * W + w];
        const auto x_at = [&](int i) {  // X[i]; zero outside
            if (i < 0)
                return p.cache ? load4(static_cast<const E*>(p.cache) + (size_t)b * p.cache_batch +
                                       (size_t)(W - 1 + i) * p.cache_row + c)
                               : zero;
            return load4(x + (size_t)i * p.x_row + c);
        };
        f32x4 xw[W], dyw[W];  // X[t - (W - 1) .. t], dy[t .. t + W - 1]
#pragma unroll
        for (int w = 0; w < W - 1; w++) {
            xw[w] = x_at(t0 + w - (W - 1));
            dyw[w] = t0 + w < T ? load4(dy + (size_t)(t0 + w) * D + c) : zero;
        }
        if (t0 == 0 && p.dcache) {  // X[j - (W - 1)] feeds y[0 .. j]
            E* dc = static_cast<E*>(p.dcache) + (size_t)b * (W - 1) * D + c;
#pragma unroll
            for (int j = 0; j < W - 1; j++) {
                f32x4 s = zero;
#pragma unroll
                for (int w = 0; w <= j; w++) s += wt[w] * dyw[j - w];
                store4(dc + (size_t)j * D, s);
            }
        }
        E* dx = p.dx ? static_cast<E*>(p.dx) + (size_t)b * T * D + c : nullptr;
        constexpr int U = 8;
        for (int tb = t0; tb < t0 + CG_RUN && tb < T; tb += U) {
            f32x4 xn[U], dn[U];  // X[tb + u] and dy[tb + u + W - 1], rows past the end read as row T - 1 and dropped
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = tb + u, j = tb + u + W - 1;
                xn[u] = load4(x + (size_t)(i < T ? i : T - 1) * p.x_row + c);
                dn[u] = load4(dy + (size_t)(j < T ? j : T - 1) * D + c);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int t = tb + u;
                xw[W - 1] = t < T ? xn[u] : zero;
                dyw[W - 1] = t + W - 1 < T ? dn[u] : zero;
                f32x4 s = zero;
#pragma unroll
                for (int w = 0; w < W; w++) {
                    s += wt[w] * dyw[W - 1 - w];
                    dw[w] += dyw[0] * xw[w];
                }
                dw[W] += dyw[0];
                if (dx && t < T) store4(dx + (size_t)t * D, s);
#pragma unroll
                for (int w = 0; w < W - 1; w++) {
                    xw[w] = xw[w + 1];
                    dyw[w] = dyw[w + 1];
                }
            }
        }
    }
#pragma unroll
    for (int w = 0; w <= W; w++) *reinterpret_cast<f32x4*>(&red[wv][w][4 * lane]) = dw[w];
    __syncthreads();
    float* part = p.part + ((size_t)b * gridDim.z + blockIdx.z) * (W + 1) * D;
    const int ch = blockIdx.x * CG_CHANNELS + threadIdx.x;
    if (ch >= D) return;
#pragma unroll
    for (int w = 0; w <= W; w++) {
        const int e = threadIdx.x;
        part[(size_t)w * D + ch] = (red[0][w][e] + red[1][w][e]) + (red[2][w][e] + red[3][w][e]);
    }
}

// Adds the nparts partials [W + 1][D] of conv_grad_kernel: 32 columns per
// workgroup, eight threads per column each adding every eighth partial in
// order (eight loads in flight), then the eight in order. Column w D + c goes
// to dweight[c][w], column W D + c to dbias[c].
template <class E>
__global__ __launch_bounds__(256) void conv_grad_reduce_kernel(const float* part, int nparts, int D, int W, E* dweight,
                                                               E* dbias) {
    __shared__ float red[8][32];
    const int n = (W + 1) * D, col = threadIdx.x & 31, g = threadIdx.x >> 5, e = blockIdx.x * 32 + col;
    float s = 0.f;
    if (e < n) {
        int i = g;
        for (; i + 56 < nparts; i += 64) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = part[(size_t)(i + 8 * u) * n + e];
#pragma unroll
            for (int u = 0; u < 8; u++) s += v[u];
        }
        for (; i < nparts; i += 8) s += part[(size_t)i * n + e];
    }
    red[g][col] = s;
    __syncthreads();
    if (g != 0 || e >= n) return;
#pragma unroll
    for (int u = 1; u < 8; u++) s += red[u][col];
    const int w = e / D, c = e % D;
    if (w < W) {
        if (dweight) dweight[(size_t)c * W + w] = (E)s;
    } else if (dbias) {
        dbias[c] = (E)s;
    }
}

template <class E>
int launch_conv_grad_as(const ConvGradParams& p, hipStream_t stream) {
    const dim3 grid((p.D + CG_CHANNELS - 1) / CG_CHANNELS, p.B, (p.T + CG_TOKENS - 1) / CG_TOKENS), block(256);
    switch (p.W) {
        case 2: hipLaunchKernelGGL((conv_grad_kernel<E, 2>), grid, block, 0, stream, p); break;
        case 3: hipLaunchKernelGGL((conv_grad_kernel<E, 3>), grid, block, 0, stream, p); break;
        case 4: hipLaunchKernelGGL((conv_grad_kernel<E, 4>), grid, block, 0, stream, p); break;
        default: return -1;
    }
    const int n = (p.W + 1) * p.D;
    hipLaunchKernelGGL(conv_grad_reduce_kernel<E>, dim3((n + 31) / 32), block, 0, stream, p.part, (int)(grid.y * grid.z),
                       p.D, p.W, static_cast<E*>(p.dweight), static_cast<E*>(p.dbias));
    return 0;
}

}  // namespace

size_t conv_grad_workspace_bytes(int B, int T, int D, int W) {
    return (size_t)B * ((T + CG_TOKENS - 1) / CG_TOKENS) * (W + 1) * D * sizeof(float);
}

int launch_conv_grad(const ConvGradParams& p, bool bf16, hipStream_t stream) {
    if (p.B < 1 || p.B > 65535 || p.T < 1 || (p.T + CG_TOKENS - 1) / CG_TOKENS > 65535 || p.D < 4 || p.D % 4) return -1;
    return bf16 ? launch_conv_grad_as<bf16_t>(p, stream) : launch_conv_grad_as<float>(p, stream);
}

}  // namespace cyfa
