// cyfa_train.hip -- the layer-side operations of a training step for gfx950:
// the adjoints of the causal depthwise short convolution (ShortConvolution,
// layers/cyfa.py:138-233), of the gated RMS norm (RMSNorm, layers/cyfa.py:62-135)
// and of the gate projections and activations (layers/cyfa.py:323-326), with
// the forwards of the last two. Streaming kernels: each input is read once, sums
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
// latency of a few waves per SIMD; q's, k's and v's channels in one call (dy in
// three parts) 16.9 us, where three calls took 32. The library's depthwise convolution, as
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
    const int part_of = c < D ? c / p.split : 0, S = p.split;  // a lane's four channels are of one part
    const E* dy = static_cast<const E*>(p.dy[part_of]) + (size_t)b * T * S + (c - part_of * S);
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
            dyw[w] = t0 + w < T ? load4(dy + (size_t)(t0 + w) * S) : zero;
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
        E* dx = p.dx ? static_cast<E*>(p.dx) + (size_t)b * T * p.dx_row + c : nullptr;
        constexpr int U = 8;
        for (int tb = t0; tb < t0 + CG_RUN && tb < T; tb += U) {
            f32x4 xn[U], dn[U];  // X[tb + u] and dy[tb + u + W - 1], rows past the end read as row T - 1 and dropped
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = tb + u, j = tb + u + W - 1;
                xn[u] = load4(x + (size_t)(i < T ? i : T - 1) * p.x_row + c);
                dn[u] = load4(dy + (size_t)(j < T ? j : T - 1) * S);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int t = tb + u;
                if (t >= T) break;  // (zero times a row of X before the end may be a NaN)
                xw[W - 1] = xn[u];
                dyw[W - 1] = t + W - 1 < T ? dn[u] : zero;
                f32x4 s = zero;
#pragma unroll
                for (int w = 0; w < W; w++) {
                    s += wt[w] * dyw[W - 1 - w];
                    dw[w] += dyw[0] * xw[w];
                }
                dw[W] += dyw[0];
                if (dx) store4(dx + (size_t)t * p.dx_row, s);
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

// The sum of column e = blockIdx.x * 32 + threadIdx.x % 32 over the rows of
// part [nparts][n], for workgroups of 256 threads: eight threads per column
// each add every eighth row in order (eight loads in flight), then the eight
// in order. Valid in the first 32 threads.
__device__ __forceinline__ float column_sum(const float* part, int nparts, int n) {
    __shared__ float red[8][32];
    const int col = threadIdx.x & 31, g = threadIdx.x >> 5, e = blockIdx.x * 32 + col;
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
    if (g == 0) {
#pragma unroll
        for (int u = 1; u < 8; u++) s += red[u][col];
    }
    return s;
}

// Adds the nparts partials [W + 1][D] of conv_grad_kernel: column w D + c goes
// to dweight[c][w], column W D + c to dbias[c].
template <class E>
__global__ __launch_bounds__(256) void conv_grad_reduce_kernel(const float* part, int nparts, int D, int W, E* dweight,
                                                               E* dbias) {
    const int n = (W + 1) * D, e = blockIdx.x * 32 + (int)threadIdx.x;
    const float s = column_sum(part, nparts, n);
    if (threadIdx.x >= 32 || e >= n) return;
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

// out[e] = the column sums of part [nparts][n].
__global__ __launch_bounds__(256) void column_sum_kernel(const float* part, int nparts, int n, float* out) {
    const float s = column_sum(part, nparts, n);
    const int e = blockIdx.x * 32 + (int)threadIdx.x;
    if (threadIdx.x < 32 && e < n) out[e] = s;
}

__device__ __forceinline__ float exact_sigmoid(float x) { return 1.f / (1.f + expf(-x)); }

// The gated RMS norm of rows x [rows, D] and its adjoint, one wave per row,
// lane l holding columns 4 l + 256 j (j < J, columns past D read as zero):
//   xs  = x prescale (rounded to E; x itself for a prescale of 1), r = (mean xs^2 + eps)^-1/2
//   out = xs r weight [sigmoid(gate)]
// and, with u = dy [sigmoid(gate)],
//   dx      = prescale (r weight u - xs r^3 / D sum_i xs_i weight_i u_i)   (the cotangent of xs rounded to E first)
//   dgate   = dy xs r weight sigmoid(gate) (1 - sigmoid(gate))
//   dweight = sum over the rows of u xs r  (a partial per workgroup of p.rows_wg rows, column_sum_kernel adds them)
// The forward reads x and gate and writes out, the adjoint reads three rows and
// writes two; as the torch chain of some 25 fp32 elementwise and reduction
// launches, a gated norm of 12000 x 256 bf16 rows cost about 200 us of a
// training step. On MI355X the forward takes 6.8 us, the adjoint with its
// column sum 18 us; at 65536 rows 26 and 52 us (a copy of the bytes: 19, 32).
// Rows of an adjoint workgroup, a quarter of them per wave: few while that
// leaves compute units idle, many where the partials would add up. us of the
// adjoint with its column sum at 8 / 16 / 32 / 64 rows (gated bf16 rows of 256):
// 2000 rows 8.1 / 9.1 / 11.9 / 17, 8192 14.6 / 12.2 / 12.1 / 17.7, 12000 20.7 /
// 17.2 / 18.6 / 20.6, 32768 44 / 33 / 29.3 / 29.7, 65536 79 / 58 / 50 / 47.
int norm_grad_rows(long long rows) { return rows >= 32768 ? 32 : rows >= 8192 ? 16 : 8; }

// xs, sigmoid(gate) (ones without a gate) and r of a row from its loaded values.
template <class E, int J>
__device__ __forceinline__ void norm_row(const NormTrainParams& p, f32x4 (&xs)[J], f32x4 (&sg)[J], float& rs) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < J; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (p.prescale != 1.f) xs[j][i] = (float)(E)(xs[j][i] * p.prescale);
            ss = fmaf(xs[j][i], xs[j][i], ss);
            sg[j][i] = p.gate ? exact_sigmoid(sg[j][i]) : 1.f;
        }
    rs = rsqrtf(wave_sum(ss) / (float)p.D + p.eps);
}

// Row `row`'s columns of this lane, zero past D and past the last row: read
// from the last row and columns there, and dropped (no branch among the loads,
// at which the compiler would wait for those in flight).
template <class E, int J>
__device__ __forceinline__ void norm_load(const void* x, long long row, const NormTrainParams& p, int lane, f32x4 (&v)[J]) {
    const E* src = static_cast<const E*>(x) + (size_t)(row < p.rows ? row : p.rows - 1) * p.D;
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int d = 4 * lane + 256 * j;
        v[j] = load4(src + (d < p.D ? d : p.D - 4));
        if (row >= p.rows || d >= p.D) v[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
}

template <int J>
__device__ __forceinline__ void norm_weight(const NormTrainParams& p, int lane, f32x4 (&w)[J]) {
#pragma unroll
    for (int j = 0; j < J; j++)
        w[j] = 4 * lane + 256 * j < p.D ? load4(p.weight + 4 * lane + 256 * j) : f32x4{0.f, 0.f, 0.f, 0.f};
}

template <class E, int J>
__global__ __launch_bounds__(256) void norm_train_kernel(NormTrainParams p) {
    const int lane = threadIdx.x & 63;
    const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= p.rows) return;
    f32x4 w[J], xs[J], sg[J];
    norm_load<E, J>(p.x, row, p, lane, xs);
    norm_load<E, J>(p.gate ? p.gate : p.x, row, p, lane, sg);
    norm_weight<J>(p, lane, w);
    float rs;
    norm_row<E, J>(p, xs, sg, rs);
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int d = 4 * lane + 256 * j;
        if (d < p.D) store4(static_cast<E*>(p.out) + (size_t)row * p.D + d, xs[j] * rs * w[j] * sg[j]);
    }
}

template <class E, int J>
__global__ __launch_bounds__(256) void norm_grad_kernel(NormTrainParams p) {
    __shared__ __align__(16) float red[4][J * 256];
    constexpr int RB = J <= 4 ? 2 : 1;  // rows whose loads are in flight together
    const int rpw = p.rows_wg / 4;      // rows of a wave, 2, 4 or 8
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    f32x4 w[J], dw[J];
    norm_weight<J>(p, lane, w);
#pragma unroll
    for (int j = 0; j < J; j++) dw[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < rpw; k += RB) {
        const long long row0 = (long long)blockIdx.x * p.rows_wg + rpw * wv + k;
        if (row0 >= p.rows) break;
        f32x4 xs[RB][J], sg[RB][J], dy[RB][J];
#pragma unroll
        for (int r = 0; r < RB; r++) {
            norm_load<E, J>(p.x, row0 + r, p, lane, xs[r]);
            norm_load<E, J>(p.gate ? p.gate : p.x, row0 + r, p, lane, sg[r]);
            norm_load<E, J>(p.dy, row0 + r, p, lane, dy[r]);
        }
#pragma unroll
        for (int r = 0; r < RB; r++) {
            float rs, sum = 0.f;
            norm_row<E, J>(p, xs[r], sg[r], rs);
#pragma unroll
            for (int j = 0; j < J; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) sum = fmaf(xs[r][j][i] * w[j][i], dy[r][j][i] * sg[r][j][i], sum);
            const float cr = rs * rs * rs * wave_sum(sum) / (float)p.D;
            const size_t base = (size_t)(row0 + r) * p.D;
            if (row0 + r >= p.rows) break;  // (a zero row's r is infinite where eps is zero)
#pragma unroll
            for (int j = 0; j < J; j++) {
                const int d = 4 * lane + 256 * j;
                const f32x4 u = dy[r][j] * sg[r][j];
                dw[j] += u * xs[r][j] * rs;
                if (d < p.D) {
                    if (p.dx) {
                        f32x4 dxs = w[j] * u * rs - xs[r][j] * cr;
                        if (p.prescale != 1.f) {
#pragma unroll
                            for (int i = 0; i < 4; i++) dxs[i] = (float)(E)dxs[i] * p.prescale;
                        }
                        store4(static_cast<E*>(p.dx) + base + d, dxs);
                    }
                    if (p.dgate) store4(static_cast<E*>(p.dgate) + base + d, u * xs[r][j] * rs * w[j] * (1.f - sg[r][j]));
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < J; j++) *reinterpret_cast<f32x4*>(&red[wv][4 * lane + 256 * j]) = dw[j];
    __syncthreads();
    for (int d = threadIdx.x; d < p.D; d += 256)
        p.part[(size_t)blockIdx.x * p.D + d] = (red[0][d] + red[1][d]) + (red[2][d] + red[3][d]);
}

template <class E, int J>
int launch_norm_train_as(NormTrainParams p, bool grad, hipStream_t stream) {
    const dim3 block(256);
    if (!grad) {
        hipLaunchKernelGGL((norm_train_kernel<E, J>), dim3((unsigned)((p.rows + 3) / 4)), block, 0, stream, p);
        return 0;
    }
    p.rows_wg = norm_grad_rows(p.rows);
    const unsigned blocks = (unsigned)((p.rows + p.rows_wg - 1) / p.rows_wg);
    hipLaunchKernelGGL((norm_grad_kernel<E, J>), dim3(blocks), block, 0, stream, p);
    if (p.dweight)
        hipLaunchKernelGGL(column_sum_kernel, dim3((p.D + 31) / 32), block, 0, stream, p.part, (int)blocks, p.D, p.dweight);
    return 0;
}

template <class E>
int launch_norm_train_j(const NormTrainParams& p, bool grad, hipStream_t stream) {
    const int j = (p.D + 255) / 256;
    return j <= 1   ? launch_norm_train_as<E, 1>(p, grad, stream)
           : j <= 2 ? launch_norm_train_as<E, 2>(p, grad, stream)
           : j <= 4 ? launch_norm_train_as<E, 4>(p, grad, stream)
                    : launch_norm_train_as<E, 8>(p, grad, stream);
}


// ---- the gates of a training step ----
//
// a = x W_a^T, b = x W_b^T + c_b, d = x W_d^T + c_d (each rounded to E), and
//   g = -exp(A_log) softplus(a + dt_bias), beta = sigmoid(b), delta = sigmoid(d)
// for H <= GATES_MAX_H heads: projections so narrow that a library GEMM per
// projection and direction spends 7 (forward), 9 (dx) and 39 us (weight
// gradient) on 3000 x 1024 bf16 tokens, where x is 6 MB, with some 20 small
// elementwise and reduction launches around them: about 240 us of a training
// step in all. Here x is read once forward (7.2 us) and once backward (4.9 us
// for the activations, 13.9 for dx and dW, 4.6 + 4.5 for the sums of their
// partials).

// softplus as F.softplus forms it (the identity above 20), and its derivative.
__device__ __forceinline__ float softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }
__device__ __forceinline__ float softplus_grad(float x) { return x > 20.f ? 1.f : exact_sigmoid(x); }

// Row n of [W_a; W_b; W_d] (H rows each).
template <class E>
__device__ __forceinline__ const E* gates_weight(const GatesTrainParams& p, int n) {
    const void* w = n < p.H ? p.wa : n < 2 * p.H ? p.wb : p.wd;
    return static_cast<const E*>(w) + (size_t)(n % p.H) * p.K;
}

// Forward: a workgroup takes 16 rows of x, its four waves a quarter of the
// columns each (8 columns per lane and step of 32), on the matrix cores: bf16
// operands on v_mfma_f32_16x16x32_bf16, fp32 ones as two v_mfma_f32_16x16x4_f32
// steps per four columns (fp32 products and sums). Lane (lr, lg) loads 8
// consecutive columns of row lr of x and of weight rows lr, lr + 16; the waves'
// partial sums meet in LDS, in wave order, where the activations are formed.
template <class E, int NT>
__global__ __launch_bounds__(256) void gates_train_kernel(GatesTrainParams p) {
    typedef E ex8 __attribute__((ext_vector_type(8), aligned(16)));
    __shared__ float part[4][16][16 * NT + 1];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lg = lane >> 4;
    const int H = p.H, N = 3 * H, r0 = blockIdx.x * 16;
    const int steps = (p.K + 31) / 32, per = (steps + 3) / 4, s0 = wv * per, s1 = min(s0 + per, steps);
    const E* x = static_cast<const E*>(p.x) + (size_t)min(r0 + lr, p.rows - 1) * p.K;
    const E* w[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) w[t] = gates_weight<E>(p, min(16 * t + lr, N - 1));
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int U = 4;  // steps whose loads are in flight together
    for (int s = s0; s < s1; s += U) {
        ex8 xv[U], wvv[U][NT];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = 32 * (s + u) + 8 * lg;
            const bool live = s + u < s1 && k < p.K;  // K is a multiple of 8
            const int kk = live ? k : 0;
            xv[u] = *reinterpret_cast<const ex8*>(x + kk);
#pragma unroll
            for (int t = 0; t < NT; t++) wvv[u][t] = *reinterpret_cast<const ex8*>(w[t] + kk);
            if (!live) {
#pragma unroll
                for (int e = 0; e < 8; e++) xv[u][e] = (E)0.f;
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int e = 0; e < 8; e++) wvv[u][t][e] = (E)0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if constexpr (sizeof(E) == 2) {
                    acc[t] = mfma_bf16(__builtin_bit_cast(bf16x8, xv[u]), __builtin_bit_cast(bf16x8, wvv[u][t]), acc[t]);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[u][e], wvv[u][t][e], acc[t], 0, 0, 0);
                }
            }
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) part[wv][4 * lg + i][16 * t + lr] = acc[t][i];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * N; e += 256) {
        const int r = e / N, n = e % N, h = n % H, kind = n / H;
        const long long row = r0 + r;
        if (row >= p.rows) break;
        float v = (part[0][r][n] + part[1][r][n]) + (part[2][r][n] + part[3][r][n]);
        if (kind) v += (float)static_cast<const E*>(kind == 1 ? p.bb : p.bd)[h];
        const E pre = (E)v;
        static_cast<E*>(p.abd)[row * N + n] = pre;
        v = (float)pre;
        float* dst = kind == 0 ? p.g : kind == 1 ? p.beta : p.delta;
        dst[row * H + h] = kind == 0 ? -expf(p.A_log[h]) * softplus(v + p.dt_bias[h]) : exact_sigmoid(v);
    }
}

// Adjoint of the activations, one row per lane, 64 rows per workgroup: dabd
// [rows, 3H] rounded to E (the projections' cotangents) as fp32, and per
// workgroup the sums over its rows of da (dt_bias), of dg g (A_log), and of
// the rounded db and dd (the biases), each H wide.
__global__ __launch_bounds__(256) void gates_grad_act_kernel(GatesTrainParams p, int bf16) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, H = p.H, N = 3 * H;
    const long long row = (long long)blockIdx.x * 64 + lane;
    const bool live = row < p.rows;
    const long long rr = live ? row : 0;
    const auto rnd = [&](float v) { return bf16 ? bf16_round(v) : v; };
    const auto pre = [&](int n) {
        return bf16 ? (float)static_cast<const bf16_t*>(p.abd)[rr * N + n] : static_cast<const float*>(p.abd)[rr * N + n];
    };
    for (int h = wv; h < H; h += 4) {
        const float z = pre(h) + p.dt_bias[h], ea = -expf(p.A_log[h]);
        const float dg = live ? p.dg[rr * H + h] : 0.f;
        const float be = exact_sigmoid(pre(H + h)), de = exact_sigmoid(pre(2 * H + h));
        const float da = dg * ea * softplus_grad(z);
        const float db = rnd(live ? p.dbeta[rr * H + h] * be * (1.f - be) : 0.f);
        const float dd = rnd(live ? p.ddelta[rr * H + h] * de * (1.f - de) : 0.f);
        if (live) {
            p.dabd[rr * N + h] = rnd(da);
            p.dabd[rr * N + H + h] = db;
            p.dabd[rr * N + 2 * H + h] = dd;
        }
        float* part = p.part_sums + (size_t)blockIdx.x * 4 * H + h;
        const float sa = wave_sum(da), sl = wave_sum(dg * ea * softplus(z)), sb = wave_sum(db), sd = wave_sum(dd);
        if (lane == 0) {
            part[0] = sa;
            part[H] = sl;
            part[2 * H] = sb;
            part[3 * H] = sd;
        }
    }
}

// Adjoint of the projections: dx = da W_a + db W_b (the clock branch passes no
// gradient into x) and dW[n] = sum over the rows of dabd[n] x. A lane holds
// four columns, a workgroup 256 columns and p.rows_wg rows, a wave every
// fourth of them, the weights and dW in registers (HM: H rounded up to 4 or
// 8); the waves' parts of dW are added in LDS, in wave order, into one partial
// per workgroup.
// Rows of a workgroup: 32, and 128 where that still leaves 256 workgroups per
// 256 columns, so that the partials, 3 H floats per column and workgroup, stay
// below x itself (65536 rows of 2048 bf16 columns, 8 heads: 101 MB, where 32
// rows made 403 MB and a step of the gates held 687 MB, 544 as torch
// operations; with 128 it holds 385 and takes 558 us, 798 before).
int gates_rows(int rows) { return rows >= 32768 ? 128 : 32; }

template <class E, int HM>
__global__ __launch_bounds__(256) void gates_grad_kernel(GatesTrainParams p) {
    __shared__ __align__(16) float red[4][4][256];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int H = p.H, N = 3 * H, K = p.K, k = blockIdx.x * 256 + 4 * lane;
    const bool live = k < K;
    const int kk = live ? k : 0;
    f32x4 w[2 * HM], dw[3 * HM];
#pragma unroll
    for (int n = 0; n < 2 * HM; n++) {
        const int h = n % HM, kind = n / HM;
        w[n] = load4(gates_weight<E>(p, h < H ? kind * H + h : 0) + kk);
    }
#pragma unroll
    for (int n = 0; n < 3 * HM; n++) dw[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int row0 = blockIdx.y * p.rows_wg;
    for (int i = 0; i < p.rows_wg && row0 + i < p.rows; i += 8) {  // two rows of this wave at a time
        f32x4 x[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int row = min(row0 + i + 4 * u + wv, p.rows - 1);
            x[u] = load4(static_cast<const E*>(p.x) + (size_t)row * K + kk);
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int row = row0 + i + 4 * u + wv;
            if (row < p.rows) {  // uniform over the wave, as dabd's addresses are
                const float* da = p.dabd + (size_t)row * N;
                f32x4 dx = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int n = 0; n < 3 * HM; n++) {
                    const int h = n % HM, kind = n / HM;
                    const float c = h < H ? da[kind * H + h] : 0.f;
                    if (kind < 2) dx += w[n] * c;
                    dw[n] += x[u] * c;
                }
                if (live && p.dx) store4(static_cast<E*>(p.dx) + (size_t)row * K + k, dx);
            }
        }
    }
    float* part = p.part_w + (size_t)blockIdx.y * N * K;
    const int col = blockIdx.x * 256 + threadIdx.x;
#pragma unroll
    for (int n0 = 0; n0 < 3 * HM; n0 += 4) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; j++) *reinterpret_cast<f32x4*>(&red[wv][j][4 * lane]) = dw[n0 + j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int h = (n0 + j) % HM, kind = (n0 + j) / HM, e = threadIdx.x;
            if (h < H && col < K)
                part[(size_t)(kind * H + h) * K + col] = (red[0][j][e] + red[1][j][e]) + (red[2][j][e] + red[3][j][e]);
        }
    }
}

// Adds the partials of gates_grad_kernel into dW_a, dW_b and dW_d.
template <class E>
__global__ __launch_bounds__(256) void gates_grad_reduce_kernel(GatesTrainParams p, int nparts) {
    const int n = 3 * p.H * p.K, e = blockIdx.x * 32 + (int)threadIdx.x;
    const float s = column_sum(p.part_w, nparts, n);
    if (threadIdx.x >= 32 || e >= n) return;
    const int hk = p.H * p.K, kind = e / hk;
    static_cast<E*>(kind == 0 ? p.dwa : kind == 1 ? p.dwb : p.dwd)[e % hk] = (E)s;
}

// Adds the partial sums of gates_grad_act_kernel: dt_bias, A_log (fp32), then
// the biases (E).
template <class E>
__global__ __launch_bounds__(256) void gates_grad_sums_kernel(GatesTrainParams p, int nparts) {
    const int n = 4 * p.H, e = blockIdx.x * 32 + (int)threadIdx.x;
    const float s = column_sum(p.part_sums, nparts, n);
    if (threadIdx.x >= 32 || e >= n) return;
    const int kind = e / p.H, h = e % p.H;
    if (kind < 2)
        (kind == 0 ? p.ddt_bias : p.dA_log)[h] = s;
    else
        static_cast<E*>(kind == 2 ? p.dbb : p.dbd)[h] = (E)s;
}

template <class E>
int launch_gates_train_as(const GatesTrainParams& p, hipStream_t stream) {
    const dim3 grid((unsigned)((p.rows + 15) / 16)), block(256);
    if (3 * p.H <= 16)
        hipLaunchKernelGGL((gates_train_kernel<E, 1>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((gates_train_kernel<E, 2>), grid, block, 0, stream, p);
    return 0;
}

template <class E>
int launch_gates_grad_as(GatesTrainParams p, hipStream_t stream) {
    const dim3 block(256);
    p.rows_wg = gates_rows(p.rows);
    const int acts = (p.rows + 63) / 64, parts = (p.rows + p.rows_wg - 1) / p.rows_wg;
    hipLaunchKernelGGL(gates_grad_act_kernel, dim3(acts), block, 0, stream, p, sizeof(E) == 2 ? 1 : 0);
    const dim3 grid((p.K + 255) / 256, parts);
    if (p.H <= 4)
        hipLaunchKernelGGL((gates_grad_kernel<E, 4>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((gates_grad_kernel<E, 8>), grid, block, 0, stream, p);
    hipLaunchKernelGGL(gates_grad_reduce_kernel<E>, dim3((3 * p.H * p.K + 31) / 32), block, 0, stream, p, parts);
    hipLaunchKernelGGL(gates_grad_sums_kernel<E>, dim3((4 * p.H + 31) / 32), block, 0, stream, p, acts);
    return 0;
}

}  // namespace

size_t gates_grad_workspace_bytes(int rows, int K, int H) {
    const int n = gates_rows(rows);
    return ((size_t)rows * 3 * H + (size_t)((rows + 63) / 64) * 4 * H + (size_t)((rows + n - 1) / n) * 3 * H * K) *
           sizeof(float);
}

// Splits the adjoint's workspace (gates_grad_workspace_bytes) into its parts.
static void gates_grad_workspace(GatesTrainParams& p, float* base) {
    p.dabd = base;
    p.part_sums = p.dabd + (size_t)p.rows * 3 * p.H;
    p.part_w = p.part_sums + (size_t)((p.rows + 63) / 64) * 4 * p.H;
}

int launch_gates_train(const GatesTrainParams& p_in, bool bf16, bool grad, float* workspace, hipStream_t stream) {
    GatesTrainParams p = p_in;
    if (p.rows < 1 || p.rows > 32 * 65535 || p.K < 8 || p.K % 8 || p.H < 1 || p.H > GATES_MAX_H ||
        (long long)3 * p.H * p.K >= 1ll << 31)
        return -1;
    if (!grad) return bf16 ? launch_gates_train_as<bf16_t>(p, stream) : launch_gates_train_as<float>(p, stream);
    gates_grad_workspace(p, workspace);
    return bf16 ? launch_gates_grad_as<bf16_t>(p, stream) : launch_gates_grad_as<float>(p, stream);
}

size_t norm_grad_workspace_bytes(long long rows, int D) {
    const int n = norm_grad_rows(rows);
    return (size_t)((rows + n - 1) / n) * D * sizeof(float);
}

int launch_norm_train(const NormTrainParams& p, bool bf16, bool grad, hipStream_t stream) {
    if (p.rows < 1 || p.rows > NORM_TRAIN_MAX_ROWS || p.D < 4 || p.D % 4 || p.D > NORM_TRAIN_MAX_D) return -1;
    return bf16 ? launch_norm_train_j<bf16_t>(p, grad, stream) : launch_norm_train_j<float>(p, grad, stream);
}

size_t conv_grad_workspace_bytes(int B, int T, int D, int W) {
    return (size_t)B * ((T + CG_TOKENS - 1) / CG_TOKENS) * (W + 1) * D * sizeof(float);
}

int launch_conv_grad(const ConvGradParams& p, bool bf16, hipStream_t stream) {
    if (p.B < 1 || p.B > 65535 || p.T < 1 || (p.T + CG_TOKENS - 1) / CG_TOKENS > 65535 || p.D < 4 || p.D % 4) return -1;
    return bf16 ? launch_conv_grad_as<bf16_t>(p, stream) : launch_conv_grad_as<float>(p, stream);
}

}  // namespace cyfa
