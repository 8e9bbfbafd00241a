// cyfa_backward.hip -- the backward pass of the chunkwise CyFA op.
//
// Replaces the autograd adjoints chunk_cyfa (ops/chunk.py:164-353) is built
// from: ScalarAttention.grad / scalar_grad for both ScalarGatedLA passes
// (ops/chunk.py:51-71, ops/chunk_bwd.py:1008-1041: state_backward,
// query_key_adjoint, value_adjoint), the slot-readout adjoint of
// FirstReadout*.grad (ops/chunk_readout.py:13-621, 776-786, 976-988),
// PhaseWrite.grad and ClockScan.grad (ops/utils.py:297-299, 589-641,
// 704-754), HeadRMSNorm.grad (ops/qk_norm.py:241-289) and the gradient of
// table = readout @ Phi (ops/chunk.py:281).
//
// The forward is recomputed from the inputs without the roundings of the bf16
// forward (the general path's clock, write vector and readout; the states before
// every 64-token chunk of both passes and the pass-1 output from the kernels
// below), and every adjoint accumulates in fp32 or double. fp32 calls are fp32
// throughout: the gradients of the op's exact arithmetic up to fp32 rounding. In
// bf16 calls the products take operands of about 16 mantissa bits (two bf16
// parts) and the stored states and state cotangents are bf16, as the reference
// stores them; those states decide the gradients' error. Per pass (o = SGLA(q, k, v, g, S0, scale),
// in-chunk cumulative log-decay G):
//   D_n  = e^{G_last} D_{n+1} + scale sum_t e^{G_t} q_t (x) dO_t      (state cotangent, reverse over chunks)
//   dq_t = scale (e^{G_t} S_n dO_t + sum_{s<=t} e^{G_t-G_s} (dO_t.v_s) k_s)
//   dk_s = scale sum_{t>=s} e^{G_t-G_s} (dO_t.v_s) q_t + e^{G_last-G_s} D_{n+1} v_s
//   dv_s = scale sum_{t>=s} e^{G_t-G_s} (q_t.k_s) dO_t + e^{G_last-G_s} D_{n+1}^T k_s
//   dL/dG_t = q_t.dq_t - k_t.dk_t + [t = last] <D_{n+1}, S_{n+1}>,  dg = in-chunk reverse cumsum
// where q_t.dq_t = o_t.dO_t (dq_t scale^-1 is what o_t's rows contract with)
// and k_t.dk_t = v_t.dv_t, so that both passes' terms come from the narrow
// rows between them: z.dz and u.du in the readout adjoint (a rotation keeps the
// dot products raw.draw and weights.dweights), and w.(dw_1 + dw_2) = beta
// dbeta.
// The states and their cotangents are one sweep per (state tile, b, h) that
// keeps its tile in registers; outputs and the rows' cotangents are then
// chunk-parallel, one workgroup per (chunk, h, b), with no reduction across
// workgroups. The readout adjoint runs per block of rows (z = U(lam) raw,
// softmax of table z, u = table^T p, weights = U(-lam) u) with the head's
// table and this workgroup's share of the table cotangent on chip (up to 128
// slots; above, as tile GEMMs that stream the table); partial sums (table,
// norm weights, per-tile boundary terms) are added in a fixed order, so the
// result does not depend on scheduling. Every product runs on the matrix
// cores: with bf16 operands the scans', chunk kernels' and the recomputed
// readout's with every fp32 operand split into two bf16 parts (about 16
// mantissa bits); with fp32 operands as fp32 products (v_mfma_f32_16x16x4_f32),
// exact to fp32 rounding.
#include <cmath>
#include <type_traits>

#include "cyfa_device.h"
#include "cyfa_internal.h"

namespace cyfa {

namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int BC = 64;           // chunk length of the recompute and the sweeps
constexpr int BW_MAX_D = 1024;   // largest K and V
constexpr int BW_TILE = 32;      // state columns per scan workgroup
constexpr double kTwoPiBw = 6.283185307179586;

// Whole-wave sum and max in every lane, on DPP moves and v_readlane (the
// fixed order of wave_sum / wave_max); every call site has the whole wave
// active. (With __shfl_xor each step was an LDS round trip.)
__device__ __forceinline__ float bw_wave_sum(float x) { return wave_sum<64>(x); }

__device__ __forceinline__ float bw_wave_max(float x) { return wave_max<64>(x); }

template <bool BF>
__device__ __forceinline__ float bw_ld(const void* p, size_t i) {
    if constexpr (BF)
        return (float)reinterpret_cast<const bf16_t*>(p)[i];
    else
        return reinterpret_cast<const float*>(p)[i];
}

template <bool BF>
__device__ __forceinline__ void bw_st(void* p, size_t i, float v) {
    if constexpr (BF)
        reinterpret_cast<bf16_t*>(p)[i] = (bf16_t)v;
    else
        reinterpret_cast<float*>(p)[i] = v;
}

// The in-chunk inclusive cumsum G of the natural-log gate over chunk n of
// (b, h), lane = token (tokens past T add zero); one wave.
// Inclusive sum over the wave's 64 lanes on DPP moves: shifts by 1, 2, 4 and
// 8 within rows of 16, then row 15's sum broadcast into the next row, and row
// 31's into the upper half (every lane active). (__shfl_up made each step an
// LDS round trip on the scans' serial path.)
template <int CTRL>
__device__ __forceinline__ float bw_dpp_shift(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float bw_wave_scan(float x) {
    x += bw_dpp_shift<0x111>(x);
    x += bw_dpp_shift<0x112>(x);
    x += bw_dpp_shift<0x114>(x);
    x += bw_dpp_shift<0x118>(x);
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x142, 0xA, 0xF, false));
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x143, 0xC, 0xF, false));
    return x;
}

__device__ __forceinline__ float chunk_gam(const float* g, int b, int h, int T, int H, int n, int lane) {
    const int t = n * BC + lane;
    return bw_wave_scan(t < T ? g[((size_t)b * T + t) * H + h] : 0.f);
}

// Rows of x [B, T, H, D] into head-major fp32 [B*H, Tp, D]: with a norm
// weight the normalised row x rs w (ops/qk_norm.py:206-233, unrounded) and rs
// per row; without, x itself; x == nullptr or t >= T gives zeros. One wave per row.
// O: the rows' element type (bf16_t only without w: a bf16 x's layout change).
template <bool BF, class O = float>
__global__ __launch_bounds__(256) void bw_rows_kernel(const void* x, const float* w, float eps, int B, int T, int Tp,
                                                      int H, int D, O* out, float* rs_out) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= B * H * Tp) return;
    const int t = row % Tp, bh = row / Tp, b = bh / H, h = bh % H;
    O* dst = out + (size_t)row * D;
    if (!x || t >= T) {
        for (int i = lane; i < D; i += 64) dst[i] = (O)0.f;
        if (rs_out && lane == 0) rs_out[row] = 0.f;
        return;
    }
    const size_t src = (((size_t)b * T + t) * H + h) * D;
    if (D == 256 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0) {
        // the tuned head size (16-byte aligned rows): four consecutive
        // elements per lane, one pass over x
        float v[4];
        if constexpr (BF) {
            const bf16x4 xv = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16_t*>(x) + src + 4 * lane);
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = (float)xv[e];
        } else {
            const float4 xv = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(x) + src + 4 * lane);
            v[0] = xv.x, v[1] = xv.y, v[2] = xv.z, v[3] = xv.w;
        }
        float4 o = {v[0], v[1], v[2], v[3]};
        if (w) {
            float ss = 0.f;
#pragma unroll
            for (int e = 0; e < 4; e++) ss = fmaf(v[e], v[e], ss);
            const float rs = rsqrtf(bw_wave_sum(ss) / (float)D + eps);
            const float4 wv = *reinterpret_cast<const float4*>(w + 4 * lane);
            o = float4{v[0] * rs * wv.x, v[1] * rs * wv.y, v[2] * rs * wv.z, v[3] * rs * wv.w};
            if (rs_out && lane == 0) rs_out[row] = rs;
        }
        if constexpr (std::is_same_v<O, bf16_t>)
            *reinterpret_cast<bf16x4*>(dst + 4 * lane) = bf16x4{(bf16_t)o.x, (bf16_t)o.y, (bf16_t)o.z, (bf16_t)o.w};
        else
            *reinterpret_cast<float4*>(dst + 4 * lane) = o;
        return;
    }
    if (!w) {
        for (int i = lane; i < D; i += 64) dst[i] = (O)bw_ld<BF>(x, src + i);
        return;
    }
    float ss = 0.f;
    for (int i = lane; i < D; i += 64) {
        const float v = bw_ld<BF>(x, src + i);
        ss = fmaf(v, v, ss);
    }
    const float rs = rsqrtf(bw_wave_sum(ss) / (float)D + eps);
    for (int i = lane; i < D; i += 64) dst[i] = bw_ld<BF>(x, src + i) * rs * w[i];
    if (rs_out && lane == 0) rs_out[row] = rs;
}

// Global accesses of the backward kernels go through buffer resources over
// regions below 2^31 bytes (a chunk's rows, one state), each out-of-range
// element predicated through its offset: no branch among the loads, at which
// the compiler would wait for every load in flight.
typedef __amdgpu_buffer_rsrc_t bw_rsrc_t;
constexpr uint32_t BW_DEAD = 0x80000000u;  // past every region below (each < 2^31 bytes)

__device__ __forceinline__ bw_rsrc_t bw_rsrc(const float* base, size_t elems) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, (int)(uint32_t)(elems * 4), 0x00020000);
}
__device__ __forceinline__ bw_rsrc_t bw_rsrc(const bf16_t* base, size_t elems) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base), (short)0, (int)(uint32_t)(elems * 2), 0x00020000);
}

// A buffer store that the range check drops when dead is set.
__device__ __forceinline__ void bw_store(bw_rsrc_t r, uint32_t off, bool live, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, off | (live ? 0u : BW_DEAD), 0, 0);
}
__device__ __forceinline__ float bw_load(bw_rsrc_t r, uint32_t off, bool live) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off | (live ? 0u : BW_DEAD), 0, 0));
}
// The same for one bf16 element (off in bytes): stored rounded, loaded widened.
__device__ __forceinline__ void bw_store_h(bw_rsrc_t r, uint32_t off, bool live, float v) {
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, (bf16_t)v), r, off | (live ? 0u : BW_DEAD), 0,
                                          0);
}
__device__ __forceinline__ float bw_load_h(bw_rsrc_t r, uint32_t off, bool live) {
    const unsigned short u = __builtin_amdgcn_raw_buffer_load_b16(r, off | (live ? 0u : BW_DEAD), 0, 0);
    return __builtin_bit_cast(float, (uint32_t)u << 16);
}
__device__ __forceinline__ f32x4 bf16x4_bits_to_f32x4(uint32_t w0, uint32_t w1) {
    return f32x4{__builtin_bit_cast(float, w0 << 16), __builtin_bit_cast(float, w0 & 0xffff0000u),
                 __builtin_bit_cast(float, w1 << 16), __builtin_bit_cast(float, w1 & 0xffff0000u)};
}

// The chunk-to-chunk scan of one pass over a [Kq, Vd] matrix X, one tile per
// workgroup (every element's recurrence is independent of the others):
//   X <- e^{G_last} X + sum_t f_t a_t (x) b_t     (a rank-64 update per chunk)
// Forward (BWD false): the states, n = 0 .. N-1, X_0 = x0 (or zero),
//   f_t = e^{G_last - G_t}, a = k, b = v; xs[n] = the state before chunk n,
//   xs[N] the final state.
// Backward (BWD true): the state cotangents, n = N-1 .. 0, X_N = x0 (the
//   final state's cotangent, or zero), f_t = scale e^{G_t}, a = q, b = dO;
//   xs[n+1] = the cotangent after chunk n, xs[0] (and x_out) the initial
//   state's; bnd[tile][n] = the 32 x 32 tile's part of <xs[n+1], S[n+1]>.
constexpr int SCAN_ROWS = BWD_SCAN_ROWS;    // rows of a boundary-term tile
// Rows of D elements per (batch row, head) and token: row t of (b, h) is at
// b * batch + h * head + t * ld, rows t >= T count as zero.
struct RowsAt {
    size_t batch, head;
    int ld, T;
    __host__ __device__ size_t at(int b, int h, int t) const { return b * batch + h * head + (size_t)t * ld; }
    __device__ int live(int t0) const { return T - t0 < 0 ? 0 : T - t0 < BC ? T - t0 : BC; }  // of the chunk at t0
};

RowsAt head_major(int H, int Tp, int D) { return {(size_t)H * Tp * D, (size_t)Tp * D, D, Tp}; }

struct StateScanArgs {
    const float *a, *b;  // head-major [B*H, Tp, Kq]; rows of Vd at bl
    RowsAt bl;
    const float* g;      // [B, T, H]
    const float* x0;     // nullable [B*H, Kq, Vd]
    float* xs;           // [B*H, N+1, Kq, Vd]
    const float* S;      // backward: the forward states [B*H, N+1, Kq, Vd]
    float* bnd;          // backward: [B*H, ntiles, N], ntiles = ceil(Vd / 32) ceil(Kq / 32)
    float* x_out;        // nullable [B*H, Kq, Vd]
    int B, T, Tp, H, Kq, Vd, N;
    float scale;
    int sbf;             // matrix-core form: xs and S hold bf16 (bf16_t) states
    int bbf;             // matrix-core form: b holds bf16 (bf16_t) rows
};

// The rank-64 update X += A^T B over the chunk's 64 tokens runs on the matrix
// cores. bf16 operands: split-bf16 products on v_mfma_f32_16x16x32_bf16 (each
// fp32 operand as a bf16 high part and a bf16 remainder, lo_a hi_b + hi_a lo_b
// + hi_a hi_b: about 16 mantissa bits, as in the chunk kernels' tile GEMMs).
// fp32 operands (F32): fp32 products on v_mfma_f32_16x16x4_f32, lane (lr, lg)
// holding tokens lg + 4 e as its k of steps e = 0 .. 7. (As
// fp32 FMA loops, one 4-byte LDS read of a per row and token, the scan of a
// 256 x 128 state over 16 chunks of 8 (b, h) took 50 us forward and 35 backward;
// here 19 and 23.)
// A workgroup takes a 32 T2 x 32 T2 tile, wave w of its 4 (T2 = 1) or 8 the
// 16 x 16 T2 block of rows 16 (w >> 1) and columns 16 T2 (w & 1) as T2
// accumulators: lane (lr, lg) of accumulator jb has rows 16 (w >> 1) + 4 lg + i,
// column 16 T2 (w & 1) + 16 jb + lr. The larger tile reads each
// chunk's rows of a and b from fewer workgroups (the scans are bound by those
// reads: every column tile reads the rows of a again, every row tile the
// columns of b). Per chunk, thread (r, q) = (tid % 32 T2, tid / 32 T2) loads
// tokens 8 q .. + 8 of row r of a and of column r of b and stages them
// transposed (row = state coordinate, 64 tokens along the row), so that every
// operand fragment is consecutive in LDS. The boundary terms go to bnd per
// 32 x 32 tile: with T2 = 2 one per pair of waves, with T2 = 1 one
// per workgroup.
constexpr int SCAN_LDT = BC + 8;  // staged row: 64 tokens + 8 of padding (bf16)
constexpr int SCAN_LDF = BC + 4;  // the same in fp32

__device__ __forceinline__ void split_bf16x8(const float* v, bf16x8& hi, bf16x8& lo) {
#pragma unroll
    for (int x = 0; x < 8; x++) {
        hi[x] = (bf16_t)v[x];
        lo[x] = (bf16_t)(v[x] - (float)hi[x]);
    }
}

// v_mfma_f32_16x16x4_f32 (fp32 operands, fp32 accumulation): lane l holds
// A[l % 16][l / 16] and B[l / 16][l % 16] of a 16 x 4 by 4 x 16 step and rows
// 4 (l / 16) .. + 3 of column l % 16 of the 16 x 16 result.
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// c += A B^T over 32 k of fp32 rows: a and b point at this lane's eight
// consecutive k (k = 8 (lane / 16) ..) of its row of A and of B.
__device__ __forceinline__ f32x4 mfma_f32x8(const float* a, const float* b, f32x4 c) {
    const f32x4 a0 = *reinterpret_cast<const f32x4*>(a), a1 = *reinterpret_cast<const f32x4*>(a + 4);
    const f32x4 b0 = *reinterpret_cast<const f32x4*>(b), b1 = *reinterpret_cast<const f32x4*>(b + 4);
#pragma unroll
    for (int e = 0; e < 4; e++) c = mfma4(a0[e], b0[e], c);
#pragma unroll
    for (int e = 0; e < 4; e++) c = mfma4(a1[e], b1[e], c);
    return c;
}

template <bool BWD, int T2, bool SB, bool BB, bool F32 = false>
__global__ __launch_bounds__(T2 == 2 ? 512 : 256) void bw_state_scan_mf_kernel(StateScanArgs p) {
    static_assert(!F32 || (!SB && !BB), "fp32 operands, fp32 states");
    using SE = std::conditional_t<SB, bf16_t, float>;  // the stored states' element
    using BE = std::conditional_t<BB, bf16_t, float>;  // b's element
    static_assert(SCAN_ROWS == 32 && BW_TILE == 32 && (T2 == 1 || T2 == 2), "32 x 32 bnd tiles");
    constexpr int TS = 32 * T2;     // tile side
    // Waves: 8 for 64 x 64 tiles (one workgroup per CU at configuration 3's
    // shapes, so that two waves share each SIMD), 4 for 32 x 32; wave w holds
    // the 16 x 16 T2 block of rows 16 (w / 2) and columns 16 T2 (w % 2).
    constexpr int NTH = T2 == 2 ? 512 : 256, NWV = NTH / 64, IB = 1;
    constexpr int TPT = BC / (NTH / TS);  // tokens per staging thread
    __shared__ __align__(16) bf16_t sAh[F32 ? 1 : TS][SCAN_LDT], sAl[F32 ? 1 : TS][SCAN_LDT];
    __shared__ __align__(16) bf16_t sBh[F32 ? 1 : TS][SCAN_LDT], sBl[F32 ? 1 : TS][SCAN_LDT];
    __shared__ __align__(16) float sAf[F32 ? TS : 1][SCAN_LDF], sBf[F32 ? TS : 1][SCAN_LDF];
    __shared__ float sF[BC];
    __shared__ float sRed[NWV];
    __shared__ float sEl;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    // Workgroups go to the eight XCDs in turn; the tiles of one (b, h), which
    // read the same rows of a and b, are taken eight apart, so that they share
    // an XCD's L2 (the last B H % 8 in order): at 32 (b, h) of 32 chunks the
    // four scans 297 -> 290 us. The small tiles, 32 workgroups to a 256 x 128
    // state, go in order: 8 (b, h) of 16 chunks 75 us, and 81 shared.
    const int ntile = gridDim.x * gridDim.y, wg = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const bool swz = T2 == 2 && wg < (int)(gridDim.z & ~7u) * ntile;
    const int bhi = swz ? wg / (8 * ntile) * 8 + wg % 8 : wg / ntile;
    const int tile = swz ? wg % (8 * ntile) / 8 : wg % ntile;
    const int tcol = tile % (int)gridDim.x, trow = tile / (int)gridDim.x;
    const int c0 = tcol * TS, r0 = trow * TS;
    const int b = bhi / p.H, h = bhi % p.H;
    const int Kq = p.Kq, Vd = p.Vd, N = p.N;
    // bnd tiles of 32 x 32: nx across Vd, ny down Kq; this workgroup's (T2 = 1)
    // or this wave's and its partner's, wave w ^ 2 (T2 = 2)
    const int nx = (Vd + 31) / 32, ny = (Kq + 31) / 32, nt = nx * ny;
    const int ty = T2 == 1 ? trow : 2 * trow + (wv >> 2);
    const int tx = T2 == 1 ? tcol : 2 * tcol + (wv & 1);
    const size_t bh = bhi, ssz = (size_t)Kq * Vd;
    SE* xs = reinterpret_cast<SE*>(p.xs) + bh * (N + 1) * ssz;
    const SE* Sx = reinterpret_cast<const SE*>(p.S);
    const float* A = p.a + bh * p.Tp * Kq;
    const BE* Bm = reinterpret_cast<const BE*>(p.b) + p.bl.at(b, h, 0);
    const int ldb = p.bl.ld;
    const int wr = 16 * IB * (wv >> 1), wc = 16 * T2 * (wv & 1);  // the wave's block
    bool ok[IB][T2][4];
    uint32_t off[IB][T2][4];
    f32x4 x[IB][T2];
    const bw_rsrc_t rx0 = bw_rsrc(p.x0 ? p.x0 + bh * ssz : nullptr, p.x0 ? ssz : 0);
#pragma unroll
    for (int ib = 0; ib < IB; ib++)
#pragma unroll
        for (int jb = 0; jb < T2; jb++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int xr = r0 + wr + 16 * ib + 4 * lg + i, xc = c0 + wc + 16 * jb + lr;
                ok[ib][jb][i] = xr < Kq && xc < Vd;
                off[ib][jb][i] = ((uint32_t)xr * (uint32_t)Vd + (uint32_t)xc) * 4u;
                x[ib][jb][i] = bw_load(rx0, off[ib][jb][i], ok[ib][jb][i]);
            }
    float sv[IB][T2][4] = {};
    const auto fetch_state = [&](int n) {
        const bw_rsrc_t rs = bw_rsrc(Sx + (bh * (N + 1) + n) * ssz, ssz);
#pragma unroll
        for (int ib = 0; ib < IB; ib++)
#pragma unroll
            for (int jb = 0; jb < T2; jb++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    sv[ib][jb][i] = SB ? bw_load_h(rs, off[ib][jb][i] / 2u, ok[ib][jb][i])
                                       : bw_load(rs, off[ib][jb][i], ok[ib][jb][i]);
    };
    const auto keep = [&](int n) {  // xs[n] = X; returns the lane's part of <X, S[n]> (backward)
        const bw_rsrc_t rs = bw_rsrc(xs + (size_t)n * ssz, ssz);
        float dot = 0.f;
#pragma unroll
        for (int ib = 0; ib < IB; ib++)
#pragma unroll
            for (int jb = 0; jb < T2; jb++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if constexpr (SB)
                        bw_store_h(rs, off[ib][jb][i] / 2u, ok[ib][jb][i], x[ib][jb][i]);
                    else
                        bw_store(rs, off[ib][jb][i], ok[ib][jb][i], x[ib][jb][i]);
                    if constexpr (BWD) dot = fmaf(x[ib][jb][i], sv[ib][jb][i], dot);
                }
        return dot;
    };
    const int sr = tid % TS, sq = tid / TS;  // staging: row / column sr, tokens TPT sq ..
    const bw_rsrc_t rgt = bw_rsrc(p.g, (size_t)p.B * p.T * p.H);  // B T H < 2^21 (host)
    // chunk n's rows of a, columns of b and gate into (ra, rb, rg)
    const auto fetch = [&](int n, float* ra, float* rb, float& rg) {
        const int t0 = n * BC;
        const int live = p.bl.live(t0);  // rows past them lie past the resource (ld >= Vd): zero
        const bw_rsrc_t rA = bw_rsrc(A + (size_t)t0 * Kq, (size_t)BC * Kq),
                        rBm = bw_rsrc(Bm + (size_t)t0 * ldb, live ? (size_t)(live - 1) * ldb + Vd : 0);
#pragma unroll
        for (int i = 0; i < TPT; i++) {
            const uint32_t t = TPT * sq + i;
            ra[i] = bw_load(rA, (t * (uint32_t)Kq + (uint32_t)(r0 + sr)) * 4u, r0 + sr < Kq);
            rb[i] = BB ? bw_load_h(rBm, (t * (uint32_t)ldb + (uint32_t)(c0 + sr)) * 2u, c0 + sr < Vd)
                       : bw_load(rBm, (t * (uint32_t)ldb + (uint32_t)(c0 + sr)) * 4u, c0 + sr < Vd);
        }
        rg = bw_load(rgt, (((uint32_t)b * (uint32_t)p.T + (uint32_t)(t0 + lane)) * (uint32_t)p.H + (uint32_t)h) * 4u,
                     t0 + lane < p.T);
    };
    // eight tokens t0 .. of an fp32 row: token t at 32 (t / 32) + 8 (t % 4) +
    // (t % 32) / 4, so that the matrix core adds the tokens in order, four per
    // step (the decayed ones of a chunk are added smallest first, as a loop
    // over the tokens adds them)
    const auto put_f32 = [](float* row, int t0, const float* v) {
#pragma unroll
        for (int m = 0; m < 4; m++)
            *reinterpret_cast<f32x2*>(row + t0 / 32 * 32 + 8 * m + t0 % 32 / 4) = f32x2{v[m], v[m + 4]};
    };
    const auto chunk_of = [&](int step) { return BWD ? N - 1 - step : step; };
    // One chunk step from the registers (ra, rb, rg), which then receive the
    // next chunk. (Two register sets, with the chunk two steps on in flight,
    // were slower: 83 -> 93 us for the forward scan at configuration 3; the
    // scan is bound by each compute unit's reads, not by their latency.)
    const auto run_step = [&](int step, float* ra, float* rb, float& rg) {
        const int n = chunk_of(step);
        const float dot = keep(BWD ? n + 1 : n);
        __syncthreads();  // the previous chunk's operands are done with
        float wsum = 0.f;
        if constexpr (BWD) {
            wsum = bw_wave_sum(dot);
            if (lane == 0) sRed[wv] = wsum;
        }
        if (wv == 0) {  // G: the in-chunk inclusive cumsum of the prefetched gate
            const float G = bw_wave_scan(rg);
            const float Gl = lane_value(G, 63);
            sF[lane] = BWD ? p.scale * expf(G) : expf(Gl - G);
            if (lane == 0) sEl = expf(Gl);
        }
#pragma unroll
        for (int u = 0; u < TPT / 8; u++) {
            if constexpr (F32) {
                put_f32(sBf[sr], TPT * sq + 8 * u, rb + 8 * u);
                continue;
            }
            bf16x8 hi, lo;
            split_bf16x8(rb + 8 * u, hi, lo);
            *reinterpret_cast<bf16x8*>(&sBh[sr][TPT * sq + 8 * u]) = hi;
            *reinterpret_cast<bf16x8*>(&sBl[sr][TPT * sq + 8 * u]) = lo;
        }
        __syncthreads();  // sF is read below
#pragma unroll
        for (int u = 0; u < TPT / 8; u++) {
            float fa[8];
#pragma unroll
            for (int i = 0; i < 8; i++) fa[i] = sF[TPT * sq + 8 * u + i] * ra[8 * u + i];
            if constexpr (F32) {
                put_f32(sAf[sr], TPT * sq + 8 * u, fa);
                continue;
            }
            bf16x8 hi, lo;
            split_bf16x8(fa, hi, lo);
            *reinterpret_cast<bf16x8*>(&sAh[sr][TPT * sq + 8 * u]) = hi;
            *reinterpret_cast<bf16x8*>(&sAl[sr][TPT * sq + 8 * u]) = lo;
        }
        __syncthreads();
        if (step + 1 < N) fetch(chunk_of(step + 1), ra, rb, rg);
        if constexpr (BWD) fetch_state(n);  // for the next step's keep(n)
        if constexpr (BWD) {
            if (T2 == 1 && tid == 0)
                p.bnd[(bh * nt + ty * nx + tx) * N + n] = (sRed[0] + sRed[1]) + (sRed[2] + sRed[3]);
            if (T2 == 2 && lane == 0 && (wv & 2) == 0 && ty < ny && tx < nx)  // the tile's two waves
                p.bnd[(bh * nt + ty * nx + tx) * N + n] = sRed[wv] + sRed[wv + 2];
        }
        const float el = sEl;
#pragma unroll
        for (int ib = 0; ib < IB; ib++)
#pragma unroll
            for (int jb = 0; jb < T2; jb++)
#pragma unroll
                for (int i = 0; i < 4; i++) x[ib][jb][i] *= el;
#pragma unroll
        for (int s = 0; s < BC / 32; s++) {
            if constexpr (F32) {
#pragma unroll
                for (int ib = 0; ib < IB; ib++)
#pragma unroll
                    for (int jb = 0; jb < T2; jb++)
                        x[ib][jb] = mfma_f32x8(&sAf[wr + 16 * ib + lr][32 * s + 8 * lg], &sBf[wc + 16 * jb + lr][32 * s + 8 * lg],
                                               x[ib][jb]);
                continue;
            }
            bf16x8 ah[IB], al[IB], bh8[T2], bl8[T2];
#pragma unroll
            for (int ib = 0; ib < IB; ib++) {
                ah[ib] = *reinterpret_cast<const bf16x8*>(&sAh[wr + 16 * ib + lr][32 * s + 8 * lg]);
                al[ib] = *reinterpret_cast<const bf16x8*>(&sAl[wr + 16 * ib + lr][32 * s + 8 * lg]);
            }
#pragma unroll
            for (int jb = 0; jb < T2; jb++) {
                bh8[jb] = *reinterpret_cast<const bf16x8*>(&sBh[wc + 16 * jb + lr][32 * s + 8 * lg]);
                bl8[jb] = *reinterpret_cast<const bf16x8*>(&sBl[wc + 16 * jb + lr][32 * s + 8 * lg]);
            }
#pragma unroll
            for (int ib = 0; ib < IB; ib++)
#pragma unroll
                for (int jb = 0; jb < T2; jb++) {
                    x[ib][jb] = mfma_bf16(al[ib], bh8[jb], x[ib][jb]);
                    x[ib][jb] = mfma_bf16(ah[ib], bl8[jb], x[ib][jb]);
                    x[ib][jb] = mfma_bf16(ah[ib], bh8[jb], x[ib][jb]);
                }
        }
    };
    float ra[TPT], rb[TPT], rg;
    fetch(chunk_of(0), ra, rb, rg);
    if constexpr (BWD) fetch_state(N);
    for (int step = 0; step < N; step++) run_step(step, ra, rb, rg);
    keep(BWD ? 0 : N);
    const bw_rsrc_t rxo = bw_rsrc(p.x_out ? p.x_out + bh * ssz : nullptr, p.x_out ? ssz : 0);
#pragma unroll
    for (int ib = 0; ib < IB; ib++)
#pragma unroll
        for (int jb = 0; jb < T2; jb++)
#pragma unroll
            for (int i = 0; i < 4; i++) bw_store(rxo, off[ib][jb][i], ok[ib][jb][i], x[ib][jb][i]);  // dropped without x_out
}

// Launches the scan over a [Kq, Vd] state, with split-bf16 products (mfma) or
// fp32 ones, in 64 x 64 tiles when they still give a workgroup per compute
// unit, else in 32 x 32 tiles.
template <bool BWD, int T2>
void launch_scan_mf(const StateScanArgs& a, bool mfma, dim3 grid, hipStream_t stream) {
    const dim3 blk(T2 == 2 ? 512 : 256);
    if (!mfma)
        hipLaunchKernelGGL((bw_state_scan_mf_kernel<BWD, T2, false, false, true>), grid, blk, 0, stream, a);
    else if (a.sbf && a.bbf)
        hipLaunchKernelGGL((bw_state_scan_mf_kernel<BWD, T2, true, true>), grid, blk, 0, stream, a);
    else if (a.sbf)
        hipLaunchKernelGGL((bw_state_scan_mf_kernel<BWD, T2, true, false>), grid, blk, 0, stream, a);
    else  // (bf16 rows come with bf16 states)
        hipLaunchKernelGGL((bw_state_scan_mf_kernel<BWD, T2, false, false>), grid, blk, 0, stream, a);
}

template <bool BWD>
void launch_state_scan(const StateScanArgs& a, bool mfma, hipStream_t stream) {
    const dim3 g32((a.Vd + 31) / 32, (a.Kq + 31) / 32, a.B * a.H), g64((a.Vd + 63) / 64, (a.Kq + 63) / 64, a.B * a.H);
    if ((long long)g64.x * g64.y * g64.z >= device_cu_count())
        launch_scan_mf<BWD, 2>(a, mfma, g64, stream);
    else
        launch_scan_mf<BWD, 1>(a, mfma, g32, stream);
}

// Tile GEMMs of the chunk kernels: a 64 x 64 NT output tile (rows = the chunk's
// tokens, columns = coordinates), accumulated over a contraction of Kd in
// k-blocks of 32 staged through LDS, the next k-block's operands prefetched
// into registers while the current one is multiplied. fa(i, kk) and fb(kk, j)
// read the operands. Wave w forms rows 16 w .. + 16 as 4 NT blocks of 16 x 16:
// acc[nb][i] = tile[16 w + 4 (lane / 16) + i][16 nb + lane % 16] (TileMap).
//  - MF true (bf16 operands): matrix cores at near-fp32 accuracy: each fp32
//    operand is split into hi = bf16(x) and lo = bf16(x - hi), staged in LDS,
//    and a.b formed as lo_a hi_b + hi_a lo_b + hi_a hi_b on
//    v_mfma_f32_16x16x32_bf16 with fp32 accumulation (about 16 mantissa
//    bits; the dropped lo_a lo_b is 2^-16 relative). The kernels are bound by
//    the staging, not the matrix cores, so the three products cost about what
//    one does.
//  - MF false (fp32 operands): fp32 products and sums on
//    v_mfma_f32_16x16x4_f32, the operands staged as fp32. (As fp32 FMA loops, a
//    4 x 4 block per thread with 4-byte operand loads, the chunk kernel took
//    181 us for 128 chunks of 256 x 128 and the output kernel 88; here, with
//    the chunk's tiles shared out over three and two workgroups, 47 and 22.)
// The wide readout's GEMMs (128 < M) keep fp32 FMA in a 4 x 4 block per thread
// (tile_gemm_fma), whose threads hold neighbouring columns.
constexpr int GT_K = 32, GT_LD = 68;  // FMA staging: [32][68] per operand
constexpr int MT_LD = 40;             // bf16 staging: [64][40] per operand part (32 k + 8 pad)
constexpr int FT_LD = 36;             // fp32 staging: [64][36] per operand
// Row r of a staged 64-row block: every 16 rows start 16 bytes further on. A
// B operand contiguous along j is staged column by column, lane (jq, kp)
// writing row 4 jq + c: at an even pitch of 20 dwords (36 in fp32) the sixteen
// jq of a store fall on four of the 64 banks; with the offset, on sixteen, so
// that a wave's store touches each bank once (at 1024 chunks of 256 x 128 the
// chunk kernels 191 -> 174 and 172 -> 157 us, the output kernel 74 -> 66; in
// fp32 at 128 chunks 50 -> 47 and 24 -> 22). The 16-byte reads of 16
// neighbouring rows keep their pitch.
__device__ __forceinline__ constexpr int mt_row(int r) { return r * MT_LD + r / 16 * 8; }
__device__ __forceinline__ constexpr int ft_row(int r) { return r * FT_LD + r / 16 * 4; }
constexpr int MT_TILE = BC * MT_LD + BC / 16 * 8, FT_TILE = BC * FT_LD + BC / 16 * 4;
constexpr int STAGE_BYTES = 4 * MT_TILE * 2;   // A and a B block, hi and lo
constexpr int STAGE2_BYTES = 6 * MT_TILE * 2;  // the same with two B blocks
static_assert(STAGE_BYTES >= 2 * GT_K * GT_LD * 4 && STAGE_BYTES >= 2 * FT_TILE * 4 && STAGE2_BYTES >= 3 * FT_TILE * 4,
              "staging must hold every form");

struct TileMap {
    __device__ static int row(int, int b) { return 16 * (threadIdx.x >> 6) + 4 * ((threadIdx.x & 63) >> 4) + b; }
    __device__ static int col(int a, int) { return 16 * a + (threadIdx.x & 15); }
};

struct FmaMap {
    __device__ static int row(int a, int) { return 4 * (threadIdx.x >> 4) + a; }
    __device__ static int col(int, int b) { return 4 * (threadIdx.x & 15) + b; }
};

// Global operands of tile_gemm, read through a buffer resource over the
// operand's region with every out-of-range element predicated to zero through
// its offset (so the next k-block's loads overlap the current one's products).
//  RowsK: element (m, kk) = base[m ld + kk] for m < nm, kk < nk (the A
//         operand, m = the tile row, and a B operand contiguous along kk,
//         m = the tile column).
//  RowsJ: element (kk, j) = base[kk ld + j] for kk < nk, j < nj (a B operand
//         contiguous along j).
struct RowsK {
    bw_rsrc_t r;
    uint32_t ld;
    int nm, nk;
    __device__ RowsK(const float* base, int ld_, int nm_, int nk_)
        : r(bw_rsrc(base, nm_ > 0 ? (size_t)(nm_ - 1) * ld_ + nk_ : 0)), ld((uint32_t)ld_), nm(nm_), nk(nk_) {}
    __device__ float load(int m, int kk) const {
        const uint32_t dead = (m < nm && kk < nk) ? 0u : BW_DEAD;
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, ((uint32_t)m * ld + (uint32_t)kk) * 4u | dead, 0, 0));
    }
};

// RowsK with 16-byte loads of four consecutive kk: the caller guarantees a
// 16-byte aligned base and ld, nk multiples of 4. In tile_gemm's matrix-core
// staging, lane (r, kg) then loads kk = k0 + 4 kg .. + 3 and k0 + 16 + 4 kg ..
// + 3, so that each load instruction covers 64 contiguous bytes of 16 rows
// (with one 4-byte load per kk, eight instructions each touched 16 lines).
struct RowsK4 : RowsK {
    __device__ RowsK4(const float* base, int ld_, int nm_, int nk_) : RowsK(base, ld_, nm_, nk_) {}
    __device__ f32x4 load4(int m, int kk0) const {
        const uint32_t dead = (m < nm && kk0 < nk) ? 0u : BW_DEAD;
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, ((uint32_t)m * ld + (uint32_t)kk0) * 4u | dead, 0, 0));
    }
};

struct RowsJ {
    bw_rsrc_t r;
    uint32_t ld;
    int nk, nj;
    __device__ RowsJ(const float* base, int ld_, int nk_, int nj_)
        : r(bw_rsrc(base, nk_ > 0 ? (size_t)(nk_ - 1) * ld_ + nj_ : 0)), ld((uint32_t)ld_), nk(nk_), nj(nj_) {}
    __device__ float load(int kk, int j) const {
        const uint32_t dead = (kk < nk && j < nj) ? 0u : BW_DEAD;
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, ((uint32_t)kk * ld + (uint32_t)j) * 4u | dead, 0, 0));
    }
};

// RowsJ with 16-byte loads of four consecutive j (16-byte aligned base, ld and
// nj multiples of 4). In tile_gemm's matrix-core staging, lane (jq, kp) =
// (tid % 16, tid / 16) loads j = 4 jq .. + 3 of rows kk = k0 + 2 kp and
// k0 + 2 kp + 1 (each load instruction covers whole 256-byte row segments)
// and writes the pairs (kk, kk + 1) of its four columns as 4-byte LDS stores.
struct RowsJ4 : RowsJ {
    __device__ RowsJ4(const float* base, int ld_, int nk_, int nj_) : RowsJ(base, ld_, nk_, nj_) {}
    __device__ f32x4 load4(int kk, int j0) const {
        const uint32_t dead = (kk < nk && j0 < nj) ? 0u : BW_DEAD;
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, ((uint32_t)kk * ld + (uint32_t)j0) * 4u | dead, 0, 0));
    }
};

// RowsK, RowsK4, RowsJ and RowsJ4 over bf16 elements (the stored states and
// state cotangents of bf16 calls): two-byte loads, and load4's four
// consecutive elements in one 8-byte load (16-byte aligned base, ld and the
// extent multiples of 4). The values widen to fp32 exactly.
struct RowsKh : RowsK {
    __device__ RowsKh(const bf16_t* base, int ld_, int nm_, int nk_) : RowsK(nullptr, ld_, nm_, nk_) {
        r = bw_rsrc(base, nm_ > 0 ? (size_t)(nm_ - 1) * ld_ + nk_ : 0);
    }
    __device__ float load(int m, int kk) const {
        return bw_load_h(r, ((uint32_t)m * ld + (uint32_t)kk) * 2u, m < nm && kk < nk);
    }
};
struct RowsK4h : RowsK4 {
    __device__ RowsK4h(const bf16_t* base, int ld_, int nm_, int nk_) : RowsK4(nullptr, ld_, nm_, nk_) {
        r = bw_rsrc(base, nm_ > 0 ? (size_t)(nm_ - 1) * ld_ + nk_ : 0);
    }
    __device__ float load(int m, int kk) const {
        return bw_load_h(r, ((uint32_t)m * ld + (uint32_t)kk) * 2u, m < nm && kk < nk);
    }
    __device__ f32x4 load4(int m, int kk0) const {
        const uint32_t dead = (m < nm && kk0 < nk) ? 0u : BW_DEAD;
        const auto w = __builtin_amdgcn_raw_buffer_load_b64(r, ((uint32_t)m * ld + (uint32_t)kk0) * 2u | dead, 0, 0);
        return bf16x4_bits_to_f32x4(w[0], w[1]);
    }
};
struct RowsJh : RowsJ {
    __device__ RowsJh(const bf16_t* base, int ld_, int nk_, int nj_) : RowsJ(nullptr, ld_, nk_, nj_) {
        r = bw_rsrc(base, nk_ > 0 ? (size_t)(nk_ - 1) * ld_ + nj_ : 0);
    }
    __device__ float load(int kk, int j) const {
        return bw_load_h(r, ((uint32_t)kk * ld + (uint32_t)j) * 2u, kk < nk && j < nj);
    }
};
struct RowsJ4h : RowsJ4 {
    __device__ RowsJ4h(const bf16_t* base, int ld_, int nk_, int nj_) : RowsJ4(nullptr, ld_, nk_, nj_) {
        r = bw_rsrc(base, nk_ > 0 ? (size_t)(nk_ - 1) * ld_ + nj_ : 0);
    }
    __device__ float load(int kk, int j) const {
        return bw_load_h(r, ((uint32_t)kk * ld + (uint32_t)j) * 2u, kk < nk && j < nj);
    }
    __device__ f32x4 load4(int kk, int j0) const {
        const uint32_t dead = (kk < nk && j0 < nj) ? 0u : BW_DEAD;
        const auto w = __builtin_amdgcn_raw_buffer_load_b64(r, ((uint32_t)kk * ld + (uint32_t)j0) * 2u | dead, 0, 0);
        return bf16x4_bits_to_f32x4(w[0], w[1]);
    }
};

// The state operands' row types: fp32, or bf16 with SB.
template <bool SB, bool V4>
using StateRowsK = std::conditional_t<SB, std::conditional_t<V4, RowsK4h, RowsKh>, std::conditional_t<V4, RowsK4, RowsK>>;
template <bool SB, bool V4>
using StateRowsJ = std::conditional_t<SB, std::conditional_t<V4, RowsJ4h, RowsJh>, std::conditional_t<V4, RowsJ4, RowsJ>>;

// Element (i, kk) of A and (kk, j) of B, for a global operand or a callable
// (LDS operands: read only at kk < Kd, contractions of BC tokens).
template <class FA>
__device__ __forceinline__ float opA(const FA& fa, int i, int kk, int Kd) {
    if constexpr (std::is_base_of_v<RowsK, FA>)
        return fa.load(i, kk);
    else
        return kk < Kd ? fa(i, kk) : 0.f;
}
template <class FB>
__device__ __forceinline__ float opB(const FB& fb, int kk, int j, int Kd) {
    if constexpr (std::is_base_of_v<RowsK, FB>)
        return fb.load(j, kk);
    else if constexpr (std::is_base_of_v<RowsJ, FB>)
        return fb.load(kk, j);
    else
        return kk < Kd ? fb(kk, j) : 0.f;
}

// A callable A operand whose contraction runs over tokens s <= t: its decayed
// terms grow with s, so fp32 sums take the tokens in order, smallest first (as
// put_f32 of the scans). In the staging's natural order, where a step of the
// matrix core adds tokens e, e + 8, e + 16 and e + 24, dq's error against 64
// bits was 1% above that of a loop over the tokens (4 x 4096 tokens of 8 heads
// 16 wide). The sums of dk and dv, over s >= t, come out 1% and 0.3% better in
// the natural order, and keep it.
template <class F>
struct InOrder {
    F f;
    __device__ float operator()(int i, int kk) const { return f(i, kk); }
};
template <class F>
__device__ __forceinline__ InOrder<F> in_order(F f) {
    return InOrder<F>{f};
}
template <class F>
constexpr bool is_in_order = false;
template <class F>
constexpr bool is_in_order<InOrder<F>> = true;

// tile_gemm (above) for an output of 64 rows by 64 NT columns in one pass over
// the contraction: A is staged once per
// k-block and multiplied against NT B tiles, so that a row block feeding
// several output tiles is read once (NT = 2 halves those reads against two
// passes).
template <bool MF, int NT, class FA, class FB>
__device__ __forceinline__ void tile_gemm(FA fa, FB fb, int Kd, unsigned char* stage, float acc[4 * NT][4]) {
    const int tid = threadIdx.x;
    {
        float* saf = reinterpret_cast<float*>(stage);  // fp32: A (64 rows), then B (64 NT rows)
        float* sbf = saf + FT_TILE;
        bf16_t* sah = reinterpret_cast<bf16_t*>(stage);  // hi and lo parts of A (64 rows) and of B (64 NT rows)
        bf16_t* sal = sah + MT_TILE;
        bf16_t* sbh = sal + MT_TILE;
        bf16_t* sbl = sbh + NT * MT_TILE;
        const int l = tid & 63, w = tid >> 6, lr = l & 15, lg = l >> 4;
        const int r = tid >> 2, kg = tid & 3;  // staging: row r, k-group kg (8 k)
        // RowsK4 operands: lane (r, kg) holds kk = k0 + 4 kg .. + 3 and
        // k0 + 16 + 4 kg .. + 3; the others kk = k0 + 8 kg .. + 7
        constexpr bool VA = std::is_base_of_v<RowsK4, FA>, VB = std::is_base_of_v<RowsK4, FB>;
        constexpr bool JB = std::is_base_of_v<RowsJ4, FB>;  // B: lane (jq, kp) as in RowsJ4
        const int jq = tid & 15, kp = tid >> 4;
        float ra[8], rb[NT][8];
        const auto fetch = [&](int k0) {
            if constexpr (VA) {
                const f32x4 lo4 = fa.load4(r, k0 + 4 * kg), hi4 = fa.load4(r, k0 + 16 + 4 * kg);
#pragma unroll
                for (int x = 0; x < 4; x++) ra[x] = lo4[x], ra[4 + x] = hi4[x];
            } else {
#pragma unroll
                for (int x = 0; x < 8; x++) ra[x] = opA(fa, r, k0 + 8 * kg + x, Kd);
            }
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {  // B's columns 64 nt ..
                if constexpr (VB) {
                    const f32x4 lo4 = fb.load4(64 * nt + r, k0 + 4 * kg), hi4 = fb.load4(64 * nt + r, k0 + 16 + 4 * kg);
#pragma unroll
                    for (int x = 0; x < 4; x++) rb[nt][x] = lo4[x], rb[nt][4 + x] = hi4[x];
                } else if constexpr (JB) {  // rb[c] = B(k0 + 2 kp, 4 jq + c), rb[4 + c] = B(k0 + 2 kp + 1, 4 jq + c)
                    const f32x4 r0 = fb.load4(k0 + 2 * kp, 64 * nt + 4 * jq), r1 = fb.load4(k0 + 2 * kp + 1, 64 * nt + 4 * jq);
#pragma unroll
                    for (int x = 0; x < 4; x++) rb[nt][x] = r0[x], rb[nt][4 + x] = r1[x];
                } else {
#pragma unroll
                    for (int x = 0; x < 8; x++) rb[nt][x] = opB(fb, k0 + 8 * kg + x, 64 * nt + r, Kd);
                }
            }
        };
        // writes the 8 staged values of one operand in its lane order
        const auto put = [&](bf16_t* base, bool split4, const bf16x8& v) {
            if (split4) {
                *reinterpret_cast<bf16x4*>(base + mt_row(r) + 4 * kg) = bf16x4{v[0], v[1], v[2], v[3]};
                *reinterpret_cast<bf16x4*>(base + mt_row(r) + 16 + 4 * kg) = bf16x4{v[4], v[5], v[6], v[7]};
            } else {
                *reinterpret_cast<bf16x8*>(base + mt_row(r) + 8 * kg) = v;
            }
        };
        constexpr bool TOK = is_in_order<FA>;  // fp32: token t of 32 at 8 (t % 4) + t / 4
        const auto put_f = [&](float* base, bool split4, const float* v) {
            if constexpr (TOK) {  // (no split4 operand holds tokens)
#pragma unroll
                for (int x = 0; x < 4; x++)
                    *reinterpret_cast<f32x2*>(base + ft_row(r) + 8 * x + 2 * kg) = f32x2{v[x], v[x + 4]};
                return;
            }
            const int c0 = split4 ? 4 * kg : 8 * kg, c1 = split4 ? 16 + 4 * kg : 8 * kg + 4;
            *reinterpret_cast<f32x4*>(base + ft_row(r) + c0) = f32x4{v[0], v[1], v[2], v[3]};
            *reinterpret_cast<f32x4*>(base + ft_row(r) + c1) = f32x4{v[4], v[5], v[6], v[7]};
        };
        fetch(0);
        for (int k0 = 0; k0 < Kd; k0 += GT_K) {
            __syncthreads();  // the staging tiles are free
            if constexpr (!MF) {
                put_f(saf, VA, ra);
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    float* b0 = sbf + nt * FT_TILE;
                    if constexpr (JB) {
#pragma unroll
                        for (int c = 0; c < 4; c++) {
                            float* row = b0 + ft_row(4 * jq + c);
                            if constexpr (TOK) {
                                row[8 * (2 * kp % 4) + kp / 2] = rb[nt][c];
                                row[8 * (2 * kp % 4) + 8 + kp / 2] = rb[nt][4 + c];
                            } else {
                                *reinterpret_cast<f32x2*>(row + 2 * kp) = f32x2{rb[nt][c], rb[nt][4 + c]};
                            }
                        }
                    } else {
                        put_f(b0, VB, rb[nt]);
                    }
                }
                __syncthreads();
                if (k0 + GT_K < Kd) fetch(k0 + GT_K);
#pragma unroll
                for (int nb = 0; nb < 4 * NT; nb++) {
                    f32x4 c = {acc[nb][0], acc[nb][1], acc[nb][2], acc[nb][3]};
                    c = mfma_f32x8(saf + ft_row(16 * w + lr) + 8 * lg, sbf + nb / 4 * FT_TILE + ft_row(16 * (nb % 4) + lr) + 8 * lg, c);
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[nb][i] = c[i];
                }
                continue;
            }
            bf16x8 vah, val;
#pragma unroll
            for (int x = 0; x < 8; x++) {
                vah[x] = (bf16_t)ra[x];
                val[x] = (bf16_t)(ra[x] - (float)vah[x]);
            }
            put(sah, VA, vah);
            put(sal, VA, val);
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                bf16x8 vbh, vbl;
#pragma unroll
                for (int x = 0; x < 8; x++) {
                    vbh[x] = (bf16_t)rb[nt][x];
                    vbl[x] = (bf16_t)(rb[nt][x] - (float)vbh[x]);
                }
                bf16_t* bh0 = sbh + nt * MT_TILE;
                bf16_t* bl0 = sbl + nt * MT_TILE;
                if constexpr (JB) {  // column 4 jq + c: the pair (k0 + 2 kp, + 1) as one 4-byte store
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        *reinterpret_cast<bf16x2*>(bh0 + mt_row(4 * jq + c) + 2 * kp) = bf16x2{vbh[c], vbh[4 + c]};
                        *reinterpret_cast<bf16x2*>(bl0 + mt_row(4 * jq + c) + 2 * kp) = bf16x2{vbl[c], vbl[4 + c]};
                    }
                } else {
                    put(bh0, VB, vbh);
                    put(bl0, VB, vbl);
                }
            }
            __syncthreads();
            if (k0 + GT_K < Kd) fetch(k0 + GT_K);
            const int ao = mt_row(16 * w + lr) + 8 * lg;
            const bf16x8 ah = *reinterpret_cast<const bf16x8*>(sah + ao);
            const bf16x8 al = *reinterpret_cast<const bf16x8*>(sal + ao);
#pragma unroll
            for (int nb = 0; nb < 4 * NT; nb++) {
                const int bo = nb / 4 * MT_TILE + mt_row(16 * (nb % 4) + lr) + 8 * lg;
                const bf16x8 bh = *reinterpret_cast<const bf16x8*>(sbh + bo);
                const bf16x8 bl = *reinterpret_cast<const bf16x8*>(sbl + bo);
                f32x4 c = {acc[nb][0], acc[nb][1], acc[nb][2], acc[nb][3]};
                c = mfma_bf16(al, bh, c);
                c = mfma_bf16(ah, bl, c);
                c = mfma_bf16(ah, bh, c);
#pragma unroll
                for (int i = 0; i < 4; i++) acc[nb][i] = c[i];
            }
        }
    }
}

// The FMA form: B_KCONTIG says whether fb is contiguous along kk (else along
// j); acc[a][b] at (FmaMap::row, FmaMap::col); A staged transposed so a
// thread's four rows are one float4.
template <bool B_KCONTIG, class FA, class FB>
__device__ __forceinline__ void tile_gemm_fma(FA fa, FB fb, int Kd, unsigned char* stage, float acc[4][4]) {
    const int tid = threadIdx.x;
    {
        float(*sa)[GT_LD] = reinterpret_cast<float(*)[GT_LD]>(stage);
        float(*sb)[GT_LD] = reinterpret_cast<float(*)[GT_LD]>(stage + GT_K * GT_LD * 4);
        constexpr int NE = BC * GT_K / 256;  // staged elements of each operand per thread
        const int ti = 4 * (tid >> 4), tj = 4 * (tid & 15);
        float ra[NE], rb[NE];
        const auto fetch = [&](int k0) {
#pragma unroll
            for (int x = 0; x < NE; x++) {
                const int e = tid + 256 * x;
                const int ka = e % GT_K, i = e / GT_K;
                ra[x] = opA(fa, i, k0 + ka, Kd);
                const int kb = B_KCONTIG ? e % GT_K : e / BC, j = B_KCONTIG ? e / GT_K : e % BC;
                rb[x] = opB(fb, k0 + kb, j, Kd);
            }
        };
        fetch(0);
        for (int k0 = 0; k0 < Kd; k0 += GT_K) {
            __syncthreads();  // the staging tiles are free
#pragma unroll
            for (int x = 0; x < NE; x++) {
                const int e = tid + 256 * x;
                sa[e % GT_K][e / GT_K] = ra[x];
                if (B_KCONTIG)
                    sb[e % GT_K][e / GT_K] = rb[x];
                else
                    sb[e / BC][e % BC] = rb[x];
            }
            __syncthreads();
            if (k0 + GT_K < Kd) fetch(k0 + GT_K);
#pragma unroll 8
            for (int kk = 0; kk < GT_K; kk++) {
                const float4 av = *reinterpret_cast<const float4*>(&sa[kk][ti]);
                const float4 bv = *reinterpret_cast<const float4*>(&sb[kk][tj]);
                const float ar[4] = {av.x, av.y, av.z, av.w}, br[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[i][j] = fmaf(ar[i], br[j], acc[i][j]);
            }
        }
    }
}

// acc[a][b] *= f(row of (a, b)); NA = 4 NT for a tile of 64 NT columns.
template <int NA, class F>
__device__ __forceinline__ void tile_scale_rows(float acc[NA][4], F f) {
#pragma unroll
    for (int a = 0; a < NA; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) acc[a][b] *= f(TileMap::row(a, b));
}

// Writes this thread's part of a 64 x 16 NA tile (columns d0 ..) into
// head-major rows dst [.., D], times a scale.
template <int NA>
__device__ __forceinline__ void tile_store(float acc[NA][4], float* dst, int D, int d0, float scale) {
#pragma unroll
    for (int a = 0; a < NA; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int t = TileMap::row(a, b), c = d0 + TileMap::col(a, b);
            if (c < D) dst[(size_t)t * D + c] = scale * acc[a][b];
        }
}

// Masked, decayed scores of one chunk into P: P[t][s] = [s <= t] e^{G_t - G_s}
// sum_j X_t[j] Y_s[j] (X, Y: the chunk's 64 rows, D wide), as one tile GEMM.
template <bool MF, bool V4, class E>
__device__ __forceinline__ void chunk_scores(const E* X, int ldx, int nx, const E* Y, int ldy, int ny, int D,
                                             const float* sG, unsigned char* stage, float (*P)[BC + 1]) {
    using RK = StateRowsK<std::is_same_v<E, bf16_t>, V4>;  // fp32 or bf16 rows
    float acc[4][4] = {};
    tile_gemm<MF, 1>(RK(X, ldx, nx, D), RK(Y, ldy, ny, D), D, stage, acc);
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int t = TileMap::row(a, b), s = TileMap::col(a, b);
            P[t][s] = s <= t ? acc[a][b] * expf(sG[t] - sG[s]) : 0.f;
        }
}

// The output of one pass, chunk-parallel (grid (N, H, B), 256 threads):
// o_t = scale (e^{G_t} q_t S_n + sum_{s<=t} A[t][s] v_s), A the masked
// decayed q.k scores, per 64-wide output tile as two tile GEMMs. The
// backward's recompute writes pass 1 head-major and unrounded; the general
// forward rounds to bf16 for bf16 inputs and writes pass 2 as [B, T, H, Vd].
struct OutArgs {
    const float *q, *k, *v;  // head-major [B*H, Tp, Kq | Vd]
    const float* g;
    const float* S;          // [B*H, N+1, Kq, Vd]: fp32, or bf16_t with sbf
    float* out;              // head-major [B*H, Tp, Vd], used when out_bthd is null
    void* out_bthd;          // nullable [B, T, H, Vd], bf16 when bf16 else fp32
    int bf16;                // round to bf16
    int B, T, Tp, H, Kq, Vd, N;
    float scale;
    int sbf;                 // S holds bf16 states
    int parts;               // workgroups per chunk: part i forms output tiles i, i + parts, ..
};

template <bool MF, bool V4, bool SB>
__global__ __launch_bounds__(256) void bw_out_kernel(OutArgs a) {
    using RK = std::conditional_t<V4, RowsK4, RowsK>;  // 16-byte row loads when aligned
    using RJ = std::conditional_t<V4, RowsJ4, RowsJ>;
    using SJ = StateRowsJ<SB, V4>;
    using SE = std::conditional_t<SB, bf16_t, float>;
    __shared__ float sA[BC][BC + 1];
    // (output tiles of 64 columns: two at a time read q once instead of twice
    // but measured slower here, 80 -> 84 us at configuration 3)
    constexpr int NA = 4;
    __shared__ __align__(16) unsigned char sStage[STAGE_BYTES];
    __shared__ float sG[BC], sEq[BC];
    const int tid = threadIdx.x, n = blockIdx.x, h = blockIdx.y, b = blockIdx.z / a.parts, part = blockIdx.z % a.parts;
    const int Kq = a.Kq, Vd = a.Vd, t0 = n * BC;
    const size_t bh = (size_t)b * a.H + h, ssz = (size_t)Kq * Vd;
    const float* q = a.q + (bh * a.Tp + t0) * Kq;
    const float* k = a.k + (bh * a.Tp + t0) * Kq;
    const float* v = a.v + (bh * a.Tp + t0) * Vd;
    const SE* S = reinterpret_cast<const SE*>(a.S) + (bh * (a.N + 1) + n) * ssz;
    if (tid < 64) {
        sG[tid] = chunk_gam(a.g, b, h, a.T, a.H, n, tid);
        sEq[tid] = expf(sG[tid]);
    }
    chunk_scores<MF, V4>(q, Kq, BC, k, Kq, BC, Kq, sG, sStage, sA);
    float* out = a.out + (bh * a.Tp + t0) * Vd;
    for (int d0 = BC * part; d0 < Vd; d0 += BC * a.parts) {
        float acc[NA][4] = {};
        tile_gemm<MF, 1>(RK(q, Kq, BC, Kq), SJ(S + d0, Vd, Kq, Vd - d0), Kq, sStage, acc);
        tile_scale_rows<NA>(acc, [&](int t) { return sEq[t]; });
        tile_gemm<MF, 1>(in_order([&](int i, int kk) { return sA[i][kk]; }), RJ(v + d0, Vd, BC, Vd - d0), BC, sStage, acc);
        if (!a.out_bthd) {
            if (a.bf16) {
#pragma unroll
                for (int i = 0; i < NA; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[i][j] = (float)(bf16_t)(a.scale * acc[i][j]);
                tile_store<NA>(acc, out, Vd, d0, 1.f);
            } else {
                tile_store<NA>(acc, out, Vd, d0, a.scale);
            }
            continue;
        }
#pragma unroll
        for (int i = 0; i < NA; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int t = t0 + TileMap::row(i, j), c = d0 + TileMap::col(i, j);
                if (c >= Vd || t >= a.T) continue;
                const size_t e = (((size_t)b * a.T + t) * a.H + h) * Vd + c;
                if (a.bf16)
                    reinterpret_cast<bf16_t*>(a.out_bthd)[e] = (bf16_t)(a.scale * acc[i][j]);
                else
                    reinterpret_cast<float*>(a.out_bthd)[e] = a.scale * acc[i][j];
            }
    }
}

// Cotangents of one chunk's rows: dq, dk (Kq) and dv (Vd) for its 64 tokens
// from S_n (state before the chunk), D_{n+1} (cotangent after it) and the
// two masked decayed score matrices A (q.k) and B (dO.v), each output tile
// (64 tokens x 64 coordinates) as two tile GEMMs. Grid (N, H, B), 256 threads.
struct ChunkGradArgs {
    const float *q, *k, *v, *dO;  // head-major [B*H, Tp, Kq]; rows of Vd at vl
    RowsAt vl;                    // v's, dO's and dv's rows
    int oT;                       // vl.T of dO
    const float* g;               // [B, T, H]
    const float *S, *D;           // [B*H, N+1, Kq, Vd]: fp32, or bf16_t with sbf
    float *dq, *dk, *dv;          // head-major; dv at vl
    int dvbf;                     // dv's rows are bf16 (as v's)
    int B, T, Tp, H, Kq, Vd, N;
    float scale;
    int sbf;                      // S and D hold bf16 states
    int rbf;                      // v and dO hold bf16 rows
    int parts;                    // workgroups per chunk (chunk_parts)
};

template <bool MF, bool V4, bool SB, bool RB, int NT>
__global__ __launch_bounds__(256) void bw_chunk_kernel(ChunkGradArgs a) {
    using RK = std::conditional_t<V4, RowsK4, RowsK>;  // 16-byte row loads when aligned
    using RJ = std::conditional_t<V4, RowsJ4, RowsJ>;
    using SK = StateRowsK<SB, V4>;  // the states' rows
    using SJ = StateRowsJ<SB, V4>;
    using SE = std::conditional_t<SB, bf16_t, float>;
    using VK = StateRowsK<RB, V4>;  // v's and dO's rows
    using VJ = StateRowsJ<RB, V4>;
    using VE = std::conditional_t<RB, bf16_t, float>;
    __shared__ float sA[BC][BC + 1], sB[BC][BC + 1];
    // Output tiles of 64 NT columns: with NT = 2 each row block a product reads
    // (dO, v, k, and the other operands' rows) is read once per pair of tiles
    // (the kernel reads HBM at its rate: 222 -> 184 us at configuration 3)
    constexpr int NA = 4 * NT;
    __shared__ __align__(16) unsigned char sStage[NT == 2 ? STAGE2_BYTES : STAGE_BYTES];
    // (the row factors e^{G_t} and e^{G_last - G_t} are formed where used)
    __shared__ float sG[BC];
    const int tid = threadIdx.x, n = blockIdx.x, h = blockIdx.y, b = blockIdx.z / a.parts, part = blockIdx.z % a.parts;
    const int Kq = a.Kq, Vd = a.Vd, t0 = n * BC;
    const size_t bh = (size_t)b * a.H + h, ssz = (size_t)Kq * Vd;
    const float* q = a.q + (bh * a.Tp + t0) * Kq;
    const float* k = a.k + (bh * a.Tp + t0) * Kq;
    const size_t v_at = a.vl.at(b, h, t0);
    const VE* v = reinterpret_cast<const VE*>(a.v) + v_at;
    const VE* dO = reinterpret_cast<const VE*>(a.dO) + v_at;
    const int ldv = a.vl.ld, nv = a.vl.live(t0), no = RowsAt{0, 0, 0, a.oT}.live(t0);
    const SE* S = reinterpret_cast<const SE*>(a.S) + (bh * (a.N + 1) + n) * ssz;
    const SE* D = reinterpret_cast<const SE*>(a.D) + (bh * (a.N + 1) + n + 1) * ssz;
    if (tid < 64) {
        const float G = chunk_gam(a.g, b, h, a.T, a.H, n, tid);
        sG[tid] = G;
    }
    // The tiles of dq and dk (nq), then those of dv: this workgroup's are part,
    // part + parts, ... Each kind needs one of the two score matrices.
    const int nq = (Kq + BC * NT - 1) / (BC * NT), tiles = nq + (Vd + BC * NT - 1) / (BC * NT);
    const int last = part + (tiles - 1 - part) / a.parts * a.parts;
    if (last >= nq) chunk_scores<MF, V4>(q, Kq, BC, k, Kq, BC, Kq, sG, sStage, sA);
    if (part < nq) chunk_scores<MF, V4>(dO, ldv, no, v, ldv, nv, Vd, sG, sStage, sB);
    const float sc = a.scale;
    for (int u = part; u < tiles; u += a.parts) {
        float acc[NA][4] = {};
        if (u < nq) {
            const int d0 = BC * NT * u;
            // dq = scale (e^{G_t} dO_t S_n^T + B k)
            tile_gemm<MF, NT>(VK(dO, ldv, no, Vd), SK(S + (size_t)d0 * Vd, Vd, Kq - d0, Vd), Vd, sStage, acc);
            tile_scale_rows<NA>(acc, [&](int t) { return expf(sG[t]); });
            tile_gemm<MF, NT>(in_order([&](int i, int kk) { return sB[i][kk]; }), RJ(k + d0, Kq, BC, Kq - d0), BC, sStage, acc);
            tile_store<NA>(acc, a.dq + (bh * a.Tp + t0) * Kq, Kq, d0, sc);
            // dk = e^{G_last - G_s} v_s D_{n+1}^T + scale B^T q
#pragma unroll
            for (int x = 0; x < NA; x++)
#pragma unroll
                for (int y = 0; y < 4; y++) acc[x][y] = 0.f;
            tile_gemm<MF, NT>(VK(v, ldv, nv, Vd), SK(D + (size_t)d0 * Vd, Vd, Kq - d0, Vd), Vd, sStage, acc);
            tile_scale_rows<NA>(acc, [&](int t) { return expf(sG[BC - 1] - sG[t]); });
            tile_gemm<MF, NT>([&](int i, int kk) { return sc * sB[kk][i]; }, RJ(q + d0, Kq, BC, Kq - d0), BC, sStage, acc);
            tile_store<NA>(acc, a.dk + (bh * a.Tp + t0) * Kq, Kq, d0, 1.f);
        } else {
            const int d0 = BC * NT * (u - nq);
            // dv = e^{G_last - G_s} k_s D_{n+1} + scale A^T dO
            tile_gemm<MF, NT>(RK(k, Kq, BC, Kq), SJ(D + d0, Vd, Kq, Vd - d0), Kq, sStage, acc);
            tile_scale_rows<NA>(acc, [&](int t) { return expf(sG[BC - 1] - sG[t]); });
            tile_gemm<MF, NT>([&](int i, int kk) { return sc * sA[kk][i]; }, VJ(dO + d0, ldv, no, Vd - d0), BC, sStage, acc);
            const auto store_dv = [&](auto* dst) {
#pragma unroll
                for (int x = 0; x < NA; x++)
#pragma unroll
                    for (int y = 0; y < 4; y++) {
                        const int t = TileMap::row(x, y), c = d0 + TileMap::col(x, y);
                        if (c < Vd && t < nv) dst[(size_t)t * ldv + c] = (std::remove_reference_t<decltype(*dst)>)acc[x][y];
                    }
            };
            if (RB && a.dvbf)
                store_dv(reinterpret_cast<bf16_t*>(a.dv) + v_at);
            else
                store_dv(a.dv + v_at);
        }
    }
}

// The slot readout of fp32 calls for blocks of 32 rows of one head: z = U(lam)
// raw, l = z table^T, p = softmax(l), u = p table, weights = U(-lam) u; the two
// products as small GEMMs against the staged table on the fp32 matrix cores
// (mfma4 below). Grid (ceil(B Tp / (32 per_wg)), H), RO_FWD_THREADS threads: a
// workgroup stages the table once and takes per_wg blocks; the LDS holds one
// workgroup per CU, and its waves put several on each SIMD.

// With BF, x rounded to bf16: z, the table, p and the weights of the general
// forward's bf16 calls (its casts to the input dtype, ops/utils.py:779-882);
// the backward's recompute is unrounded.
template <bool BF>
__device__ __forceinline__ float bw_rnd(float x) {
    if constexpr (BF)
        return (float)(bf16_t)x;
    else
        return x;
}

// The readouts' block inputs, read from the buffers of all rows: fewer than 2^23
// of them (the general forward; 2^21 in the backward) of at most 128 floats, so
// regions of at most 2^32 - 2^15 bytes, past which a dead load's offset lies (in
// one with the top bit set it would reach into another row's values from 2^31
// bytes on).
constexpr uint32_t RO_DEAD = 0xfffff000u;

__device__ __forceinline__ float ro_load(bw_rsrc_t r, uint32_t off, bool live) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, live ? off : RO_DEAD, 0, 0));
}
__device__ __forceinline__ f32x2 ro_load2(bw_rsrc_t r, uint32_t off, bool live) {
    return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, live ? off : RO_DEAD, 0, 0));
}

constexpr int RO_LD = BWD_TABLE_M + 4;  // staged table and row rows, 16-byte aligned
constexpr int RO_FWD_THREADS = 1024;

__global__ __launch_bounds__(RO_FWD_THREADS) void bw_fwd_readout_kernel(const float* raw, const float* cs, const float* sn,
                                                             const float* table, int B, int Tp, int H, int M,
                                                             int per_wg, float* wts) {
    constexpr int TM = BWD_TABLE_M, LD = RO_LD, RB = 32, NT = RO_FWD_THREADS, NW = NT / 64, CPW = 16 / NW;
    static_assert(TM == 128 && (NW == 8 || NW == 16), "eight 16-wide tiles of slots, two of rows");
    __shared__ float sTab[TM * LD];  // rows R .. 127 and columns M .. 127 zero
    __shared__ float sZ[RB][LD], sP[RB][LD];
    __shared__ float sCs[RB][TM / 2], sSn[RB][TM / 2];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, h = blockIdx.y;
    const int lr = lane & 15, lk = lane >> 4;
    const int R = M - 1, P = M / 2, rows = B * Tp;
    for (int e = tid; e < TM * LD; e += NT) {
        const int r = e / LD, m = e % LD;
        sTab[e] = (r < R && m < M) ? table[((size_t)h * R + r) * M + m] : 0.f;
    }
    const auto row_of = [&](int rho) { return ((size_t)(rho / Tp) * H + h) * Tp + rho % Tp; };
    // wave wv: row tile it = wv & 1, column tiles CPW (wv >> 1) .. + CPW - 1 (of r, then of m)
    const int it = wv & 1, ct0 = CPW * (wv >> 1);
    // A block's inputs, element x of this thread = (row i, pair pr) = e / 64,
    // e % 64, e = tid + NT x: loaded one block ahead through buffer
    // resources, predicated through the offset (ro_load), so that no block
    // waits for its own loads.
    constexpr int NX = RB * (TM / 2) / NT;
    const int b_end = min(rows, (int)(blockIdx.x + 1) * per_wg * RB);
    const bw_rsrc_t rcs = bw_rsrc(cs, (size_t)rows * H * P), rsn = bw_rsrc(sn, (size_t)rows * H * P),
                    rraw = bw_rsrc(raw, (size_t)rows * H * M);  // every head's rows
    float nc[NX], ns[NX], nre[NX], nro[NX];
    const auto load_block = [&](int b0) {
#pragma unroll
        for (int x = 0; x < NX; x++) {
            const int e = tid + NT * x, i = e / (TM / 2), pr = e % (TM / 2), rho = b0 + i;
            const bool live = rho < b_end && pr < P;
            const uint32_t row = live ? (uint32_t)row_of(rho) : 0u;
            nc[x] = ro_load(rcs, (row * (uint32_t)P + (uint32_t)pr) * 4u, live);
            ns[x] = ro_load(rsn, (row * (uint32_t)P + (uint32_t)pr) * 4u, live);
            nre[x] = ro_load(rraw, (row * (uint32_t)M + 2u * (uint32_t)pr) * 4u, live);
            nro[x] = ro_load(rraw, (row * (uint32_t)M + 2u * (uint32_t)pr + 1u) * 4u, live);
        }
    };
    const int b_first = blockIdx.x * per_wg * RB;
    load_block(b_first);
    for (int b0 = b_first; b0 < b_end; b0 += RB) {
        __syncthreads();  // the table is staged; the previous block's tiles are done with
#pragma unroll
        for (int x = 0; x < NX; x++) {
            const int e = tid + NT * x, i = e / (TM / 2), pr = e % (TM / 2);
            const bool live = b0 + i < b_end && pr < P;
            const float c = live ? nc[x] : 1.f, s = ns[x];
            sCs[i][pr] = c;
            sSn[i][pr] = s;
            sZ[i][2 * pr] = c * nre[x] - s * nro[x];  // zero where !live
            sZ[i][2 * pr + 1] = s * nre[x] + c * nro[x];
        }
        load_block(b0 + RB);  // the next block (past the end: dead loads)
        __syncthreads();
        {  // logits l[i][r] = sum_m z[i][m] table[r][m]
            f32x4 acc[CPW];
#pragma unroll
            for (int t = 0; t < CPW; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int k0 = 0; k0 < TM; k0 += 4) {
                const float az = sZ[16 * it + lr][k0 + lk];
#pragma unroll
                for (int t = 0; t < CPW; t++) acc[t] = mfma4(az, sTab[(16 * (ct0 + t) + lr) * LD + k0 + lk], acc[t]);
            }
#pragma unroll
            for (int t = 0; t < CPW; t++)
#pragma unroll
                for (int q = 0; q < 4; q++) sP[16 * it + 4 * lk + q][16 * (ct0 + t) + lr] = acc[t][q];
        }
        __syncthreads();
        for (int i = wv; i < RB; i += NW) {
            const float l0 = lane < R ? sP[i][lane] : -INFINITY, l1 = lane + 64 < R ? sP[i][lane + 64] : -INFINITY;
            const float mx = bw_wave_max(fmaxf(l0, l1));
            const float e0 = lane < R ? expf(l0 - mx) : 0.f, e1 = lane + 64 < R ? expf(l1 - mx) : 0.f;
            const float inv = 1.f / bw_wave_sum(e0 + e1);
            sP[i][lane] = e0 * inv;
            sP[i][lane + 64] = e1 * inv;
        }
        __syncthreads();
        // u[i][m] = sum_r p[i][r] table[r][m] (p and the table zero at r >= R); the
        // weights' pair (2 pr, 2 pr + 1) sits in lanes (lr, lr ^ 1), swapped in by
        // quad_perm [1,0,3,2]
        f32x4 acc[CPW];
#pragma unroll
        for (int t = 0; t < CPW; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int k0 = 0; k0 < TM; k0 += 4) {
            const float ap = sP[16 * it + lr][k0 + lk];
#pragma unroll
            for (int t = 0; t < CPW; t++) acc[t] = mfma4(ap, sTab[(k0 + lk) * LD + 16 * (ct0 + t) + lr], acc[t]);
        }
        const bool odd = (lr & 1) != 0;
#pragma unroll
        for (int t = 0; t < CPW; t++) {
            const int m = 16 * (ct0 + t) + lr, pr = m >> 1;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float un = acc[t][q], ux = dpp_mov<0xB1>(un);
                const float ue = odd ? ux : un, uo = odd ? un : ux;
                const int i = 16 * it + 4 * lk + q, rho = b0 + i;
                if (rho < rows && pr < P) {
                    const float c = sCs[i][pr], s = sSn[i][pr];
                    wts[row_of(rho) * M + m] = odd ? -s * ue + c * uo : c * ue + s * uo;
                }
            }
        }
    }
}

// The readout and its adjoint for calls with bf16 operands, every product as
// split-bf16 products on v_mfma_f32_16x16x32_bf16 (each fp32 operand as a bf16
// high part and a bf16 remainder, lo_a hi_b + hi_a lo_b + hi_a hi_b: about 16
// mantissa bits; with BF, the general bf16 forward, the operands are bf16
// values and the products exact). Per block of 32 rows of a head (the formulas
// are those of bw_fwd_readout_kernel and bw_readout_kernel):
//   z (and du) as two bf16 parts into LDS; logits (and dp); softmax (and dl);
//   u (and dz); weights, or draw, the clock's and the gate's shares; dtable.
// Wave w of eight owns slots and coordinates 16 w .. + 15 of every product and
// holds the table's rows and columns for them as operand registers (64 with both parts), so that the table takes no
// LDS and no reads per block; its part of dtable stays in accumulators. The
// products are formed transposed, slots (coordinates) by rows: a lane then
// holds four neighbouring slots of one row, a row's reductions are three adds
// and two lane swaps, and a coordinate pair sits in one lane. Row maxima and
// sums cross the waves through LDS (8 floats per row and step). p and dl are
// kept twice, by rows (operands of u and dz) and by slots (of dtable), so that
// each operand is one 16-byte LDS read; du's and z's columns are gathered. Tp
// is a multiple of 64, so a block's rows are consecutive rows of one batch
// row, at one scalar base, and none is past the end. Grid (workgroups per
// head, H); a workgroup takes per_wg blocks (bwd_ro_per_wg).
// The adjoint's LDS (130 KB) holds one workgroup of eight waves per CU; sixteen
// waves at 128 registers would spill. 65536 rows of 128 slots on MI355X: the
// adjoint 76 us and the forward 40 us, where the table staged in LDS, sixteen
// waves and the adjoint's products on the fp32 matrix cores took 164 and 76;
// 16384 rows: 25 and 19 us, where they took 53 and 27. Products by rows instead
// of slots, with a division per row and sums over 16 lanes: 119 and 62, 48 and
// 30. Bound by the reads of p, dl, z and du from LDS and the vector ALU.
// Against 64 bits, over 12 inputs each of four shapes, the gradients are as far
// off as with the adjoint's products in fp32 (the largest error of a pass 1.0000
// to 1.0003 of it, the readout's gradient 1.0002): the bf16 states decide it.
constexpr int RO_LDB = BWD_TABLE_M + 8;    // bf16 row blocks [32][RO_LDB]
constexpr int RO_LDP = BWD_RO_BLOCK + 8;   // p and dl by slots [128][RO_LDP]
constexpr int RO_LDC = BWD_TABLE_M / 2 + 4;  // phases [32][RO_LDC]
constexpr int RO_MF_WAVES = 8;

// lane (lr, lg) gets X[r0 + lr][k0 + 8 lg .. + 7] of a row-major bf16 tile
template <int LD>
__device__ __forceinline__ bf16x8 ro_row(const bf16_t* X, int r0, int k0) {
    const int l = threadIdx.x & 63;
    return *reinterpret_cast<const bf16x8*>(X + (r0 + (l & 15)) * LD + k0 + 8 * (l >> 4));
}

// lane (lr, lg) gets X[8 lg + j][c0 + lr], j = 0..7, of a row-major bf16 tile
// (an operand of its transpose), as eight 2-byte LDS reads
__device__ __forceinline__ bf16x8 ro_col(const bf16_t* X, int c0) {
    const int l = threadIdx.x & 63;
    const bf16_t* p = X + 8 * (l >> 4) * RO_LDB + c0 + (l & 15);
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; e++) r[e] = p[e * RO_LDB];
    return r;
}

// c += A B over 32 k with both operands in two bf16 parts (ONE: in one, the
// remainders zero)
template <bool ONE>
__device__ __forceinline__ f32x4 mfma_split(const bf16x8& ah, const bf16x8& al, const bf16x8& bh, const bf16x8& bl,
                                            f32x4 c) {
    if constexpr (!ONE) {
        c = mfma_bf16(al, bh, c);
        c = mfma_bf16(ah, bl, c);
    }
    return mfma_bf16(ah, bh, c);
}

__device__ __forceinline__ bf16_t bf16_lo(float v) { return (bf16_t)(v - (float)(bf16_t)v); }

// Four floats as bf16 high parts and remainders.
__device__ __forceinline__ void bf16_split4(const f32x4& v, bf16x4& hi, bf16x4& lo) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
        hi[q] = (bf16_t)v[q];
        lo[q] = bf16_lo(v[q]);
    }
}

// Sum (max) over the four lanes l, l ^ 16, l ^ 32, l ^ 48, in each of them:
// permlane16_swap of a register with itself leaves lanes of 16-lane rows 0 and
// 1 (2 and 3) with both rows' values, permlane32_swap both halves'.
template <bool MX>
__device__ __forceinline__ float rows4_reduce(float x) {
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    auto w = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    uint32_t a = w[0], b = w[1];
    float fa = __builtin_bit_cast(float, a), fb = __builtin_bit_cast(float, b);
    u = __builtin_bit_cast(uint32_t, MX ? fmaxf(fa, fb) : fa + fb);
    w = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    a = w[0], b = w[1];
    fa = __builtin_bit_cast(float, a), fb = __builtin_bit_cast(float, b);
    return MX ? fmaxf(fa, fb) : fa + fb;
}

struct ReadoutGradArgs {
    const float *raw, *cs, *sn, *table, *dwts;  // head-major rows; table [H, M-1, M]
    float* wts;                                 // the forward's slot weights
    float *draw, *dtab;                         // dtab: [H, workgroups, (M-1) M]
    double *dlam, *dgq;                         // per row: the clock's share; z.dz + u.du
    int B, Tp, H, M;
    int per_wg;                                 // blocks of 32 rows per workgroup
};

template <bool ADJ, bool BF>
__global__ __launch_bounds__(64 * RO_MF_WAVES, ADJ ? 2 : 4) void bw_readout_mf_kernel(ReadoutGradArgs a) {
    static_assert(!(ADJ && BF), "the adjoint is unrounded");
    constexpr int TM = BWD_TABLE_M, RB = BWD_RO_BLOCK, LB = RO_LDB, KS = TM / 32, NT = 64 * RO_MF_WAVES;
    constexpr int RT = RB / 16, DT = TM / 16;  // row tiles and dtable slot tiles of a wave
    static_assert(TM == 16 * RO_MF_WAVES && RB == 32, "a 16-wide tile of slots per wave, two of rows");
    __shared__ __align__(16) bf16_t sZ[2][RB * LB], sP[2][RB * LB];                      // [part][row][m | slot]
    __shared__ __align__(16) bf16_t sDU[ADJ ? 2 : 1][ADJ ? RB * LB : 8], sDL[ADJ ? 2 : 1][ADJ ? RB * LB : 8];
    __shared__ __align__(16) bf16_t sPt[ADJ ? 2 : 1][ADJ ? TM * RO_LDP : 8], sDt[ADJ ? 2 : 1][ADJ ? TM * RO_LDP : 8];
    __shared__ __align__(16) float sCs[RB * RO_LDC], sSn[RB * RO_LDC];
    __shared__ __align__(16) float sMx[RB][8], sSum[RB][8], sSd[RB][8];
    __shared__ float sLam[RB][8], sGq[RB][8];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), h = blockIdx.y;
    const int lr = lane & 15, lg = lane >> 4, cw = wv;
    const int M = a.M, R = M - 1, P = M / 2, rows = a.B * a.Tp;
    const auto load2 = [](bw_rsrc_t r, uint32_t off, bool live) {
        return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off | (live ? 0u : BW_DEAD), 0, 0));
    };
    // the table's operands: rows r = 16 cw + lr (logits, dp) and columns m = 16 cw + lr (u, dz)
    bf16x8 trh[KS], trl[KS], tch[KS], tcl[KS];
    {
        const int mine = 16 * cw + lr;
        const bw_rsrc_t rt = bw_rsrc(a.table + (size_t)h * R * M, (size_t)R * M);
        const auto put = [](bf16x8& hi, bf16x8& lo, int e, float v) {
            v = bw_rnd<BF>(v);
            hi[e] = (bf16_t)v;
            lo[e] = bf16_lo(v);
        };
#pragma unroll
        for (int k = 0; k < KS; k++)
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const int kk = 32 * k + 8 * lg + e;  // even, as M is
                const f32x2 vr = load2(rt, (uint32_t)(mine * M + kk) * 4u, mine < R && kk < M);
                put(trh[k], trl[k], e, vr[0]);
                put(trh[k], trl[k], e + 1, vr[1]);
                put(tch[k], tcl[k], e, bw_load(rt, (uint32_t)(kk * M + mine) * 4u, kk < R && mine < M));
                put(tch[k], tcl[k], e + 1, bw_load(rt, (uint32_t)(kk * M + M + mine) * 4u, kk + 1 < R && mine < M));
            }
    }
    const int s0 = 16 * cw + 4 * lg;  // this lane's slots and coordinates s0 .. s0 + 3: pairs s0 / 2, s0 / 2 + 1
    float kappa[2];
#pragma unroll
    for (int j = 0; j < 2; j++) kappa[j] = s0 / 2 + j < P ? (float)(kTwoPiBw * (s0 / 2 + j) / R) : 0.f;
    f32x4 dacc[ADJ ? DT : 1];  // dtable rows 16 rt .. of column 16 cw + lr
#pragma unroll
    for (int rt = 0; rt < (ADJ ? DT : 1); rt++) dacc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
    // A block's inputs, element x of this thread = (row i, pair pr) = e / 64,
    // e % 64, e = tid + NT x: loaded one block ahead through buffer resources,
    // predicated through the offset (ro_load), so that no block waits for its
    // own loads.
    constexpr int NX = RB * (TM / 2) / NT;
    const int b_first = blockIdx.x * a.per_wg * RB, b_end = min(rows, b_first + a.per_wg * RB);
    const auto base_of = [&](int b0) { return ((size_t)(b0 / a.Tp) * a.H + h) * a.Tp + b0 % a.Tp; };
    const bw_rsrc_t rcs = bw_rsrc(a.cs, (size_t)rows * a.H * P), rsn = bw_rsrc(a.sn, (size_t)rows * a.H * P),
                    rraw = bw_rsrc(a.raw, (size_t)rows * a.H * M),
                    rdw = bw_rsrc(a.dwts, ADJ ? (size_t)rows * a.H * M : 0);
    const int pr_in = tid % (TM / 2), i_in = tid / (TM / 2);
    float nc[NX], ns[NX];
    f32x2 nr[NX], nd[NX];
    const auto load_block = [&](int b0) {
        const bool live = b0 < b_end && pr_in < P;
        const uint32_t row0 = (b0 < b_end ? (uint32_t)base_of(b0) : 0u) + (uint32_t)i_in;
#pragma unroll
        for (int x = 0; x < NX; x++) {
            const uint32_t at = ((row0 + (uint32_t)(NT / (TM / 2) * x)) * (uint32_t)P + (uint32_t)pr_in) * 4u;
            nc[x] = ro_load(rcs, at, live);
            ns[x] = ro_load(rsn, at, live);
            nr[x] = ro_load2(rraw, 2u * at, live);
            if constexpr (ADJ) nd[x] = ro_load2(rdw, 2u * at, live);
        }
    };
    load_block(b_first);
    for (int b0 = b_first; b0 < b_end; b0 += RB) {
        __syncthreads();  // the previous block's tiles are done with
#pragma unroll
        for (int x = 0; x < NX; x++) {
            const int i = i_in + NT / (TM / 2) * x;
            const float c = pr_in < P ? nc[x] : 1.f, s = ns[x];  // zero inputs past P
            sCs[i * RO_LDC + pr_in] = c;
            sSn[i * RO_LDC + pr_in] = s;
            const auto put2 = [&](bf16_t* hi, bf16_t* lo, float v0, float v1) {
                *reinterpret_cast<bf16x2*>(hi + i * LB + 2 * pr_in) = bf16x2{(bf16_t)v0, (bf16_t)v1};
                if constexpr (!BF) *reinterpret_cast<bf16x2*>(lo + i * LB + 2 * pr_in) = bf16x2{bf16_lo(v0), bf16_lo(v1)};
            };
            put2(sZ[0], sZ[1], bw_rnd<BF>(c * nr[x][0] - s * nr[x][1]), bw_rnd<BF>(s * nr[x][0] + c * nr[x][1]));
            if constexpr (ADJ) put2(sDU[0], sDU[1], c * nd[x][0] - s * nd[x][1], s * nd[x][0] + c * nd[x][1]);
        }
        load_block(b0 + RB);  // the next block (past the end: dead loads)
        __syncthreads();
        // logits l[r][i] = table[r] . z[i] and dp[r][i] = table[r] . du[i]: lane holds
        // slots s0 + q of row 16 t + lr
        f32x4 l[RT], dp[RT];
#pragma unroll
        for (int t = 0; t < RT; t++) {
            const int i0 = 16 * t;
            l[t] = dp[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KS; k++) {
                l[t] = mfma_split<BF>(trh[k], trl[k], ro_row<LB>(sZ[0], i0, 32 * k), ro_row<LB>(sZ[1], i0, 32 * k), l[t]);
                if constexpr (ADJ)
                    dp[t] = mfma_split<BF>(trh[k], trl[k], ro_row<LB>(sDU[0], i0, 32 * k), ro_row<LB>(sDU[1], i0, 32 * k), dp[t]);
            }
            // softmax over the slots (this wave's 16, then the eight waves), and dl = p (dp - p . dp)
#pragma unroll
            for (int q = 0; q < 4; q++) l[t][q] = s0 + q < R ? l[t][q] : -INFINITY;
            const float mx = rows4_reduce<true>(fmaxf(fmaxf(l[t][0], l[t][1]), fmaxf(l[t][2], l[t][3])));
            if (lg == 0) sMx[i0 + lr][cw] = mx;
        }
        __syncthreads();
        const auto across = [&](const float* v, bool mx) {  // over the waves, in wave order
            const f32x4 v0 = *reinterpret_cast<const f32x4*>(v), v1 = *reinterpret_cast<const f32x4*>(v + 4);
            if (mx) return fmaxf(fmaxf(fmaxf(v0[0], v0[1]), fmaxf(v0[2], v0[3])), fmaxf(fmaxf(v1[0], v1[1]), fmaxf(v1[2], v1[3])));
            return ((v0[0] + v0[1]) + (v0[2] + v0[3])) + ((v1[0] + v1[1]) + (v1[2] + v1[3]));
        };
#pragma unroll
        for (int t = 0; t < RT; t++) {
            const int i = 16 * t + lr;
            const float mx = across(sMx[i], true);
            float sum = 0.f, sd = 0.f;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                l[t][q] = s0 + q < R ? expf(l[t][q] - mx) : 0.f;
                sum += l[t][q];
                if constexpr (ADJ) sd += l[t][q] * dp[t][q];
            }
            sum = rows4_reduce<false>(sum);
            if (lg == 0) sSum[i][cw] = sum;
            if constexpr (ADJ) {
                sd = rows4_reduce<false>(sd);
                if (lg == 0) sSd[i][cw] = sd;
            }
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < RT; t++) {
            const int i = 16 * t + lr;
            const float inv = 1.f / across(sSum[i], false);
            const float pdp = ADJ ? across(sSd[i], false) * inv : 0.f;
            f32x4 p, d;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                p[q] = bw_rnd<BF>(l[t][q] * inv);
                d[q] = ADJ ? p[q] * (dp[t][q] - pdp) : 0.f;
            }
            bf16x4 hi, lo;
            bf16_split4(p, hi, lo);
            *reinterpret_cast<bf16x4*>(sP[0] + i * LB + s0) = hi;
            if constexpr (!BF) *reinterpret_cast<bf16x4*>(sP[1] + i * LB + s0) = lo;
            if constexpr (ADJ) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    sPt[0][(s0 + q) * RO_LDP + i] = hi[q];
                    sPt[1][(s0 + q) * RO_LDP + i] = lo[q];
                }
                bf16_split4(d, hi, lo);
                *reinterpret_cast<bf16x4*>(sDL[0] + i * LB + s0) = hi;
                *reinterpret_cast<bf16x4*>(sDL[1] + i * LB + s0) = lo;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    sDt[0][(s0 + q) * RO_LDP + i] = hi[q];
                    sDt[1][(s0 + q) * RO_LDP + i] = lo[q];
                }
            }
        }
        __syncthreads();
        // u[m][i] = sum_r table[r][m] p[i][r] and dz[m][i] = sum_r table[r][m] dl[i][r]
        // (p, dl and the table are zero at r >= R): lane holds coordinates s0 + q of row
        // 16 t + lr
        const size_t row0 = base_of(b0);
#pragma unroll
        for (int t = 0; t < RT; t++) {
            const int i0 = 16 * t, i = i0 + lr;
            f32x4 u = {0.f, 0.f, 0.f, 0.f}, dz = u;
#pragma unroll
            for (int k = 0; k < KS; k++) {
                u = mfma_split<BF>(tch[k], tcl[k], ro_row<LB>(sP[0], i0, 32 * k), ro_row<LB>(sP[1], i0, 32 * k), u);
                if constexpr (ADJ)
                    dz = mfma_split<BF>(tch[k], tcl[k], ro_row<LB>(sDL[0], i0, 32 * k), ro_row<LB>(sDL[1], i0, 32 * k), dz);
            }
            const f32x2 c2 = *reinterpret_cast<const f32x2*>(sCs + i * RO_LDC + s0 / 2);
            const f32x2 s2 = *reinterpret_cast<const f32x2*>(sSn + i * RO_LDC + s0 / 2);
            float* dst = (ADJ ? a.draw : a.wts) + (row0 + i) * M + s0;
            const f32x4 x = ADJ ? dz : u;
#pragma unroll
            for (int j = 0; j < 2; j++) {  // U(-lam) of a pair
                const float c = c2[j], s = s2[j], e = x[2 * j], o = x[2 * j + 1];
                if (s0 / 2 + j < P)
                    *reinterpret_cast<f32x2*>(dst + 2 * j) = f32x2{bw_rnd<BF>(c * e + s * o), bw_rnd<BF>(-s * e + c * o)};
            }
            if constexpr (ADJ) {
                // With z = U(lam) raw and du = U(lam) dweights, the clock's share
                // kappa_p [dz . dU(lam)/dlam raw + dweights . dU(-lam)/dlam u] is
                // kappa_p [(z_e dz_o - z_o dz_e) + (du_e u_o - du_o u_e)] (a rotation keeps
                // the 2-d cross product); the gate's is z . dz + u . du.
                const auto sum4 = [&](const bf16_t* hi, const bf16_t* lo) {
                    const bf16x4 vh = *reinterpret_cast<const bf16x4*>(hi + i * LB + s0);
                    const bf16x4 vl = *reinterpret_cast<const bf16x4*>(lo + i * LB + s0);
                    return f32x4{(float)vh[0] + (float)vl[0], (float)vh[1] + (float)vl[1], (float)vh[2] + (float)vl[2],
                                 (float)vh[3] + (float)vl[3]};
                };
                const f32x4 z = sum4(sZ[0], sZ[1]), du = sum4(sDU[0], sDU[1]);
                float v = 0.f, g = 0.f;  // zero past M
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const int e = 2 * j, o = 2 * j + 1;
                    v += kappa[j] * ((z[e] * dz[o] - z[o] * dz[e]) + (du[e] * u[o] - du[o] * u[e]));
                    g += (z[e] * dz[e] + du[e] * u[e]) + (z[o] * dz[o] + du[o] * u[o]);
                }
                v = rows4_reduce<false>(v);
                g = rows4_reduce<false>(g);
                if (lg == 0) {
                    sLam[i][cw] = v;
                    sGq[i][cw] = g;
                }
            }
        }
        if constexpr (ADJ) {
            // dtable[r][m] += sum_i p[i][r] du[i][m] + dl[i][r] z[i][m] over the block's rows
            const bf16x8 uh = ro_col(sDU[0], 16 * cw), ul = ro_col(sDU[1], 16 * cw);
            const bf16x8 zh = ro_col(sZ[0], 16 * cw), zl = ro_col(sZ[1], 16 * cw);
#pragma unroll
            for (int rt = 0; rt < DT; rt++) {
                const int r0 = 16 * rt;
                dacc[rt] = mfma_split<BF>(ro_row<RO_LDP>(sPt[0], r0, 0), ro_row<RO_LDP>(sPt[1], r0, 0), uh, ul, dacc[rt]);
                dacc[rt] = mfma_split<BF>(ro_row<RO_LDP>(sDt[0], r0, 0), ro_row<RO_LDP>(sDt[1], r0, 0), zh, zl, dacc[rt]);
            }
            __syncthreads();
            if (tid < RB) {  // the clock's and the gate's share per row, in wave order
                float v = sLam[tid][0], g = sGq[tid][0];
#pragma unroll
                for (int j = 1; j < 8; j++) v += sLam[tid][j], g += sGq[tid][j];
                a.dlam[row0 + tid] = v;
                a.dgq[row0 + tid] = g;
            }
        }
    }
    if constexpr (ADJ) {  // lane holds dtable rows 16 rt + 4 lg + q of column 16 cw + lr
        float* dst = a.dtab + ((size_t)h * gridDim.x + blockIdx.x) * R * M;
        const int m = 16 * cw + lr;
#pragma unroll
        for (int rt = 0; rt < DT; rt++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = 16 * rt + 4 * lg + q;
                if (r < R && m < M) dst[r * M + m] = dacc[rt][q];
            }
    }
}

// The slot-readout adjoint of fp32 calls for blocks of 32 rows of one head (z = U(lam) raw,
// l = table z, p = softmax(l), u = table^T p, weights = U(-lam) u):
//   du = U(lam) dweights, dp = table du, dl = p (dp - p.dp), dz = table^T dl,
//   draw = U(-lam) dz, dtable += p du^T + dl z^T, and the clock's share
//   dlam = sum_p kappa_p [dz . dU(lam)/dlam raw + dweights . dU(-lam)/dlam u]
// with kappa_p = 2 pi p / (M - 1). Every product over the block is a small
// GEMM against the head's table (staged once in LDS, rows RO_LD floats apart)
// on the fp32 matrix cores, v_mfma_f32_16x16x4_f32 (fp32 operands, fp32
// accumulation): lane l holds A[l % 16][l / 16] and B[l / 16][l % 16] of a
// 16 x 4 by 4 x 16 step and rows 4 (l / 16) .. + 3 of column l % 16 of the
// 16 x 16 result. Grid (workgroups per head, H), RO_ADJ_THREADS threads: a
// workgroup takes per_wg blocks of 32 rows (bwd_ro_per_wg) and keeps its part
// of dtable in the accumulators (wave w owns the 16 x 16 tiles (r, m) of
// columns m in 16 (w % 8) .. + 15 and rows r in 16 DRT (w / 8) .. + 16 DRT - 1,
// DRT = 64 / waves). The LDS holds one workgroup per CU; its waves put
// several on each SIMD, so that one wave's LDS reads overlap another's
// matrix-core steps.
constexpr int RO_BLK = BWD_RO_BLOCK;
constexpr int RO_ADJ_THREADS = 1024;

__global__ __launch_bounds__(RO_ADJ_THREADS) void bw_readout_kernel(ReadoutGradArgs a) {
    constexpr int TM = BWD_TABLE_M, LD = RO_LD, NT = RO_ADJ_THREADS, NW = NT / 64;
    constexpr int CPW = 16 / NW, DRT = 64 / NW;  // slot tiles per wave in the block products; dtable row tiles
    static_assert(NW == 8 || NW == 16, "two row tiles x eight slot tiles over the waves; eight dtable column tiles");
    static_assert(RO_BLK == 32 && TM == 128, "two 16-row tiles of rows, eight 16-wide tiles of slots");
    __shared__ float sTab[TM * LD];  // rows R .. 127 and columns M .. 127 zero
    __shared__ float sZ[RO_BLK][LD], sDU[RO_BLK][LD], sP[RO_BLK][LD], sDL[RO_BLK][LD];
    __shared__ float sCs[RO_BLK][TM / 2], sSn[RO_BLK][TM / 2];
    __shared__ double sLam[RO_BLK][NW / 2], sGq[RO_BLK][NW / 2];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, blk = blockIdx.x, h = blockIdx.y;
    const int lr = lane & 15, lk = lane >> 4;  // operand row / column and k of this lane
    const int M = a.M, R = M - 1, P = M / 2, RM = R * M;
    for (int e = tid; e < TM * LD; e += NT) {  // the table, zero beyond R x M
        const int r = e / LD, m = e % LD;
        sTab[e] = (r < R && m < M) ? a.table[((size_t)h * R + r) * M + m] : 0.f;
    }
    // GEMMs over the block: wave wv takes row tile it = wv & 1 and the column
    // tiles CPW (wv >> 1) .. + CPW - 1 of the logits (r) and of dz, u (m)
    const int it = wv & 1, ct0 = CPW * (wv >> 1), dm = wv & 7, dr0 = DRT * (wv >> 3);
    f32x4 dacc[DRT];  // dtable tiles (r tile dr0 + rt, m tile dm)
#pragma unroll
    for (int rt = 0; rt < DRT; rt++) dacc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int rows = a.B * a.Tp;
    // A block's inputs, element x of this thread = (row i, pair pr) = e / 64,
    // e % 64, e = tid + NT x: loaded one block ahead through buffer
    // resources, predicated through the offset (ro_load), so that no block
    // waits for its own loads.
    constexpr int NX = RO_BLK * (TM / 2) / NT;
    const int b_end = min(rows, (blk + 1) * a.per_wg * RO_BLK);
    const bw_rsrc_t rcs = bw_rsrc(a.cs, (size_t)rows * a.H * P), rsn = bw_rsrc(a.sn, (size_t)rows * a.H * P),
                    rraw = bw_rsrc(a.raw, (size_t)rows * a.H * M), rdw = bw_rsrc(a.dwts, (size_t)rows * a.H * M);
    float nc[NX], ns[NX], nre[NX], nro[NX], nde[NX], ndd[NX];
    const auto load_block = [&](int b0) {
#pragma unroll
        for (int x = 0; x < NX; x++) {
            const int e = tid + NT * x, i = e / (TM / 2), pr = e % (TM / 2), rho = b0 + i;
            const bool live = rho < b_end && pr < P;
            const uint32_t row = live ? (uint32_t)(((rho / a.Tp) * a.H + h) * a.Tp + rho % a.Tp) : 0u;
            nc[x] = ro_load(rcs, (row * (uint32_t)P + (uint32_t)pr) * 4u, live);
            ns[x] = ro_load(rsn, (row * (uint32_t)P + (uint32_t)pr) * 4u, live);
            nre[x] = ro_load(rraw, (row * (uint32_t)M + 2u * (uint32_t)pr) * 4u, live);
            nro[x] = ro_load(rraw, (row * (uint32_t)M + 2u * (uint32_t)pr + 1u) * 4u, live);
            nde[x] = ro_load(rdw, (row * (uint32_t)M + 2u * (uint32_t)pr) * 4u, live);
            ndd[x] = ro_load(rdw, (row * (uint32_t)M + 2u * (uint32_t)pr + 1u) * 4u, live);
        }
    };
    const int b_first = blk * a.per_wg * RO_BLK;
    load_block(b_first);
    for (int b0 = b_first; b0 < b_end; b0 += RO_BLK) {
        __syncthreads();  // the previous block's tiles are done with
        // z = U(lam) raw and du = U(lam) dweights
#pragma unroll
        for (int x = 0; x < NX; x++) {
            const int e = tid + NT * x, i = e / (TM / 2), pr = e % (TM / 2);
            const bool live = b0 + i < b_end && pr < P;
            const float c = live ? nc[x] : 1.f, s = ns[x];  // zero inputs where !live
            sCs[i][pr] = c;
            sSn[i][pr] = s;
            sZ[i][2 * pr] = c * nre[x] - s * nro[x];
            sZ[i][2 * pr + 1] = s * nre[x] + c * nro[x];
            sDU[i][2 * pr] = c * nde[x] - s * ndd[x];
            sDU[i][2 * pr + 1] = s * nde[x] + c * ndd[x];
        }
        load_block(b0 + RO_BLK);  // the next block (past the end: dead loads)
        __syncthreads();
        // logits l[i][r] = sum_m z[i][m] table[r][m] and dp[i][r] = sum_m du[i][m] table[r][m]
        {
            f32x4 accl[CPW], accd[CPW];
#pragma unroll
            for (int t = 0; t < CPW; t++) accl[t] = accd[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int k0 = 0; k0 < TM; k0 += 4) {
                const float az = sZ[16 * it + lr][k0 + lk], ad = sDU[16 * it + lr][k0 + lk];
#pragma unroll
                for (int t = 0; t < CPW; t++) {
                    const float bt = sTab[(16 * (ct0 + t) + lr) * LD + k0 + lk];
                    accl[t] = mfma4(az, bt, accl[t]);
                    accd[t] = mfma4(ad, bt, accd[t]);
                }
            }
#pragma unroll
            for (int t = 0; t < CPW; t++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    sP[16 * it + 4 * lk + q][16 * (ct0 + t) + lr] = accl[t][q];
                    sDL[16 * it + 4 * lk + q][16 * (ct0 + t) + lr] = accd[t][q];
                }
        }
        __syncthreads();
        // softmax and dl per row: wave wv takes rows wv, wv + NW, ...; lanes take slots lane, lane + 64
        for (int i = wv; i < RO_BLK; i += NW) {
            const float l0 = lane < R ? sP[i][lane] : -INFINITY, l1 = lane + 64 < R ? sP[i][lane + 64] : -INFINITY;
            const float mx = bw_wave_max(fmaxf(l0, l1));
            const float e0 = lane < R ? expf(l0 - mx) : 0.f, e1 = lane + 64 < R ? expf(l1 - mx) : 0.f;
            const float inv = 1.f / bw_wave_sum(e0 + e1);
            const float p0 = e0 * inv, p1 = e1 * inv;
            const float d0 = sDL[i][lane], d1 = sDL[i][lane + 64];
            const float pdp = bw_wave_sum(p0 * d0 + p1 * d1);
            sP[i][lane] = p0;
            sP[i][lane + 64] = p1;
            sDL[i][lane] = p0 * (d0 - pdp);
            sDL[i][lane + 64] = p1 * (d1 - pdp);
        }
        __syncthreads();
        // dz[i][m] = sum_r dl[i][r] table[r][m] and u[i][m] = sum_r p[i][r] table[r][m]
        // (p and dl are zero at r >= R, as is the table); then draw and the clock's share
        {
            f32x4 accz[CPW], accu[CPW];
#pragma unroll
            for (int t = 0; t < CPW; t++) accz[t] = accu[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int k0 = 0; k0 < TM; k0 += 4) {
                const float al = sDL[16 * it + lr][k0 + lk], ap = sP[16 * it + lr][k0 + lk];
#pragma unroll
                for (int t = 0; t < CPW; t++) {
                    const float bt = sTab[(k0 + lk) * LD + 16 * (ct0 + t) + lr];
                    accz[t] = mfma4(al, bt, accz[t]);
                    accu[t] = mfma4(ap, bt, accu[t]);
                }
            }
            // lane holds rows i = 16 it + 4 lk + q of column m = 16 (ct0 + t) + lr; the pair
            // (2 pr, 2 pr + 1) sits in lanes (lr, lr ^ 1), swapped in by quad_perm [1,0,3,2].
            // With z = U(lam) raw and du = U(lam) dweights, the clock's share
            // kappa_p [dz . dU(lam)/dlam raw + dweights . dU(-lam)/dlam u] is
            // kappa_p [(z_e dz_o - z_o dz_e) + (du_e u_o - du_o u_e)] (a rotation keeps
            // the 2-d cross product); the even lane of a pair forms it.
            const bool odd = (lr & 1) != 0;
            // (Every lane adds its column's z dz + u du to the gate's share.) Both in
            // double: bw_token_kernel's terms cancel most of them.
            double dl[4] = {0.0, 0.0, 0.0, 0.0}, gq[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int t = 0; t < CPW; t++) {
                const int m = 16 * (ct0 + t) + lr, pr = m >> 1;
                const double kappa = kTwoPiBw * pr / R;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float gz = accz[t][q], gx = dpp_mov<0xB1>(gz);
                    const float gu = accu[t][q], ux = dpp_mov<0xB1>(gu);
                    const float zm = sZ[16 * it + 4 * lk + q][m], dm = sDU[16 * it + 4 * lk + q][m];
                    const float zx = dpp_mov<0xB1>(zm), dx = dpp_mov<0xB1>(dm);
                    gq[q] += (double)zm * gz + (double)dm * gu;  // zero past M and past the last row
                    const float ge = odd ? gx : gz, go = odd ? gz : gx, ue = odd ? ux : gu, uo = odd ? gu : ux;
                    const int i = 16 * it + 4 * lk + q, rho = b0 + i;
                    if (rho < rows && pr < P) {
                        const size_t row = ((size_t)(rho / a.Tp) * a.H + h) * a.Tp + rho % a.Tp;
                        const float c = sCs[i][pr], s = sSn[i][pr];
                        a.draw[row * M + m] = odd ? -s * ge + c * go : c * ge + s * go;
                        if (!odd)
                            dl[q] += kappa * (((double)zm * go - (double)zx * ge) + ((double)dm * uo - (double)dx * ue));
                    }
                }
            }
            // the row's share over this wave's 16 lanes (its column tiles summed above,
            // in tile order), then the waves of the row tile in wave order
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const double v = wave_sum<16>(dl[q]), g = wave_sum<16>(gq[q]);
                if (lr == 0) {
                    sLam[16 * it + 4 * lk + q][wv >> 1] = v;
                    sGq[16 * it + 4 * lk + q][wv >> 1] = g;
                }
            }
        }
        __syncthreads();
        if (tid < RO_BLK && b0 + tid < rows) {  // the clock's and the gate's share per row
            const int rho = b0 + tid;
            double v = sLam[tid][0], g = sGq[tid][0];
#pragma unroll
            for (int j = 1; j < NW / 2; j++) v += sLam[tid][j], g += sGq[tid][j];
            const size_t row = ((size_t)(rho / a.Tp) * a.H + h) * a.Tp + rho % a.Tp;
            a.dlam[row] = v;
            a.dgq[row] = g;
        }
        // dtable[r][m] += sum_i p[i][r] du[i][m] + dl[i][r] z[i][m] over the block's rows,
        // each block's sum added to the workgroup's (one chain over all of its rows
        // left the readout's gradient 2 to 3% further off at two blocks)
        f32x4 dblk[DRT];
#pragma unroll
        for (int rt = 0; rt < DRT; rt++) dblk[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int k0 = 0; k0 < RO_BLK; k0 += 4) {
            const float bu = sDU[k0 + lk][16 * dm + lr], bz = sZ[k0 + lk][16 * dm + lr];
#pragma unroll
            for (int rt = 0; rt < DRT; rt++) {
                const float ap = sP[k0 + lk][16 * (dr0 + rt) + lr], al = sDL[k0 + lk][16 * (dr0 + rt) + lr];
                dblk[rt] = mfma4(ap, bu, dblk[rt]);
                dblk[rt] = mfma4(al, bz, dblk[rt]);
            }
        }
#pragma unroll
        for (int rt = 0; rt < DRT; rt++) dacc[rt] += dblk[rt];
    }
    // lane holds dtable rows 16 (dr0 + rt) + 4 lk + q of column 16 dm + lr
    float* dst = a.dtab + ((size_t)h * gridDim.x + blk) * RM;
#pragma unroll
    for (int rt = 0; rt < DRT; rt++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r = 16 * (dr0 + rt) + 4 * lk + q, m = 16 * dm + lr;
            if (r < R && m < M) dst[r * M + m] = dacc[rt][q];
        }
}

// The readout and its adjoint for 128 < M <= 256 slots, where a head's table
// (up to 255 x 256 fp32) does not fit in LDS beside the row blocks: every
// product is a 64 x 64 fp32 tile GEMM (tile_gemm_fma) that streams the
// table from memory, and the softmax and its adjoint run per row between
// them. Token rows rho of head h are the B Tp rows (b, h, t), rho = b Tp + t,
// at head-major row ((b H + h) Tp + t); X_lam(rho)[m] is U(lam) x (pairs
// rotated by the row's phases, as z = U(lam) raw and du = U(lam) dweights).
// Per-row intermediates have MW = 256 columns.
constexpr int BW_WIDE_MW = BWD_WIDE_MW;        // columns of the wide path's per-row buffers
constexpr int BW_WIDE_SPLIT = BWD_WIDE_SPLIT;  // token rows per dtable partial
constexpr int BW_WIDE_CT = BW_WIDE_MW / BC;    // column tiles of a row (the clock's partials)

struct WideArgs {
    const float *raw, *cs, *sn, *table, *dwts;  // head-major rows; table [H, M-1, M]
    float *lg, *dl;                             // [B H Tp, MW]: logits then p; dp then dl
    float *wts, *draw, *dlp;                    // dlp [B H Tp, 2 BW_WIDE_CT]: the clock's and the gate's partials
    double *dlam, *dgq;
    float* dtab;                                // [H, splits, (M-1) M]
    int B, Tp, H, M, splits;
    int bf;                                     // forward: round z, the table, p and the weights to bf16
};

__device__ __forceinline__ float wide_rnd(const WideArgs& a, float x) { return a.bf ? (float)(bf16_t)x : x; }

__device__ __forceinline__ size_t wide_row(const WideArgs& a, int h, int rho) {
    return ((size_t)(rho / a.Tp) * a.H + h) * a.Tp + rho % a.Tp;
}

// Element m of U(lam) x for head-major row `row` (x = raw or dweights).
__device__ __forceinline__ float wide_rot(const WideArgs& a, const float* x, size_t row, int m) {
    const int P = a.M / 2, pr = m >> 1;
    const float c = a.cs[row * P + pr], s = a.sn[row * P + pr];
    const float e = x[row * a.M + 2 * pr], o = x[row * a.M + 2 * pr + 1];
    return (m & 1) ? s * e + c * o : c * e - s * o;
}

// out[row][r] = sum_m X_lam(rho)[m] table[h][r][m] for a 64-row block and 64
// table rows (X = raw: the logits into lg; X = dweights: dp into dl).
// Grid (ceil(B Tp / 64), ceil((M - 1) / 64), H).
template <bool ADJ>
__global__ __launch_bounds__(256) void bw_wide_logits_kernel(WideArgs a) {
    __shared__ __align__(16) unsigned char sStage[STAGE_BYTES];
    const int rho0 = blockIdx.x * BC, r0 = blockIdx.y * BC, h = blockIdx.z;
    const int M = a.M, R = M - 1, rows = a.B * a.Tp;
    const float* x = ADJ ? a.dwts : a.raw;
    const float* tb = a.table + (size_t)h * R * M;
    float acc[4][4] = {};
    tile_gemm_fma<true>(
        [&](int i, int m) {
            return rho0 + i < rows ? wide_rnd(a, wide_rot(a, x, wide_row(a, h, rho0 + i), m)) : 0.f;
        },
        [&](int m, int j) { return r0 + j < R ? wide_rnd(a, tb[(size_t)(r0 + j) * M + m]) : 0.f; }, M, sStage, acc);
    float* out = ADJ ? a.dl : a.lg;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int rho = rho0 + FmaMap::row(i, 0);
        if (rho >= rows) continue;
        const size_t row = wide_row(a, h, rho);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = r0 + FmaMap::col(i, j);
            if (r < R) out[row * BW_WIDE_MW + r] = acc[i][j];
        }
    }
}

// Per row, one wave: p = softmax(logits) over the R = M - 1 slots into lg;
// ADJ: dl = p (dp - p.dp) into dl (p already in lg). Grid ceil(B H Tp / 4).
template <bool ADJ>
__global__ __launch_bounds__(256) void bw_wide_softmax_kernel(WideArgs a) {
    const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, R = a.M - 1;
    if (row >= (size_t)a.B * a.H * a.Tp) return;
    float* lg = a.lg + row * BW_WIDE_MW;
    float v[4];
    if (!ADJ) {
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = lane + 64 * i;
            v[i] = r < R ? lg[r] : -INFINITY;
            mx = fmaxf(mx, v[i]);
        }
        mx = bw_wave_max(mx);
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = lane + 64 * i < R ? expf(v[i] - mx) : 0.f;
            sum += v[i];
        }
        const float inv = 1.f / bw_wave_sum(sum);
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (lane + 64 * i < R) lg[lane + 64 * i] = wide_rnd(a, v[i] * inv);
    } else {
        float* dl = a.dl + row * BW_WIDE_MW;
        float pv[4], pdp = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = lane + 64 * i;
            pv[i] = r < R ? lg[r] : 0.f;
            v[i] = r < R ? dl[r] : 0.f;
            pdp += pv[i] * v[i];
        }
        pdp = bw_wave_sum(pdp);
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (lane + 64 * i < R) dl[lane + 64 * i] = pv[i] * (v[i] - pdp);
    }
}

// u = p table for a 64-row block and 64 columns (m0 ..), then
//   forward: weights = U(-lam) u into wts;
//   ADJ: dz = dl table as well; draw = U(-lam) dz, and the clock's share of
//   the block's pairs, kappa_p [(z_e dz_o - z_o dz_e) + (du_e u_o - du_o u_e)],
//   and the gate's, z.dz + u.du, each summed over the tile's pairs in column
//   order into dlp[row][m0 / 64] and dlp[row][BW_WIDE_CT + m0 / 64].
// Grid (ceil(B Tp / 64), ceil(M / 64), H).
template <bool ADJ>
__global__ __launch_bounds__(256) void bw_wide_u_kernel(WideArgs a) {
    __shared__ __align__(16) unsigned char sStage[STAGE_BYTES];
    __shared__ float sPart[BC][17], sGate[BC][17];
    const int tid = threadIdx.x, rho0 = blockIdx.x * BC, m0 = blockIdx.y * BC, h = blockIdx.z;
    const int M = a.M, R = M - 1, P = M / 2, rows = a.B * a.Tp;
    const float* tb = a.table + (size_t)h * R * M;
    const auto tab = [&](int r, int j) { return m0 + j < M ? wide_rnd(a, tb[(size_t)r * M + m0 + j]) : 0.f; };
    float u[4][4] = {}, dz[4][4] = {};
    tile_gemm_fma<false>(
        [&](int i, int r) { return rho0 + i < rows ? a.lg[wide_row(a, h, rho0 + i) * BW_WIDE_MW + r] : 0.f; }, tab, R,
        sStage, u);
    if (ADJ)
        tile_gemm_fma<false>(
            [&](int i, int r) { return rho0 + i < rows ? a.dl[wide_row(a, h, rho0 + i) * BW_WIDE_MW + r] : 0.f; },
            tab, R, sStage, dz);
    const int cg = tid & 15;  // this thread's four columns m0 + 4 cg ..: pairs (m0 + 4 cg) / 2 and + 1
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int ri = FmaMap::row(i, 0), rho = rho0 + ri;
        float dls = 0.f, gqs = 0.f;
        if (rho < rows) {
            const size_t row = wide_row(a, h, rho);
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
                const int m = m0 + FmaMap::col(i, j), pr = m >> 1;
                if (pr >= P) continue;
                const float c = a.cs[row * P + pr], s = a.sn[row * P + pr];
                if (!ADJ) {
                    a.wts[row * M + m] = wide_rnd(a, c * u[i][j] + s * u[i][j + 1]);
                    a.wts[row * M + m + 1] = wide_rnd(a, -s * u[i][j] + c * u[i][j + 1]);
                } else {
                    const float ge = dz[i][j], go = dz[i][j + 1], ue = u[i][j], uo = u[i][j + 1];
                    a.draw[row * M + m] = c * ge + s * go;
                    a.draw[row * M + m + 1] = -s * ge + c * go;
                    const float ze = wide_rot(a, a.raw, row, m), zo = wide_rot(a, a.raw, row, m + 1);
                    const float de = wide_rot(a, a.dwts, row, m), dd = wide_rot(a, a.dwts, row, m + 1);
                    dls += (float)(kTwoPiBw * pr / R) * ((ze * go - zo * ge) + (de * uo - dd * ue));
                    gqs += (ze * ge + zo * go) + (de * ue + dd * uo);
                }
            }
        }
        if (ADJ) sPart[ri][cg] = dls, sGate[ri][cg] = gqs;
    }
    if (ADJ) {
        __syncthreads();
        if (tid < BC && rho0 + tid < rows) {
            float t = 0.f, u2 = 0.f;
            for (int g = 0; g < 16; g++) t += sPart[tid][g], u2 += sGate[tid][g];
            float* dst = a.dlp + wide_row(a, h, rho0 + tid) * 2 * BW_WIDE_CT + blockIdx.y;
            dst[0] = t;
            dst[BW_WIDE_CT] = u2;
        }
    }
}

// The readout's share of the clock and gate cotangents: the column tiles'
// partials in order. One thread per head-major row.
__global__ __launch_bounds__(256) void bw_wide_dlam_kernel(WideArgs a) {
    const size_t row = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (row >= (size_t)a.B * a.H * a.Tp) return;
    const int nt = (a.M + BC - 1) / BC;
    float t = 0.f, g = 0.f;
    for (int c = 0; c < nt; c++) t += a.dlp[row * 2 * BW_WIDE_CT + c], g += a.dlp[row * 2 * BW_WIDE_CT + BW_WIDE_CT + c];
    a.dlam[row] = t;
    a.dgq[row] = g;
}

// dtable[h][r][m] partial over token rows [split BW_WIDE_SPLIT, + BW_WIDE_SPLIT):
// sum_rho p[rho][r] du[rho][m] + dl[rho][r] z[rho][m], for 64 table rows and
// 64 columns. Grid (ceil((M - 1) / 64), ceil(M / 64), H splits).
__global__ __launch_bounds__(256) void bw_wide_dtable_kernel(WideArgs a) {
    __shared__ __align__(16) unsigned char sStage[STAGE_BYTES];
    const int r0 = blockIdx.x * BC, m0 = blockIdx.y * BC, h = blockIdx.z / a.splits, sp = blockIdx.z % a.splits;
    const int M = a.M, R = M - 1, rows = a.B * a.Tp, k0 = sp * BW_WIDE_SPLIT;
    const int Kd = min(BW_WIDE_SPLIT, rows - k0);
    float acc[4][4] = {};
    tile_gemm_fma<false>(
        [&](int i, int k) { return r0 + i < R ? a.lg[wide_row(a, h, k0 + k) * BW_WIDE_MW + r0 + i] : 0.f; },
        [&](int k, int j) { return m0 + j < M ? wide_rot(a, a.dwts, wide_row(a, h, k0 + k), m0 + j) : 0.f; }, Kd,
        sStage, acc);
    tile_gemm_fma<false>(
        [&](int i, int k) { return r0 + i < R ? a.dl[wide_row(a, h, k0 + k) * BW_WIDE_MW + r0 + i] : 0.f; },
        [&](int k, int j) { return m0 + j < M ? wide_rot(a, a.raw, wide_row(a, h, k0 + k), m0 + j) : 0.f; }, Kd,
        sStage, acc);
    float* dst = a.dtab + ((size_t)h * a.splits + sp) * R * M;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = r0 + FmaMap::row(i, j), m = m0 + FmaMap::col(i, j);
            if (r < R && m < M) dst[(size_t)r * M + m] = acc[i][j];
        }
}

// Per chunk of (b, h): the write vector's cotangents (w = beta a(lam), a[2p] =
// s_p cos theta_p, a[2p+1] = -s_p sin theta_p, dw = the pass-1 value cotangent
// + the pass-2 key cotangent): dbeta = dw . a and dlam = beta dw . da/dlam +
// the readout's share; and the gate cotangent of both passes, dL/dG_t = dgq_t -
// beta_t dbeta_t (the header's identities), plus <D_{n+1}, S_{n+1}> at the
// chunk's last token, then the in-chunk reverse cumsum. Grid (N, B*H), 256
// threads: wave w forms rows TG_U at a time with its lanes across the pairs,
// then wave 0 scans. Bound by HBM: dw_1, dw_2 and the phases, 100 MB at 65536
// rows of 128 slots, 23 us; reading the rows of q, k and their cotangents for
// the dot products themselves it took 104 us (470 MB).
// A: the accumulator of the gate's and the clock's terms, which cancel those of
// the readout in part: float for bf16 calls, double for fp32 ones. Against 64
// bits, over 30 inputs each of seven fp32 shapes, dg's error is 0.89 to 0.96 of
// what the rows' dot products left (in float 0.98 to 1.04 of it), ddelta's 0.84
// to 0.99 of that in float.
struct TokenGradArgs {
    const float *dw1, *dw2;              // [.., M]
    const float *cs, *sn;                // [.., M/2]
    const float *bnd1, *bnd2;            // [B*H, nt, N]
    const double* dgq;                   // [B*H, Tp]: q.dq of both passes
    const float* beta;                   // [B, T, H]
    double* dlam;                        // [B*H, Tp]: in, the readout's share; out, the total
    float *dg, *dbeta;                   // [B, T, H]
    int B, T, Tp, H, M, N, nt1, nt2;
};
constexpr int TG_U = 8;  // rows whose loads a wave has in flight

template <class A>
__global__ __launch_bounds__(256) void bw_token_kernel(TokenGradArgs a) {
    __shared__ A sdB[BC], sdL[BC], sBnd;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int n = blockIdx.x, bh = blockIdx.y, b = bh / a.H, h = bh % a.H;
    const int M = a.M, P = M / 2, R = M - 1;
    // the write vector's per-pair factors: sqrt(1/R) for p = 0, sqrt(2/R) after;
    // the phase derivative's 2 pi p / R for the lane's pairs p = lane, lane + 64
    const A sp0 = (A)sqrt(1.0 / R), sp1 = (A)sqrt(2.0 / R);
    const A kp[2] = {(A)(kTwoPiBw * lane / R), (A)(kTwoPiBw * (lane + 64) / R)};
    if (wv == 3) {  // the chunk's boundary terms of both passes
        A x = 0;
        for (int i = lane; i < a.nt1; i += 64) x += a.bnd1[((size_t)bh * a.nt1 + i) * a.N + n];
        for (int i = lane; i < a.nt2; i += 64) x += a.bnd2[((size_t)bh * a.nt2 + i) * a.N + n];
        x = wave_sum(x);
        if (lane == 0) sBnd = x;
    }
    for (int i0 = 16 * wv; i0 < 16 * wv + 16; i0 += TG_U) {
        A db[TG_U], dl[TG_U];
        const size_t row0 = (size_t)bh * a.Tp + n * BC + i0;
#pragma unroll
        for (int u = 0; u < TG_U; u++) db[u] = dl[u] = 0;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int p = lane + 64 * c;
            if (64 * c >= P) break;
            const int pp = p < P ? p : P - 1;  // lanes past the last pair read it and drop it
            f32x2 d2[TG_U], d1[TG_U];
            float cs[TG_U], sn[TG_U];
#pragma unroll
            for (int u = 0; u < TG_U; u++) {
                const size_t e = (row0 + u) * M + 2 * pp, f = (row0 + u) * P + pp;
                d2[u] = *reinterpret_cast<const f32x2*>(a.dw2 + e);
                d1[u] = *reinterpret_cast<const f32x2*>(a.dw1 + e);
                cs[u] = a.cs[f];
                sn[u] = a.sn[f];
            }
            const A sp = p >= P ? (A)0 : p == 0 ? sp0 : sp1;
#pragma unroll
            for (int u = 0; u < TG_U; u++) {
                const A we = (A)d1[u][0] + d2[u][0], wo = (A)d1[u][1] + d2[u][1];
                if (p < P) {
                    db[u] = fma(sp, we * cs[u] - wo * sn[u], db[u]);
                    dl[u] = fma(sp * kp[c], -we * sn[u] - wo * cs[u], dl[u]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < TG_U; u++) {
            const A bb = wave_sum(db[u]), ll = wave_sum(dl[u]);
            if (lane == 0) {
                sdB[i0 + u] = bb;
                sdL[i0 + u] = ll;
            }
        }
    }
    __syncthreads();
    if (wv != 0) return;
    const int t = n * BC + lane;
    const size_t row = (size_t)bh * a.Tp + t;
    const float bt = t < a.T ? a.beta[((size_t)b * a.T + t) * a.H + h] : 0.f;
    A x = fma((A)-bt, sdB[lane], (A)a.dgq[row]);
    if (lane == BC - 1) x += sBnd;
    for (int o = 1; o < 64; o <<= 1) {
        const A y = __shfl_down(x, o);
        if (lane + o < 64) x += y;
    }
    a.dlam[row] = fma((A)bt, sdL[lane], (A)a.dlam[row]);
    if (t < a.T) {
        a.dg[((size_t)b * a.T + t) * a.H + h] = (float)x;
        a.dbeta[((size_t)b * a.T + t) * a.H + h] = (float)sdB[lane];
    }
}

// ddelta_s = sum_{t >= s} dlam_t + dclock (lam_t = clock0 + sum_{s <= t}
// delta_s; the final clock is clock0 + sum delta), dclock0 = sum_t dlam_t +
// dclock, in double. One wave per (b, h): each lane sums a run of tokens, the
// runs' suffix sums cross the lanes.
__global__ __launch_bounds__(64) void bw_clock_kernel(const double* dlam, const float* d_clock, int B, int T, int Tp,
                                                      int H, float* ddelta, float* dclock0) {
    const int bh = blockIdx.x, b = bh / H, h = bh % H, lane = threadIdx.x;
    const int per = (Tp + 63) / 64, t0 = lane * per, t1 = min(t0 + per, Tp);
    // tokens t, t - 1, .. of the run, zero before t0: CLOCK_U loads in flight
    // for each part of a lane's serial sum
    constexpr int CLOCK_U = 16;
    const auto fetch = [&](int t, double* v) {
#pragma unroll
        for (int u = 0; u < CLOCK_U; u++) v[u] = dlam[(size_t)bh * Tp + max(min(t, Tp - 1) - u, 0)];
#pragma unroll
        for (int u = 0; u < CLOCK_U; u++) v[u] = t - u >= t0 ? v[u] : 0.0;
    };
    double v[CLOCK_U];
    double s = 0.0;
    for (int t = t1 - 1; t >= t0; t -= CLOCK_U) {
        fetch(t, v);
#pragma unroll
        for (int u = 0; u < CLOCK_U; u++) s += v[u];
    }
    double suf = s;  // sum over this lane's run and every later lane's
    for (int o = 1; o < 64; o <<= 1) {
        const double y = __shfl_down(suf, o);
        if (lane + o < 64) suf += y;
    }
    const double extra = d_clock ? (double)d_clock[bh] : 0.0;
    double run = suf - s + extra;  // the later lanes' sum
    for (int t = t1 - 1; t >= t0; t -= CLOCK_U) {
        fetch(t, v);
#pragma unroll
        for (int u = 0; u < CLOCK_U; u++) {
            run += v[u];
            if (t - u >= t0 && t - u < T) ddelta[((size_t)b * T + t - u) * H + h] = (float)run;
        }
    }
    if (dclock0 && lane == 0) dclock0[bh] = (float)(suf + extra);
}

// RMS-norm adjoint of rows x [B, T, H, D] (x_hat = x rs w, rs = (mean x^2 +
// eps)^-1/2): dx = rs w dx_hat - rs^3 / D (sum_i x_i w_i dx_hat_i) x, and
// per block the partial dw = sum_rows dx_hat x rs. A workgroup takes 64 rows
// (16 per wave, in order), lanes own coordinates j = lane + 64 jj.
template <bool BF, int NJ>
__global__ __launch_bounds__(256) void bw_norm_kernel(const void* x, const float* w, const float* rs,
                                                      const float* dxh, int B, int T, int Tp, int H, int D, void* dx,
                                                      float* dw_part) {
    // Lane l holds columns l + 64 jj (jj < NJ, NJ 64 >= D); the global
    // accesses go through buffer resources over one row, columns past D
    // predicated through the offset (no branch among the loads), and a wave
    // takes its rows in groups of RB: every load of a group is issued before
    // the first row's arithmetic, so the group waits for memory once.
    constexpr int ES = BF ? 2 : 4;
    constexpr int RPW = BWD_NORM_ROWS / 4;                   // rows per wave
    constexpr int RB = 32 / NJ < RPW ? (32 / NJ > 0 ? 32 / NJ : 1) : RPW;
    static_assert(RPW % RB == 0, "whole groups");
    __shared__ float sdw[4][NJ * 64];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, blk = blockIdx.x;
    const int total = B * T * H;
    float dwa[NJ], wj[NJ];
    const bw_rsrc_t rw = bw_rsrc(w, (size_t)D);
#pragma unroll
    for (int jj = 0; jj < NJ; jj++) {
        dwa[jj] = 0.f;
        wj[jj] = bw_load(rw, (uint32_t)(lane + 64 * jj) * 4u, lane + 64 * jj < D);
    }
    const int row0 = blk * BWD_NORM_ROWS + wv * RPW;
    for (int g = 0; g < RPW; g += RB) {
        float xv[RB][NJ], dv[RB][NJ], r[RB];
        bool live[RB];
#pragma unroll
        for (int k = 0; k < RB; k++) {
            const int row = row0 + g + k;
            live[k] = row < total;
            // (the row and its coordinates through readfirstlane: in vector
            // registers, every buffer access built on them would become a
            // waterfall loop)
            const int rr = __builtin_amdgcn_readfirstlane(live[k] ? row : 0);
            const int h = __builtin_amdgcn_readfirstlane(rr % H), t = __builtin_amdgcn_readfirstlane((rr / H) % T),
                      b = __builtin_amdgcn_readfirstlane(rr / (H * T));
            const size_t hm = ((size_t)b * H + h) * Tp + t;
            const bw_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<char*>(reinterpret_cast<const char*>(x)) + (size_t)rr * D * ES, (short)0, live[k] ? D * ES : 0,
                0x00020000);
            const bw_rsrc_t rd = bw_rsrc(dxh + hm * D, live[k] ? (size_t)D : 0);
#pragma unroll
            for (int jj = 0; jj < NJ; jj++) {
                const int j = lane + 64 * jj;
                const uint32_t dead = j < D ? 0u : BW_DEAD;
                if constexpr (BF)
                    xv[k][jj] = (float)__builtin_bit_cast(
                        bf16_t, (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(rx, ((uint32_t)j * 2u) | dead, 0, 0));
                else
                    xv[k][jj] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, ((uint32_t)j * 4u) | dead, 0, 0));
                dv[k][jj] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, ((uint32_t)j * 4u) | dead, 0, 0));
            }
            r[k] = bw_load(bw_rsrc(rs + hm, 1), 0u, live[k]);
        }
#pragma unroll
        for (int k = 0; k < RB; k++) {
            const int row = row0 + g + k;
            float sum = 0.f;
#pragma unroll
            for (int jj = 0; jj < NJ; jj++) {
                sum = fmaf(xv[k][jj] * wj[jj], dv[k][jj], sum);
                dwa[jj] = fmaf(dv[k][jj] * xv[k][jj], r[k], dwa[jj]);  // zero for a row past the end
            }
            const float cr = r[k] * r[k] * r[k] * bw_wave_sum(sum) / (float)D;
            const bw_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<char*>(dx) + (size_t)(live[k] ? row : 0) * D * ES,
                                                                   (short)0, live[k] ? D * ES : 0, 0x00020000);
#pragma unroll
            for (int jj = 0; jj < NJ; jj++) {
                const int j = lane + 64 * jj;
                const uint32_t dead = j < D ? 0u : BW_DEAD;
                const float o = r[k] * wj[jj] * dv[k][jj] - cr * xv[k][jj];
                if constexpr (BF)
                    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, (bf16_t)o), ro,
                                                          ((uint32_t)j * 2u) | dead, 0, 0);
                else
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, o), ro, ((uint32_t)j * 4u) | dead, 0, 0);
            }
        }
    }
#pragma unroll
    for (int jj = 0; jj < NJ; jj++) sdw[wv][lane + 64 * jj] = dwa[jj];
    __syncthreads();
    for (int j = threadIdx.x; j < D; j += 256)
        dw_part[(size_t)blk * D + j] = (sdw[0][j] + sdw[1][j]) + (sdw[2][j] + sdw[3][j]);
}

// bw_norm_kernel for D columns: NJ the power of two with 64 NJ >= D.
template <bool BF>
void launch_norm_adjoint(dim3 nb, const void* x, const float* w, const float* rs, const float* dxh, int B, int T,
                         int Tp, int H, int D, void* dx, float* dw_part, hipStream_t stream) {
    const dim3 blk(256);
#define CYFA_BW_NORM(NJ_) \
    hipLaunchKernelGGL((bw_norm_kernel<BF, NJ_>), nb, blk, 0, stream, x, w, rs, dxh, B, T, Tp, H, D, dx, dw_part)
    if (D <= 64)
        CYFA_BW_NORM(1);
    else if (D <= 128)
        CYFA_BW_NORM(2);
    else if (D <= 256)
        CYFA_BW_NORM(4);
    else if (D <= 512)
        CYFA_BW_NORM(8);
    else
        CYFA_BW_NORM(16);
#undef CYFA_BW_NORM
}

// out[i] = sum over the nb partial rows of part[.][i]: one wave per column,
// lane l adding rows l, l + 64, .. in order, then the wave's fixed-order sum.
// blockIdx.y: q's partials or k's.
__global__ __launch_bounds__(256) void bw_reduce_kernel(const float* part_q, const float* part_k, int nb, size_t n,
                                                        float* out_q, float* out_k) {
    const float* part = blockIdx.y ? part_k : part_q;
    float* out = blockIdx.y ? out_k : out_q;
    const size_t i = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (i >= n) return;
    float s = 0.f;
    int b = lane;
    for (; b + 7 * 64 < nb; b += 8 * 64) {  // eight loads in flight
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = part[(size_t)(b + 64 * u) * n + i];
#pragma unroll
        for (int u = 0; u < 8; u++) s += v[u];
    }
    for (; b < nb; b += 64) s += part[(size_t)b * n + i];
    s = bw_wave_sum(s);
    if (lane == 0) out[i] = s;
}

// The table cotangent: per head, sum the readout blocks' partials in order.
__global__ __launch_bounds__(256) void bw_table_reduce_kernel(const float* part, int nb, int RM, float* out) {
    const int h = blockIdx.y, e = blockIdx.x * 256 + threadIdx.x;
    if (e >= RM) return;
    const float* p = part + (size_t)h * nb * RM + e;
    float s = 0.f;
    int b = 0;
    for (; b + 16 <= nb; b += 16) {  // sixteen loads in flight, then the sums in order
        float v[16];
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = p[(size_t)(b + i) * RM];
#pragma unroll
        for (int i = 0; i < 16; i++) s += v[i];
    }
    for (; b < nb; b++) s += p[(size_t)b * RM];
    out[(size_t)h * RM + e] = s;
}

// dreadout[h][r][j] = sum_m dtable[h][r][m] Phi[j][m] (table = readout Phi,
// ops/chunk.py:82-103, 281); Phi's angle 2 pi ((pair j) mod R) / R is reduced
// exactly in integers. One block per (h, r), thread j.
// The R angles' sine and cosine are formed once per block in LDS and indexed
// by the exact integer reduction (pair j) mod R, stepped by j per pair: the
// same values as a sincosf per term.
__global__ __launch_bounds__(256) void bw_dreadout_kernel(const float* dtable, int M, float* dreadout) {
    const int R = M - 1, hr = blockIdx.x, j = threadIdx.x;
    __shared__ float row[BWD_MAX_M], sin_k[BWD_MAX_M], cos_k[BWD_MAX_M];
    if (j < M) row[j] = dtable[(size_t)hr * M + j];
    if (j < R) sincosf((float)((double)j * (kTwoPiBw / R)), &sin_k[j], &cos_k[j]);
    __syncthreads();
    if (j >= R) return;
    float acc = 0.f;
    int k = 0;  // (pair j) mod R
    for (int pair = 0; pair < M / 2; pair++) {
        const float sc = (float)sqrt((pair == 0 ? 1.0 : 2.0) / R);
        acc = fmaf(row[2 * pair], sc * cos_k[k], acc);
        if (pair > 0) acc = fmaf(row[2 * pair + 1], sc * sin_k[k], acc);  // column 1 is not a basis vector
        k += j;
        k = k >= R ? k - R : k;
    }
    dreadout[(size_t)hr * R + j] = acc;
}

// Head-major fp32 [B*H, Tp, D] rows into [B, T, H, D] in the operands' dtype.
template <bool BF>
__global__ __launch_bounds__(256) void bw_pack_kernel(const float* src, int B, int T, int Tp, int H, int D, void* dst) {
    // four consecutive elements per thread (D % 4 == 0, the launcher checks;
    // a row's four never straddle two rows)
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4, n = (size_t)B * T * H * D;
    if (i >= n) return;
    const int j = (int)(i % D);
    const size_t row = i / D;
    const int h = (int)(row % H), t = (int)((row / H) % T), b = (int)(row / ((size_t)H * T));
    const float4 v = *reinterpret_cast<const float4*>(src + (((size_t)b * H + h) * Tp + t) * D + j);
    if constexpr (BF) {
        const bf16x4 o = {(bf16_t)v.x, (bf16_t)v.y, (bf16_t)v.z, (bf16_t)v.w};
        *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16_t*>(dst) + i) = o;
    } else {
        *reinterpret_cast<float4*>(reinterpret_cast<float*>(dst) + i) = v;
    }
}

// The same, one element per thread (any D, any alignment of dst).
template <bool BF>
__global__ __launch_bounds__(256) void bw_pack1_kernel(const float* src, int B, int T, int Tp, int H, int D, void* dst) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, n = (size_t)B * T * H * D;
    if (i >= n) return;
    const int j = (int)(i % D);
    const size_t row = i / D;
    const int h = (int)(row % H), t = (int)((row / H) % T), b = (int)(row / ((size_t)H * T));
    bw_st<BF>(dst, i, src[(((size_t)b * H + h) * Tp + t) * D + j]);
}

// Workgroups per chunk of the chunk kernels for `chunks` chunks of `tiles`
// output tiles: one where the chunks give every compute unit two workgroups;
// below that the tiles are shared out over up to four workgroups per compute
// unit, each forming its own scores again. One backward on MI355X, us with 1
// and with 3 (two 64 NT = 128 wide tiles of dq and dk, one of dv): 78 chunks
// (bf16) 347 / 289, 128 (fp32) 416 / 348, 192 (bf16) 468 / 434, 512 (bf16)
// 756 / 769, 1024 (bf16) 1266 / 1316.
int chunk_parts(long long chunks, int tiles) {
    const long long cus = device_cu_count();
    if (chunks >= 2 * cus) return 1;
    const long long parts = (4 * cus + chunks - 1) / chunks;
    return parts > tiles ? tiles : (int)parts;
}

template <int NT>
void launch_chunk_grad_nt(const ChunkGradArgs& a, bool mfma, bool v4, hipStream_t stream) {
    const dim3 grid(a.N, a.H, a.B * a.parts), blk(256);
#define CYFA_BW_CHUNK(MF_, V4_, SB_, RB_) \
    hipLaunchKernelGGL((bw_chunk_kernel<MF_, V4_, SB_, RB_, NT>), grid, blk, 0, stream, a)
    // (the flags pair as the backward sets them: sbf for bf16 calls, rbf for pass 2's)
    if (mfma && v4) {
        if (a.rbf)
            CYFA_BW_CHUNK(true, true, true, true);
        else
            CYFA_BW_CHUNK(true, true, true, false);
    } else if (mfma) {
        if (a.rbf)
            CYFA_BW_CHUNK(true, false, true, true);
        else
            CYFA_BW_CHUNK(true, false, true, false);
    } else if (v4) {
        CYFA_BW_CHUNK(false, true, false, false);
    } else {
        CYFA_BW_CHUNK(false, false, false, false);
    }
#undef CYFA_BW_CHUNK
}

int launch_chunk_grad(ChunkGradArgs a, bool mfma, hipStream_t stream) {
    if (mfma != (a.sbf != 0)) return -1;  // bf16 calls keep bf16 states, fp32 calls fp32 ones
    // rows and states 16-byte aligned (workspace buffers, rows of Kq and Vd floats)
    const bool v4 = a.Kq % 4 == 0 && a.Vd % 4 == 0;
    const long long chunks = (long long)a.N * a.H * a.B;
    const auto tiles = [&](int w) { return (a.Kq + w - 1) / w + (a.Vd + w - 1) / w; };
    // 64-wide tiles where even they leave compute units idle (78 chunks: 284 us
    // against 289 with 128-wide ones, 20 chunks: 217 against 227)
    if (v4 && chunks * tiles(2 * BC) >= device_cu_count()) {
        a.parts = chunk_parts(chunks, tiles(2 * BC));
        launch_chunk_grad_nt<2>(a, mfma, v4, stream);
    } else {
        a.parts = chunk_parts(chunks, tiles(BC));
        launch_chunk_grad_nt<1>(a, mfma, v4, stream);
    }
    return 0;
}

}  // namespace

int launch_chunk_pass(const ChunkPassParams& p, hipStream_t stream) {
    if (p.B < 1 || p.H < 1 || p.T < 1 || p.Tp < p.T || p.Tp % BC || p.Kq < 1 || p.Kq > BW_MAX_D || p.Vd < 1 ||
        p.Vd > BW_MAX_D || (!p.out && !p.out_bthd) || !p.states)
        return -1;
    const int N = p.Tp / BC;
    StateScanArgs sa{};
    sa.a = p.k;
    sa.b = p.v;
    sa.bl = head_major(p.H, p.Tp, p.Vd);
    sa.g = p.g;
    sa.x0 = p.s0;
    sa.xs = p.states;
    sa.x_out = p.s_final;
    sa.B = p.B;
    sa.T = p.T;
    sa.Tp = p.Tp;
    sa.H = p.H;
    sa.Kq = p.Kq;
    sa.Vd = p.Vd;
    sa.N = N;
    sa.scale = 1.f;
    sa.sbf = p.mfma && p.sbf16;
    launch_state_scan<false>(sa, p.mfma, stream);
    OutArgs oa{};
    oa.q = p.q;
    oa.k = p.k;
    oa.v = p.v;
    oa.g = p.g;
    oa.S = p.states;
    oa.out = p.out;
    oa.out_bthd = p.out_bthd;
    oa.bf16 = p.bf16;
    oa.B = p.B;
    oa.T = p.T;
    oa.Tp = p.Tp;
    oa.H = p.H;
    oa.Kq = p.Kq;
    oa.Vd = p.Vd;
    oa.N = N;
    oa.scale = p.scale;
    oa.sbf = p.mfma && p.sbf16;
    // rows and states 16-byte aligned (workspace buffers, rows of Kq and Vd floats)
    const bool v4 = p.Kq % 4 == 0 && p.Vd % 4 == 0;
    oa.parts = chunk_parts((long long)N * p.H * p.B, (p.Vd + BC - 1) / BC);
    const dim3 og(N, p.H, p.B * oa.parts);
    if (p.mfma && v4)
        hipLaunchKernelGGL((oa.sbf ? bw_out_kernel<true, true, true> : bw_out_kernel<true, true, false>), og, dim3(256),
                           0, stream, oa);
    else if (p.mfma)
        hipLaunchKernelGGL((oa.sbf ? bw_out_kernel<true, false, true> : bw_out_kernel<true, false, false>), og,
                           dim3(256), 0, stream, oa);
    else if (v4)
        hipLaunchKernelGGL((bw_out_kernel<false, true, false>), og, dim3(256), 0, stream, oa);
    else
        hipLaunchKernelGGL((bw_out_kernel<false, false, false>), og, dim3(256), 0, stream, oa);
    return 0;
}

int launch_chunk_readout(const float* raw, const float* cs, const float* sn, const float* table, float* lg, int B,
                         int Tp, int H, int M, int bf16, int split, float* wts, hipStream_t stream) {
    if (B < 1 || H < 1 || Tp < 1 || Tp % BC || M < 4 || M > BWD_MAX_M || M % 2) return -1;
    const dim3 blk(256);
    if (M > BWD_TABLE_M) {  // logits, softmax, then the weights, streaming the table
        if (!lg) return -1;
        WideArgs wa{};
        wa.raw = raw;
        wa.cs = cs;
        wa.sn = sn;
        wa.table = table;
        wa.lg = lg;
        wa.wts = wts;
        wa.B = B;
        wa.Tp = Tp;
        wa.H = H;
        wa.M = M;
        wa.bf = bf16;
        const int rows_h = B * Tp;
        const size_t rows = (size_t)rows_h * H;
        hipLaunchKernelGGL(bw_wide_logits_kernel<false>, dim3((rows_h + BC - 1) / BC, (M - 1 + BC - 1) / BC, H), blk,
                           0, stream, wa);
        hipLaunchKernelGGL(bw_wide_softmax_kernel<false>, dim3((unsigned)((rows + 3) / 4)), blk, 0, stream, wa);
        hipLaunchKernelGGL(bw_wide_u_kernel<false>, dim3((rows_h + BC - 1) / BC, (M + BC - 1) / BC, H), blk, 0,
                           stream, wa);
        return 0;
    }
    const int per = bwd_ro_per_wg(B, Tp, H, split ? 512 : 256), blocks = (B * Tp + BWD_RO_BLOCK - 1) / BWD_RO_BLOCK;
    const dim3 grid((blocks + per - 1) / per, H);
    ReadoutGradArgs ro{};
    ro.raw = raw;
    ro.cs = cs;
    ro.sn = sn;
    ro.table = table;
    ro.wts = wts;
    ro.B = B;
    ro.Tp = Tp;
    ro.H = H;
    ro.M = M;
    ro.per_wg = per;
    if (split && bf16)
        hipLaunchKernelGGL((bw_readout_mf_kernel<false, true>), grid, dim3(64 * RO_MF_WAVES), 0, stream, ro);
    else if (split)
        hipLaunchKernelGGL((bw_readout_mf_kernel<false, false>), grid, dim3(64 * RO_MF_WAVES), 0, stream, ro);
    else if (bf16)
        return -1;  // bf16 operands come with the split form
    else
        hipLaunchKernelGGL(bw_fwd_readout_kernel, grid, dim3(RO_FWD_THREADS), 0, stream, raw, cs, sn, table, B, Tp, H, M, per,
                           wts);
    return 0;
}

int launch_chunk_bwd(const BwdParams& p, hipStream_t stream) {
    const int B = p.B, T = p.T, H = p.H, K = p.K, V = p.V, M = p.M;
    if (B < 1 || T < 1 || H < 1 || K < 1 || K > BW_MAX_D || V < 1 || V > BW_MAX_D || M < 4 || M > BWD_MAX_M || M % 2)
        return -1;
    const int Tp = (T + BC - 1) / BC * BC;
    const BwdWorkspace ws = bwd_workspace(B, T, H, K, V, M, p.workspace);
    const int N = ws.N;
    const size_t rows = (size_t)B * H * Tp;
    const dim3 blk(256), rb((unsigned)((rows + 3) / 4));
    const bool bf = p.bf16 != 0;
    // v, the output cotangent and v's cotangent are read and written in place,
    // [B, T, H, V], where their rows take 16-byte accesses and a chunk of them
    // stays within the kernels' 32-bit offsets; otherwise through head-major
    // copies (65536 rows of 256 bf16: 33 us for the two copies, 22 us for v's
    // cotangent, of a training pass of 1178 us in all, 1119 so).
    const bool direct = V % 4 == 0 && ((uintptr_t)p.v | (uintptr_t)p.d_o | (uintptr_t)p.dv) % 16 == 0 &&
                        (long long)H * V * BC * 4 < (1ll << 31);
    const RowsAt vl = direct ? RowsAt{(size_t)T * H * V, (size_t)V, H * V, T} : head_major(H, Tp, V);
    const float* v_rows = direct ? static_cast<const float*>(p.v) : ws.vh;
    const float* o_rows = direct ? static_cast<const float*>(p.d_o) : ws.dO;
    const int oT = direct && !p.d_o ? 0 : vl.T;
    // the normalised rows, head-major fp32; v and dO
#define CYFA_BW_ROWS(BFV)                                                                                           \
    hipLaunchKernelGGL(bw_rows_kernel<BFV>, rb, blk, 0, stream, p.q, p.q_w, p.q_eps, B, T, Tp, H, K, ws.qh, ws.rq); \
    hipLaunchKernelGGL(bw_rows_kernel<BFV>, rb, blk, 0, stream, p.k, p.k_w, p.k_eps, B, T, Tp, H, K, ws.kh, ws.rk); \
    if (!direct) {                                                                                                  \
        hipLaunchKernelGGL((bw_rows_kernel<BFV, RowT>), rb, blk, 0, stream, p.v, (const float*)nullptr, 0.f, B, T, Tp, H, \
                           V, reinterpret_cast<RowT*>(ws.vh), (float*)nullptr);                                    \
        hipLaunchKernelGGL((bw_rows_kernel<BFV, RowT>), rb, blk, 0, stream, p.d_o, (const float*)nullptr, 0.f, B, T, Tp, \
                           H, V, reinterpret_cast<RowT*>(ws.dO), (float*)nullptr);                                 \
    }
    // v and dO of bf16 calls stay bf16 in head-major rows (exact): the pass-2
    // scans and chunk kernels read half the bytes.
    if (bf) {
        using RowT = bf16_t;
        CYFA_BW_ROWS(true)
    } else {
        using RowT = float;
        CYFA_BW_ROWS(false)
    }
#undef CYFA_BW_ROWS
    // the forward, recomputed in fp32: clock, write vector, the states before
    // every chunk of both passes, the pass-1 output and the slot weights
    if (launch_general_clock_write(p.delta, p.clock0, p.beta, B, T, Tp, H, M, ws.lam, ws.w, ws.cs, ws.sn, stream) != 0)
        return -1;
    // The stored states and state cotangents of bf16 calls are bf16, as the
    // reference stores its chunk states and their cotangents (the recurrence
    // itself runs in fp32 registers; ops/chunk_h.py:212-214, 329-331).
    StateScanArgs f1{};
    f1.sbf = bf;
    f1.a = ws.kh;
    f1.b = ws.w;
    f1.bl = head_major(H, Tp, M);
    f1.g = p.g;
    f1.x0 = p.h0_k;
    f1.xs = ws.sk;
    f1.B = B;
    f1.T = T;
    f1.Tp = Tp;
    f1.H = H;
    f1.Kq = K;
    f1.Vd = M;
    f1.N = N;
    f1.scale = 1.f;
    ChunkPassParams p1{};
    p1.q = ws.qh;
    p1.k = ws.kh;
    p1.v = ws.w;
    p1.g = p.g;
    p1.s0 = p.h0_k;
    p1.states = ws.sk;
    p1.out = ws.raw;
    p1.mfma = bf;
    p1.sbf16 = bf;
    p1.B = B;
    p1.T = T;
    p1.Tp = Tp;
    p1.H = H;
    p1.Kq = K;
    p1.Vd = M;
    p1.scale = p.scale;
    if (launch_chunk_pass(p1, stream) != 0 ||
        launch_chunk_readout(ws.raw, ws.cs, ws.sn, p.table, ws.lg, B, Tp, H, M, 0, bf, ws.wts, stream) != 0)
        return -1;
    const int ro_per_wg = bwd_ro_per_wg(B, Tp, H, 256);
    const bool wide = M > BWD_TABLE_M;
    WideArgs wa{};
    wa.raw = ws.raw;
    wa.cs = ws.cs;
    wa.sn = ws.sn;
    wa.table = p.table;
    wa.dwts = ws.dwts;
    wa.lg = ws.lg;
    wa.dl = ws.dlw;
    wa.wts = ws.wts;
    wa.draw = ws.draw;
    wa.dlp = ws.dlp;
    wa.dlam = ws.dlam;
    wa.dgq = ws.dgq;
    wa.dtab = ws.dtab;
    wa.B = B;
    wa.Tp = Tp;
    wa.H = H;
    wa.M = M;
    wa.splits = ws.ro_blocks;
    const int rows_h = B * Tp;
    const dim3 g_logits((rows_h + BC - 1) / BC, (M - 1 + BC - 1) / BC, H), g_u((rows_h + BC - 1) / BC, (M + BC - 1) / BC, H);
    const dim3 g_rows((unsigned)((rows + 3) / 4));
    StateScanArgs f2 = f1;
    f2.a = ws.w;
    f2.b = v_rows;
    f2.bl = vl;
    f2.x0 = p.h0_v;
    f2.xs = ws.sv;
    f2.bbf = bf;  // v's rows
    f2.Kq = M;
    f2.Vd = V;
    launch_state_scan<false>(f2, bf, stream);
    // pass 2: state cotangents, then the rows' (slot weights, write vector, v)
    StateScanArgs s2 = f2;
    s2.a = ws.wts;
    s2.b = o_rows;
    s2.bl.T = oT;
    s2.x0 = p.d_hv;
    s2.xs = ws.dsv;
    s2.S = ws.sv;
    s2.bnd = ws.bnd2;
    s2.x_out = p.dh0_v;
    launch_state_scan<true>(s2, bf, stream);
    ChunkGradArgs c2{};
    c2.sbf = bf;
    c2.rbf = bf;  // v's and dO's rows
    c2.q = ws.wts;
    c2.k = ws.w;
    c2.v = v_rows;
    c2.dO = o_rows;
    c2.vl = vl;
    c2.oT = oT;
    c2.g = p.g;
    c2.S = ws.sv;
    c2.D = ws.dsv;
    c2.dq = ws.dwts;
    c2.dk = ws.dw2;
    c2.dv = direct ? static_cast<float*>(p.dv) : ws.dvh;
    c2.dvbf = direct && bf;
    c2.B = B;
    c2.T = T;
    c2.Tp = Tp;
    c2.H = H;
    c2.Kq = M;
    c2.Vd = V;
    c2.N = N;
    c2.scale = 1.f;
    if (launch_chunk_grad(c2, bf, stream) != 0) return -1;
    // the readout: the pass-1 output's cotangent, the clock's share and the table's
    ReadoutGradArgs ro{};
    ro.raw = ws.raw;
    ro.cs = ws.cs;
    ro.sn = ws.sn;
    ro.table = p.table;
    ro.dwts = ws.dwts;
    ro.draw = ws.draw;
    ro.dlam = ws.dlam;
    ro.dgq = ws.dgq;
    ro.dtab = ws.dtab;
    ro.B = B;
    ro.Tp = Tp;
    ro.H = H;
    ro.M = M;
    ro.per_wg = ro_per_wg;
    if (wide) {  // dp, dl, then dz with draw and the clock's share, and the table cotangent's partials
        hipLaunchKernelGGL(bw_wide_logits_kernel<true>, g_logits, blk, 0, stream, wa);
        hipLaunchKernelGGL(bw_wide_softmax_kernel<true>, g_rows, blk, 0, stream, wa);
        hipLaunchKernelGGL(bw_wide_u_kernel<true>, g_u, blk, 0, stream, wa);
        hipLaunchKernelGGL(bw_wide_dlam_kernel, dim3((unsigned)((rows + 255) / 256)), blk, 0, stream, wa);
        hipLaunchKernelGGL(bw_wide_dtable_kernel, dim3((M - 1 + BC - 1) / BC, (M + BC - 1) / BC, H * ws.ro_blocks), blk, 0,
                           stream, wa);
    } else if (bf) {
        hipLaunchKernelGGL((bw_readout_mf_kernel<true, false>), dim3(ws.ro_blocks, H), dim3(64 * RO_MF_WAVES), 0, stream, ro);
    } else {
        hipLaunchKernelGGL(bw_readout_kernel, dim3(ws.ro_blocks, H), dim3(RO_ADJ_THREADS), 0, stream, ro);
    }
    // pass 1, with the pass-1 output's cotangent as dO
    StateScanArgs s1 = f1;
    s1.a = ws.qh;
    s1.b = ws.draw;
    s1.x0 = p.d_hk;
    s1.xs = ws.dsk;
    s1.S = ws.sk;
    s1.bnd = ws.bnd1;
    s1.x_out = p.dh0_k;
    s1.scale = p.scale;
    launch_state_scan<true>(s1, bf, stream);
    ChunkGradArgs c1 = c2;
    c1.rbf = 0;  // pass 1's rows (the write vector, draw) are fp32
    c1.q = ws.qh;
    c1.k = ws.kh;
    c1.vl = head_major(H, Tp, M);
    c1.oT = Tp;
    c1.dvbf = 0;
    c1.v = ws.w;
    c1.dO = ws.draw;
    c1.S = ws.sk;
    c1.D = ws.dsk;
    c1.dq = ws.dqh;
    c1.dk = ws.dkh;
    c1.dv = ws.dw1;
    c1.Kq = K;
    c1.Vd = M;
    c1.scale = p.scale;
    if (launch_chunk_grad(c1, bf, stream) != 0) return -1;
    // gates, write vector and clock
    TokenGradArgs tg{};
    tg.dgq = ws.dgq;
    tg.dw2 = ws.dw2;
    tg.dw1 = ws.dw1;
    tg.cs = ws.cs;
    tg.sn = ws.sn;
    tg.bnd1 = ws.bnd1;
    tg.bnd2 = ws.bnd2;
    tg.beta = p.beta;
    tg.dlam = ws.dlam;
    tg.dg = p.dg;
    tg.dbeta = p.dbeta;
    tg.B = B;
    tg.T = T;
    tg.Tp = Tp;
    tg.H = H;
    tg.M = M;
    tg.N = N;
    tg.nt1 = ws.nt1;
    tg.nt2 = ws.nt2;
    if (bf)
        hipLaunchKernelGGL(bw_token_kernel<float>, dim3(N, B * H), blk, 0, stream, tg);
    else
        hipLaunchKernelGGL(bw_token_kernel<double>, dim3(N, B * H), blk, 0, stream, tg);
    hipLaunchKernelGGL(bw_clock_kernel, dim3(B * H), dim3(64), 0, stream, ws.dlam, p.d_clock, B, T, Tp, H, p.ddelta,
                       p.dclock0);
    // the q/k norms, their weights, v's layout
    const dim3 nb(ws.norm_blocks);
    if (bf) {
        launch_norm_adjoint<true>(nb, p.q, p.q_w, ws.rq, ws.dqh, B, T, Tp, H, K, p.dq, ws.dnq, stream);
        launch_norm_adjoint<true>(nb, p.k, p.k_w, ws.rk, ws.dkh, B, T, Tp, H, K, p.dk, ws.dnk, stream);
    } else {
        launch_norm_adjoint<false>(nb, p.q, p.q_w, ws.rq, ws.dqh, B, T, Tp, H, K, p.dq, ws.dnq, stream);
        launch_norm_adjoint<false>(nb, p.k, p.k_w, ws.rk, ws.dkh, B, T, Tp, H, K, p.dk, ws.dnk, stream);
    }
    hipLaunchKernelGGL(bw_reduce_kernel, dim3((unsigned)((K + 3) / 4), 2), blk, 0, stream, ws.dnq, ws.dnk, ws.norm_blocks,
                       (size_t)K, p.dq_w, p.dk_w);
    if (!direct) {
        const size_t nv = (size_t)B * T * H * V;
        const dim3 vb((unsigned)((nv + 255) / 256)), vb4((unsigned)((nv / 4 + 255) / 256));
        const bool pack4 = V % 4 == 0 && ((uintptr_t)p.dv & (bf ? 7 : 15)) == 0;
        if (bf && pack4)
            hipLaunchKernelGGL(bw_pack_kernel<true>, vb4, blk, 0, stream, ws.dvh, B, T, Tp, H, V, p.dv);
        else if (pack4)
            hipLaunchKernelGGL(bw_pack_kernel<false>, vb4, blk, 0, stream, ws.dvh, B, T, Tp, H, V, p.dv);
        else if (bf)
            hipLaunchKernelGGL(bw_pack1_kernel<true>, vb, blk, 0, stream, ws.dvh, B, T, Tp, H, V, p.dv);
        else
            hipLaunchKernelGGL(bw_pack1_kernel<false>, vb, blk, 0, stream, ws.dvh, B, T, Tp, H, V, p.dv);
    }
    const int RM = (M - 1) * M;
    hipLaunchKernelGGL(bw_table_reduce_kernel, dim3((RM + 255) / 256, H), blk, 0, stream, ws.dtab, ws.ro_blocks, RM,
                       p.dtable);
    if (p.dreadout)
        hipLaunchKernelGGL(bw_dreadout_kernel, dim3(H * (M - 1)), blk, 0, stream, p.dtable, M, p.dreadout);
    return 0;
}

}  // namespace cyfa
