// Kernels of the warm-start network (the math is stated in mpnn.h): input
// features, dense layers (LDS-staged weights, FP32 accumulation), mean
// aggregation over A's rows or columns (a wave per node, features on the
// lanes), the output head, the loss, and the backward pass: ReLU masks,
// input gradients, weight gradients as fixed-order block partials, the
// transposed aggregation, and Adam.  Nothing uses atomics: every sum has a
// fixed order, so training is bitwise reproducible.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "launch.h"
#include "mpnn.h"

namespace help {

namespace {

constexpr int kB = 256;
inline int grid_for(int64_t n) { return (int)std::max<int64_t>(1, (n + kB - 1) / kB); }
inline int grid_cap(int64_t n, int cap) { return (int)std::min<int64_t>(cap, std::max<int64_t>(1, n)); }

__device__ inline float ldv(float x) { return x; }
__device__ inline float ldv(Bf16 x) { return __uint_as_float((uint32_t)x.v << 16); }
__device__ inline void stv(float& d, float x) { d = x; }
__device__ inline void stv(Bf16& d, float x) {   // round to nearest even
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x7fffffu)) { d.v = 0x7fc0; return; }
    u += 0x7fffu + ((u >> 16) & 1u);
    d.v = (uint16_t)(u >> 16);
}
__device__ inline float round_bf16(float x) {
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7f800000u) == 0x7f800000u) return x;
    u += 0x7fffu + ((u >> 16) & 1u);
    return __uint_as_float(u & 0xffff0000u);
}

// ---------------------------------------------------------------- features
__global__ void k_feat_row(int32_t m, const double* __restrict__ g, const double* __restrict__ r, double rs,
                           double mu, float* __restrict__ xr) {
    const int32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= m) return;
    const double gi = g[i] > 0 ? g[i] : 1.0;
    const double jac = fmin(10.0, fmax(-10.0, exp(mu) * r[i] / (rs * gi)));
    xr[(int64_t)i * kNnFR + 0] = (float)(r[i] / rs);
    xr[(int64_t)i * kNnFR + 1] = (float)((log(gi) - mu) / 10.0);
    xr[(int64_t)i * kNnFR + 2] = (float)(jac / 10.0);
    xr[(int64_t)i * kNnFR + 3] = 1.0f;
}

__global__ void k_feat_col(int32_t n, const double* __restrict__ dinv, double nu, float* __restrict__ xc) {
    const int32_t j = blockIdx.x * kB + threadIdx.x;
    if (j >= n) return;
    xc[(int64_t)j * kNnFC + 0] = (float)((log(dinv[j]) - nu) / 10.0);
    xc[(int64_t)j * kNnFC + 1] = 1.0f;
}

// Partial sums of the input statistics, blockIdx.y = 0: log g_i and the
// count of g_i > 0, 1: the same for 1/d, 2: r_i^2 (rows of gridDim.x partials
// in that order).  Bound by the launches and the copy to the host: one of
// each for the three.
__global__ __launch_bounds__(256) void k_stats(int64_t m, int64_t n, const double* __restrict__ g,
                                               const double* __restrict__ dinv, const double* __restrict__ r,
                                               double* __restrict__ part) {
    __shared__ double s0[kB], s1[kB];
    const int what = blockIdx.y;
    const double* x = what == 0 ? g : what == 1 ? dinv : r;
    const int64_t cnt = what == 1 ? n : m;
    part += 2 * what * gridDim.x;
    double a = 0.0, c = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kB + threadIdx.x; i < cnt; i += (int64_t)gridDim.x * kB) {
        const double v = x[i];
        if (what < 2) {
            if (v > 0) { a += log(v); c += 1.0; }
        } else {
            a += v * v;
        }
    }
    s0[threadIdx.x] = a;
    s1[threadIdx.x] = c;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) { s0[threadIdx.x] += s0[threadIdx.x + w]; s1[threadIdx.x] += s1[threadIdx.x + w]; }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[blockIdx.x] = s0[0];
        if (what < 2) part[gridDim.x + blockIdx.x] = s1[0];
    }
}

// ---------------------------------------------------------------- rows
// Eight consecutive features of a node's row as FP32: one 16-byte load (BF16)
// or two (FP32), so a row is 8 lanes wide and a wave moves eight rows at once.
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

__device__ inline void load8(const Bf16* __restrict__ p, float (&v)[8]) {
    const u32x4_t u = *reinterpret_cast<const u32x4_t*>(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[2 * e] = __uint_as_float(u[e] << 16);
        v[2 * e + 1] = __uint_as_float(u[e] & 0xffff0000u);
    }
}
__device__ inline void load8(const float* __restrict__ p, float (&v)[8]) {
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p), b = *reinterpret_cast<const f32x4_t*>(p + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { v[e] = a[e]; v[4 + e] = b[e]; }
}
__device__ inline void store8(Bf16* __restrict__ p, const float (&v)[8]) {
    u32x4_t u;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        Bf16 lo, hi;
        stv(lo, v[2 * e]);
        stv(hi, v[2 * e + 1]);
        u[e] = (uint32_t)lo.v | ((uint32_t)hi.v << 16);
    }
    *reinterpret_cast<u32x4_t*>(p) = u;
}
__device__ inline void store8(float* __restrict__ p, const float (&v)[8]) {
    *reinterpret_cast<f32x4_t*>(p) = f32x4_t{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4_t*>(p + 4) = f32x4_t{v[4], v[5], v[6], v[7]};
}
// four consecutive features
__device__ inline f32x4_t load4(const Bf16* __restrict__ p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    return f32x4_t{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                   __uint_as_float(u.y & 0xffff0000u)};
}
__device__ inline f32x4_t load4(const float* __restrict__ p) { return *reinterpret_cast<const f32x4_t*>(p); }

// ------------------------------------------------------------ dense layers
template <typename AT>
__global__ __launch_bounds__(256) void k_dense(int64_t N, const AT* __restrict__ in1, int k1,
                                               const AT* __restrict__ in2, int k2, const float* __restrict__ W,
                                               const float* __restrict__ b, AT* __restrict__ out) {
    __shared__ float Ws[2 * kNnH * kNnH];
    __shared__ float xs[4][2 * kNnH];
    const int K = k1 + k2;
    for (int t = threadIdx.x; t < K * kNnH; t += kB) Ws[t] = W[t];
    const int q = threadIdx.x >> 6, o = threadIdx.x & 63;
    const float bo = b[o];
    __syncthreads();
    for (int64_t base = (int64_t)blockIdx.x * 4; base < N; base += (int64_t)gridDim.x * 4) {
        for (int t = threadIdx.x; t < 4 * K; t += kB) {
            const int qq = t / K, k = t - qq * K;
            const int64_t node = base + qq;
            float v = 0.0f;
            if (node < N) v = (k < k1) ? ldv(in1[node * k1 + k]) : ldv(in2[node * k2 + (k - k1)]);
            xs[qq][k] = v;
        }
        __syncthreads();
        const int64_t node = base + q;
        if (node < N) {
            float acc = bo;
            for (int k = 0; k < K; ++k) acc += xs[q][k] * Ws[k * kNnH + o];
            stv(out[node * kNnH + o], fmaxf(acc, 0.0f));
        }
        __syncthreads();
    }
}

// The input layers (K = 4 row or 2 column features): a thread per 8 outputs of
// a node, the terms in the order of k_dense.  Bound by the write of the N x 64
// activations; k_dense, which stages four nodes at a time behind two barriers,
// took 89 us where this takes 23 us (mean of the two layers, m + n =
// 1.07 million nodes, BF16).
template <typename AT, int K>
__global__ __launch_bounds__(256) void k_dense_in(int64_t N, const float* __restrict__ in, const float* __restrict__ W,
                                                  const float* __restrict__ b, AT* __restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * kB + threadIdx.x;
    const int64_t node = t >> 3;
    const int o = 8 * (int)(t & 7);
    if (node >= N) return;
    float x[K], v[8];
#pragma unroll
    for (int k = 0; k < K; ++k) x[k] = in[node * K + k];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float acc = b[o + e];
#pragma unroll
        for (int k = 0; k < K; ++k) acc = __builtin_fmaf(x[k], W[k * kNnH + o + e], acc);
        v[e] = fmaxf(acc, 0.0f);
    }
    store8(out + node * kNnH + o, v);
}

// The BF16 layers with K = k1 + k2 a multiple of 32 (the message layers and
// the head) run on V_MFMA_F32_16X16X32_BF16 with FP32 accumulation: a
// workgroup takes 64 nodes, each wave 16 of them across the 64 outputs (four
// 16x16 tiles, the bias as the accumulators' start).  Lane layout (checked by
// help_selftest_mfma_bf16): A[i][k] in lane i + 16 (k/8), element k%8;
// B[k][j] in lane j + 16 (k/8), element k%8; D[i][j] in lane j + 16 (i/4),
// element i%4.  A lane's 8 inputs are 16 contiguous bytes of one node's row;
// the weights are staged in LDS transposed (row o holds W[.][o], padded by 8
// elements against bank conflicts) as BF16, which is exact: the BF16 mode's
// weights are BF16-rounded.
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;

__device__ inline uint16_t bf16_bits(float x) {
    Bf16 h;
    stv(h, x);
    return h.v;
}

__global__ __launch_bounds__(256) void k_dense_mfma(int64_t N, const Bf16* __restrict__ in1, int k1,
                                                    const Bf16* __restrict__ in2, int k2,
                                                    const float* __restrict__ W, const float* __restrict__ b,
                                                    Bf16* __restrict__ out) {
    constexpr int kLd = 2 * kNnH + 8;
    __shared__ __attribute__((aligned(16))) uint16_t Wt[kNnH * kLd];
    const int K = k1 + k2;
    for (int t = threadIdx.x; t < K * kNnH; t += kB) {
        const int k = t / kNnH, o = t - k * kNnH;
        Wt[o * kLd + k] = bf16_bits(W[t]);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lk = lane >> 4;
    float bias[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) bias[t] = b[16 * t + li];
    __syncthreads();
    for (int64_t base = (int64_t)blockIdx.x * 64; base < N; base += (int64_t)gridDim.x * 64) {
        const int64_t row = base + wave * 16 + li;
        const int64_t rc = row < N ? row : N - 1;
        f32x4_t acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = f32x4_t{bias[t], bias[t], bias[t], bias[t]};
        for (int kk = 0; kk < K; kk += 32) {
            const int k0 = kk + 8 * lk;
            const Bf16* src = k0 < k1 ? in1 + rc * k1 + k0 : in2 + rc * k2 + (k0 - k1);
            const bf16x8_t a = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(src));
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bf16x8_t bv =
                    __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(&Wt[(16 * t + li) * kLd + k0]));
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bv, acc[t], 0, 0, 0);
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t node = base + wave * 16 + 4 * lk + r;
                if (node < N) stv(out[node * kNnH + 16 * t + li], fmaxf(acc[t][r], 0.0f));
            }
    }
}

// lane-layout probe: lane l feeds a[8l .. 8l+7] and b[8l .. 8l+7] (BF16-exact
// values) to one V_MFMA_F32_16X16X32_BF16 from zero; out[4l + r] = element r
__global__ void k_mfma_bf16_probe(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ out) {
    const int l = threadIdx.x;
    uint16_t ua[8], ub[8];
    for (int e = 0; e < 8; ++e) { ua[e] = bf16_bits(a[8 * l + e]); ub[e] = bf16_bits(b[8 * l + e]); }
    const bf16x8_t va = __builtin_bit_cast(bf16x8_t, ua);
    const bf16x8_t vb = __builtin_bit_cast(bf16x8_t, ub);
    const f32x4_t d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, vb, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
    for (int r = 0; r < 4; ++r) out[4 * l + r] = d[r];
}

// out[node] = sum_{p in adj(node)} val[p] src[idx[p]] / max(deg, 1), p ascending.
// Bound by the gathered rows (128 or 256 bytes each).  Eight lanes per node,
// eight features each, so a wave gathers eight rows per load and four of a
// node's rows are in flight (indices past the end repeat the last one; their
// terms are dropped): 54 us per layer where a wave per node with one row in
// flight took 251 us (mean of four, 2.23 million nonzeros, 1.07 million nodes, BF16).
template <typename AT>
__global__ __launch_bounds__(256) void k_mean(int32_t N, const int64_t* __restrict__ ptr,
                                              const int32_t* __restrict__ idx, const double* __restrict__ val,
                                              const AT* __restrict__ src, AT* __restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * kB + threadIdx.x;
    const int64_t node = t >> 3;
    const int f = 8 * (int)(t & 7);
    if (node >= N) return;
    const int64_t b = ptr[node], e = ptr[node + 1];
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int64_t p = b; p < e; p += 4) {
        float w[4], x[4][8];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t q = p + u < e ? p + u : e - 1;
            w[u] = (float)val[q];
            load8(src + (int64_t)idx[q] * kNnH + f, x[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int k = 0; k < 8; ++k) acc[k] = p + u < e ? __builtin_fmaf(w[u], x[u][k], acc[k]) : acc[k];
    }
    const float deg = (float)(e - b > 1 ? e - b : 1);
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = acc[k] / deg;
    store8(out + node * kNnH + f, acc);
}

// y_i = z_i wo + bo: eight lanes per row, eight features each, so a wave takes
// eight rows with one load; the features' sum keeps its butterfly (features 32,
// 16, 8 apart over the lanes, then 4, 2, 1 apart in a lane).  180 thousand
// rows in BF16: 12 us, 50 us with a wave per row.
template <typename AT>
__global__ __launch_bounds__(256) void k_output(int32_t m, const AT* __restrict__ z, const float* __restrict__ wo,
                                                const float* __restrict__ bo, const double* __restrict__ g,
                                                double rs, float* __restrict__ y, double* __restrict__ x0) {
    const int f = 8 * (threadIdx.x & 7);
    const int64_t row = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 3);
    if (row >= m) return;   // (eight lanes together)
    float v[8];
    load8(z + row * kNnH + f, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] *= wo[f + k];
#pragma unroll
    for (int off = 4; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] += __shfl_xor(v[k], off);
#pragma unroll
    for (int off = 4; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < off; ++k) v[k] += v[k + off];
    if (f == 0) {
        const float yy = v[0] + bo[0];
        y[row] = yy;
        if (x0) x0[row] = g[row] > 0 ? (double)yy * rs / g[row] : 0.0;
    }
}

// ----------------------------------------------------------------- loss
__global__ __launch_bounds__(256) void k_loss(int32_t m, const float* __restrict__ y, const double* __restrict__ dy,
                                              const double* __restrict__ g, double rs, double* __restrict__ part) {
    __shared__ double s0[kB], s1[kB];
    double a = 0.0, c = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kB + threadIdx.x; i < m; i += (int64_t)gridDim.x * kB) {
        const double t = dy[i] * g[i] / rs;
        const double e = (double)y[i] - t;
        a += e * e;
        c += t * t;
    }
    s0[threadIdx.x] = a;
    s1[threadIdx.x] = c;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) { s0[threadIdx.x] += s0[threadIdx.x + w]; s1[threadIdx.x] += s1[threadIdx.x + w]; }
        __syncthreads();
    }
    if (threadIdx.x == 0) { part[blockIdx.x] = s0[0]; part[gridDim.x + blockIdx.x] = s1[0]; }
}

__global__ void k_out_grad(int32_t m, const float* __restrict__ y, const double* __restrict__ dy,
                           const double* __restrict__ g, double rs, double T, float* __restrict__ dyv) {
    const int32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= m) return;
    const double t = dy[i] * g[i] / rs;
    dyv[i] = (float)(2.0 * ((double)y[i] - t) / T);
}

// ------------------------------------------------------------- backward
// dpre[i][o] = dyv_i wo[o] (z[i][o] > 0)
template <typename AT>
__global__ void k_out_bwd(int32_t m, const AT* __restrict__ z, const float* __restrict__ dyv,
                          const float* __restrict__ wo, float* __restrict__ dpre) {
    const int64_t t = (int64_t)blockIdx.x * kB + threadIdx.x;
    if (t >= (int64_t)m * kNnH) return;
    const int64_t i = t / kNnH;
    const int o = (int)(t - i * kNnH);
    dpre[t] = ldv(z[t]) > 0.0f ? dyv[i] * wo[o] : 0.0f;
}

// Weight gradients.  Every block leaves one partial of the whole gradient of
// its layer, nn_wgrad_blocks(N) of them, and k_reduce_blocks adds them up in
// block order; the waves of a block add into LDS one after the other.

// the 4 (wave) x 4 (lane group) partial sums of four consecutive outputs per
// lane, added over the lane groups by a fixed butterfly
__device__ inline f32x4_t sum_groups(f32x4_t v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[e] += __shfl_xor(v[e], 16);
        v[e] += __shfl_xor(v[e], 32);
    }
    return v;
}

// partial[blk][o] = sum_i dyv_i z[i][o] (o < 64), partial[blk][64] = sum_i dyv_i:
// 16 lanes per node, four outputs each; bound by reading z
template <typename AT>
__global__ __launch_bounds__(256) void k_out_w(int32_t m, const AT* __restrict__ z, const float* __restrict__ dyv,
                                               float* __restrict__ partial) {
    __shared__ float red[4][kNnH + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lc = lane & 15, lk = lane >> 4;
    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f}, bs = acc;
    for (int64_t i0 = ((int64_t)blockIdx.x * 4 + wave) * 4; i0 < m; i0 += (int64_t)gridDim.x * 16) {
        const int64_t i = i0 + lk < m ? i0 + lk : m - 1;
        const float d = i0 + lk < m ? dyv[i] : 0.0f;
        f32x4_t v = load4(z + i * kNnH + 4 * lc);
        if (i0 + lk >= m) v = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};   // (0 times an infinite z is no zero)
        acc += d * v;
        bs[0] += d;
    }
    acc = sum_groups(acc);
    bs = sum_groups(bs);
    if (lk == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) red[wave][4 * lc + e] = acc[e];
        if (lc == 0) red[wave][kNnH] = bs[0];
    }
    __syncthreads();
    const int t = threadIdx.x;
    if (t <= kNnH) partial[(int64_t)blockIdx.x * (kNnH + 1) + t] = ((red[0][t] + red[1][t]) + red[2][t]) + red[3][t];
}

// The gradient entering a layer's products: dh masked by the layer's ReLU
// output h (h null: dh as it is).  Masking here saves a pass that would read
// dh and h and write the masked rows for two readers.
template <typename AT>
__device__ inline f32x4_t masked4(const float* __restrict__ dh, const AT* __restrict__ h, int64_t at) {
    f32x4_t d = load4(dh + at);
    if (h) {
        const f32x4_t a = load4(h + at);
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = a[e] > 0.0f ? d[e] : 0.0f;
    }
    return d;
}

// din[node][k] = sum_o dpre[node][o] W[k][o]; k < 64 -> din1 (+= if acc1), the
// others -> din2.  V_MFMA_F32_16X16X4_F32 with FP32 accumulation: a wave takes
// 16 nodes; A holds 16 rows of W (features), B the nodes, and inner slot 4 s + g
// (step s, lane group g) stands for o = 16 g + s, so a lane's 16 values of a
// node are 64 contiguous bytes and its 16 x kTiles weights stay in registers.
// D[feature][node] leaves four consecutive features of a node in a lane.
// Bound by reading dpre and writing din; a thread per output with the weights
// in LDS took 543 us where this takes 49 us (mean of five layers,
// m = 98,799, n = 262,080).
template <typename AT, int kTiles>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void k_dense_bwd_in(int64_t N, const float* __restrict__ dh, const AT* __restrict__ h, const float* __restrict__ W,
                    float* __restrict__ din1, float* __restrict__ din2, int acc1) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lc = lane & 15, lk = lane >> 4;
    float wv[kTiles][16];
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x4_t v = load4(W + (16 * t + lc) * kNnH + 16 * lk + 4 * q);
#pragma unroll
            for (int e = 0; e < 4; ++e) wv[t][4 * q + e] = v[e];
        }
    for (int64_t n0 = ((int64_t)blockIdx.x * 4 + wave) * 16; n0 < N; n0 += (int64_t)gridDim.x * 64) {
        const int64_t node = n0 + lc;
        const int64_t at = (node < N ? node : N - 1) * kNnH + 16 * lk;
        f32x4_t d[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = masked4(dh, h, at + 4 * q);
        f32x4_t acc[kTiles];
#pragma unroll
        for (int t = 0; t < kTiles; ++t) acc[t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 16; ++s)
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[t][s], d[s >> 2][s & 3], acc[t], 0, 0, 0);
        if (node < N) {
#pragma unroll
            for (int t = 0; t < kTiles; ++t) {
                float* p = (t < 4 ? din1 : din2) + node * kNnH + 16 * (t & 3) + 4 * lk;
                f32x4_t v = acc[t];
                if (t < 4 && acc1) v += *reinterpret_cast<const f32x4_t*>(p);
                *reinterpret_cast<f32x4_t*>(p) = v;
            }
        }
    }
}

// partial[blk][k][o] = sum over the block's nodes of x_k dpre_o, x = [in1 in2 1]
// with 64 features per input (kTiles = 4 or 8 tiles of 16).
// V_MFMA_F32_16X16X4_F32 with the nodes as the inner dimension: lane group g
// carries node 4 q + g of a wave's four, a lane four consecutive features of
// each input and four consecutive outputs, so rows are read as whole lines
// straight into operand registers (tile t's row i stands for feature 4 i + t,
// its column j of output tile u for output 4 j + u).  kDeep groups of four
// nodes are loaded ahead of the products.  Bound by the matrix cores in FP32;
// the form it replaces (products on the vector units, operands from LDS one
// element at a time) took 1,668 us where this takes 41 us (mean of five
// layers, m = 98,799, n = 262,080).
template <typename AT, int kTiles>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void k_dense_bwd_w(int64_t N, const AT* __restrict__ in1, const AT* __restrict__ in2, const float* __restrict__ dh,
                   const AT* __restrict__ h, float* __restrict__ partial) {
    constexpr int kDeep = 2, kIn = kTiles / 4;
    constexpr int K = kTiles * 16;
    __shared__ __attribute__((aligned(16))) float Wg[(K + 1) * kNnH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lc = lane & 15, lk = lane >> 4;
    f32x4_t acc[kTiles][4], bs = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[t][u] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4_t x[kDeep][kIn], d[kDeep];
    const int64_t step = (int64_t)gridDim.x * 4 * 4 * kDeep;
    auto load = [&](int64_t base) {
#pragma unroll
        for (int q = 0; q < kDeep; ++q) {
            const int64_t node = base + 4 * q + lk;
            const int64_t at = (node < N ? node : N - 1) * kNnH + 4 * lc;
            x[q][0] = load4(in1 + at);
            if constexpr (kIn == 2) x[q][1] = load4(in2 + at);
            d[q] = masked4(dh, h, at);
            if (node >= N) {   // contributes zeros
                d[q] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < kIn; ++k) x[q][k] = d[q];
            }
        }
    };
    int64_t base = ((int64_t)blockIdx.x * 4 + wave) * 4 * kDeep;
    if (base < N) load(base);
    for (; base < N; base += step) {
        f32x4_t xc[kDeep][kIn], dc[kDeep];
#pragma unroll
        for (int q = 0; q < kDeep; ++q) {
#pragma unroll
            for (int k = 0; k < kIn; ++k) xc[q][k] = x[q][k];
            dc[q] = d[q];
        }
        if (base + step < N) load(base + step);
#pragma unroll
        for (int q = 0; q < kDeep; ++q) {
            bs += dc[q];
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(xc[q][t >> 2][t & 3], dc[q][u], acc[t][u], 0, 0, 0);
        }
    }
    bs = sum_groups(bs);
    // D's row i = 4 lk + r of tile t is feature 4 i + t, its column lc of u is
    // output 4 lc + u: four outputs of a feature are 16 bytes
    for (int w = 0; w < 4; ++w) {
        if (wave == w) {
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    f32x4_t* p = reinterpret_cast<f32x4_t*>(
                        &Wg[(64 * (t >> 2) + 16 * lk + 4 * r + (t & 3)) * kNnH + 4 * lc]);
                    const f32x4_t v = {acc[t][0][r], acc[t][1][r], acc[t][2][r], acc[t][3][r]};
                    *p = w ? *p + v : v;
                }
            if (lk == 0) {
                f32x4_t* p = reinterpret_cast<f32x4_t*>(&Wg[K * kNnH + 4 * lc]);
                *p = w ? *p + bs : bs;
            }
        }
        __syncthreads();
    }
    float* out = partial + (int64_t)blockIdx.x * (K + 1) * kNnH;
    for (int t = threadIdx.x; t < (K + 1) * kNnH; t += kB) out[t] = Wg[t];
}

// the same for the input layers (K = 4 row or 2 column features): 16 lanes per
// node, four outputs each, on the vector units; bound by reading dh and h
// (28 us per layer, 501 us before)
template <typename AT, int K>
__global__ __launch_bounds__(256) void k_dense_bwd_w_in(int64_t N, const float* __restrict__ in,
                                                        const float* __restrict__ dh, const AT* __restrict__ h,
                                                        float* __restrict__ partial) {
    __shared__ float red[4][(K + 1) * kNnH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lc = lane & 15, lk = lane >> 4;
    f32x4_t acc[K + 1];
#pragma unroll
    for (int k = 0; k <= K; ++k) acc[k] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 2
    for (int64_t n0 = ((int64_t)blockIdx.x * 4 + wave) * 4; n0 < N; n0 += (int64_t)gridDim.x * 16) {
        const int64_t node = n0 + lk < N ? n0 + lk : N - 1;
        f32x4_t d = masked4(dh, h, node * kNnH + 4 * lc);
        float x[K];
#pragma unroll
        for (int k = 0; k < K; ++k) x[k] = in[node * K + k];
        if (n0 + lk >= N) d = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < K; ++k) acc[k] += x[k] * d;
        acc[K] += d;
    }
#pragma unroll
    for (int k = 0; k <= K; ++k) {
        acc[k] = sum_groups(acc[k]);
        if (lk == 0)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[wave][k * kNnH + 4 * lc + e] = acc[k][e];
    }
    __syncthreads();
    float* out = partial + (int64_t)blockIdx.x * (K + 1) * kNnH;
    for (int t = threadIdx.x; t < (K + 1) * kNnH; t += kB) out[t] = ((red[0][t] + red[1][t]) + red[2][t]) + red[3][t];
}

// out[p] = sum over the blocks of partial[blk][p]: 64 parameters per
// workgroup, 16 waves over the blocks (one chain per thread over all of them
// took 39 us where this takes 5 us)
__global__ __launch_bounds__(1024) void k_reduce_blocks(int npar, int nblk, const float* __restrict__ partial,
                                                        float* __restrict__ out) {
    __shared__ float red[16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    const int pc = p < npar ? p : npar - 1;
    float s = 0.0f;
#pragma unroll 4
    for (int b = wave; b < nblk; b += 16) s += partial[(int64_t)b * npar + pc];
    red[wave][lane] = s;
    __syncthreads();
    if (wave != 0 || p >= npar) return;
    s = 0.0f;
#pragma unroll
    for (int w = 0; w < 16; ++w) s += red[w][lane];
    out[p] = s;
}

// din[src][f] (+)= sum_{p in adjT(src)} valT[p] / deg(idxT[p]) dout[idxT[p]][f],
// laid out as k_mean (38 us per layer, 106 us with a wave per node)
template <bool kAdd>
__global__ __launch_bounds__(256) void k_mean_bwd(int32_t Nsrc, const int64_t* __restrict__ ptrT,
                                                  const int32_t* __restrict__ idxT, const double* __restrict__ valT,
                                                  const int64_t* __restrict__ ptrF, const float* __restrict__ dout,
                                                  float* __restrict__ din) {
    const int64_t t = (int64_t)blockIdx.x * kB + threadIdx.x;
    const int64_t node = t >> 3;
    const int f = 8 * (int)(t & 7);
    if (node >= Nsrc) return;
    const int64_t b = ptrT[node], e = ptrT[node + 1];
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int64_t p = b; p < e; p += 4) {
        float w[4], x[4][8];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t q = p + u < e ? p + u : e - 1;
            const int32_t j = idxT[q];
            const int64_t deg = ptrF[j + 1] - ptrF[j];
            w[u] = (float)valT[q] / (float)(deg > 1 ? deg : 1);
            load8(dout + (int64_t)j * kNnH + f, x[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int k = 0; k < 8; ++k) acc[k] = p + u < e ? acc[k] + w[u] * x[u][k] : acc[k];
    }
    float* o = din + node * kNnH + f;
    if (kAdd) {
        float old[8];
        load8(o, old);
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] += old[k];
    }
    store8(o, acc);
}

__global__ void k_adam(int npar, float* __restrict__ p, const float* __restrict__ g, float* __restrict__ mo,
                       float* __restrict__ ve, float lr, float b1, float b2, float eps, float c1, float c2,
                       int bf16, float* __restrict__ pw) {
    const int i = blockIdx.x * kB + threadIdx.x;
    if (i >= npar) return;
    const float gi = g[i];
    const float m = b1 * mo[i] + (1.0f - b1) * gi;
    const float v = b2 * ve[i] + (1.0f - b2) * gi * gi;
    mo[i] = m;
    ve[i] = v;
    const float np = p[i] - lr * (m / c1) / (sqrtf(v / c2) + eps);
    p[i] = np;
    pw[i] = bf16 ? round_bf16(np) : np;
}

__global__ void k_finite(int32_t m, const double* __restrict__ x, int32_t* __restrict__ flag) {
    const int32_t i = blockIdx.x * kB + threadIdx.x;
    if (i < m && !isfinite(x[i])) *flag = 1;
}

}  // namespace

void nn_features(int32_t m, int32_t n, const double* g, const double* r, const double* dinv, double rs, double mu,
                 double nu, float* xr, float* xc, hipStream_t st) {
    help::launch_kernel(k_feat_row, grid_for(m), kB, 0, st, m, g, r, rs, mu, xr);
    help::launch_kernel(k_feat_col, grid_for(n), kB, 0, st, n, dinv, nu, xc);
}

void nn_stats_partials(int64_t m, int64_t n, const double* g, const double* dinv, const double* r, double* part,
                       int nblk, hipStream_t st) {
    help::launch_kernel(k_stats, dim3(nblk, 3), kB, 0, st, m, n, g, dinv, r, part);
}

template <typename AT>
void nn_dense(int64_t N, const AT* in1, int k1, const AT* in2, int k2, const float* W, const float* b, AT* out,
              hipStream_t st) {
    if (N <= 0) return;
    if constexpr (std::is_same<AT, Bf16>::value) {
        if ((k1 + k2) % 32 == 0 && k1 % 8 == 0 && k1 + k2 <= 2 * kNnH) {
            help::launch_kernel(k_dense_mfma, grid_cap((N + 63) / 64, 2048), kB, 0, st, N, in1, k1, in2, k2, W, b, out);
            return;
        }
    }
    help::launch_kernel(k_dense<AT>, grid_cap((N + 3) / 4, 2048), kB, 0, st, N, in1, k1, in2, k2, W, b, out);
}

template <typename AT, int K>
void nn_dense_in(int64_t N, const float* in, const float* W, const float* b, AT* out, hipStream_t st) {
    if (N > 0) help::launch_kernel(k_dense_in<AT, K>, grid_for(8 * N), kB, 0, st, N, in, W, b, out);
}

void nn_mfma_bf16_probe(const float* a, const float* b, float* out, hipStream_t st) {
    help::launch_kernel(k_mfma_bf16_probe, 1, 64, 0, st, a, b, out);
}

template <typename AT>
void nn_mean(int32_t N, const int64_t* ptr, const int32_t* idx, const double* val, const AT* src, AT* out,
             hipStream_t st) {
    if (N > 0) help::launch_kernel(k_mean<AT>, grid_for(8 * (int64_t)N), kB, 0, st, N, ptr, idx, val, src, out);
}

template <typename AT>
void nn_output(int32_t m, const AT* z, const float* wo, const float* bo, const double* g, double rs, float* y,
               double* x0, hipStream_t st) {
    if (m > 0) help::launch_kernel(k_output<AT>, (m + 31) / 32, kB, 0, st, m, z, wo, bo, g, rs, y, x0);
}

void nn_loss_partials(int32_t m, const float* y, const double* dy, const double* g, double rs, double* part,
                      int nblk, hipStream_t st) {
    help::launch_kernel(k_loss, nblk, kB, 0, st, m, y, dy, g, rs, part);
}

void nn_output_grad(int32_t m, const float* y, const double* dy, const double* g, double rs, double T, float* dyv,
                    hipStream_t st) {
    if (m > 0) help::launch_kernel(k_out_grad, grid_for(m), kB, 0, st, m, y, dy, g, rs, T, dyv);
}

template <typename AT>
void nn_out_bwd(int32_t m, const AT* z, const float* dyv, const float* wo, float* dpre, hipStream_t st) {
    if (m > 0) help::launch_kernel(k_out_bwd<AT>, grid_for((int64_t)m * kNnH), kB, 0, st, m, z, dyv, wo, dpre);
}

// one block per 64 nodes (each of its waves then has 16), at most two per CU
int nn_wgrad_blocks(int64_t N) { return grid_cap((N + 63) / 64, kNnMaxBlocks); }

template <typename AT>
void nn_out_w(int32_t m, const AT* z, const float* dyv, float* partial, hipStream_t st) {
    if (m > 0) help::launch_kernel(k_out_w<AT>, nn_wgrad_blocks(m), kB, 0, st, m, z, dyv, partial);
}

template <typename AT>
void nn_dense_bwd_in(int64_t N, const float* dh, const AT* h, const float* W, float* din1, float* din2,
                     bool accumulate1, hipStream_t st) {
    if (N <= 0) return;
    const int nb = grid_cap((N + 63) / 64, kNnMaxBlocks);
    if (din2) help::launch_kernel(k_dense_bwd_in<AT, 8>, nb, kB, 0, st, N, dh, h, W, din1, din2, accumulate1 ? 1 : 0);
    else help::launch_kernel(k_dense_bwd_in<AT, 4>, nb, kB, 0, st, N, dh, h, W, din1, din2, accumulate1 ? 1 : 0);
}

template <typename AT>
void nn_dense_bwd_w(int64_t N, const AT* in1, const AT* in2, const float* dh, const AT* h, float* partial,
                    hipStream_t st) {
    if (N <= 0) return;
    if (in2) help::launch_kernel(k_dense_bwd_w<AT, 8>, nn_wgrad_blocks(N), kB, 0, st, N, in1, in2, dh, h, partial);
    else help::launch_kernel(k_dense_bwd_w<AT, 4>, nn_wgrad_blocks(N), kB, 0, st, N, in1, in2, dh, h, partial);
}

template <typename AT, int K>
void nn_dense_bwd_w_in(int64_t N, const float* in, const float* dh, const AT* h, float* partial, hipStream_t st) {
    if (N > 0) help::launch_kernel(k_dense_bwd_w_in<AT, K>, nn_wgrad_blocks(N), kB, 0, st, N, in, dh, h, partial);
}

void nn_reduce_blocks(int npar, int nblk, const float* partial, float* out, hipStream_t st) {
    help::launch_kernel(k_reduce_blocks, (npar + 63) / 64, 1024, 0, st, npar, nblk, partial, out);
}

void nn_mean_bwd(int32_t Nsrc, const int64_t* ptrT, const int32_t* idxT, const double* valT, const int64_t* ptrF,
                 const float* dout, float* din, bool accumulate, hipStream_t st) {
    if (Nsrc <= 0) return;
    const int nb = grid_for(8 * (int64_t)Nsrc);
    if (accumulate) help::launch_kernel(k_mean_bwd<true>, nb, kB, 0, st, Nsrc, ptrT, idxT, valT, ptrF, dout, din);
    else help::launch_kernel(k_mean_bwd<false>, nb, kB, 0, st, Nsrc, ptrT, idxT, valT, ptrF, dout, din);
}

void nn_adam(int npar, float* p, const float* g, float* mo, float* ve, float lr, float b1, float b2, float eps,
             int t, int bf16, float* pw, hipStream_t st) {
    const float c1 = 1.0f - std::pow(b1, (float)t), c2 = 1.0f - std::pow(b2, (float)t);
    help::launch_kernel(k_adam, grid_for(npar), kB, 0, st, npar, p, g, mo, ve, lr, b1, b2, eps, c1, c2, bf16, pw);
}

void nn_check_finite(int32_t m, const double* x, int32_t* flag, hipStream_t st) {
    if (m > 0) help::launch_kernel(k_finite, grid_for(m), kB, 0, st, m, x, flag);
}

#define NN_INST(AT)                                                                                              \
    template void nn_dense<AT>(int64_t, const AT*, int, const AT*, int, const float*, const float*, AT*,       \
                                   hipStream_t);                                                                 \
    template void nn_mean<AT>(int32_t, const int64_t*, const int32_t*, const double*, const AT*, AT*, hipStream_t); \
    template void nn_output<AT>(int32_t, const AT*, const float*, const float*, const double*, double, float*,     \
                                double*, hipStream_t);                                                           \
    template void nn_out_bwd<AT>(int32_t, const AT*, const float*, const float*, float*, hipStream_t);            \
    template void nn_out_w<AT>(int32_t, const AT*, const float*, float*, hipStream_t);                           \
    template void nn_dense_bwd_in<AT>(int64_t, const float*, const AT*, const float*, float*, float*, bool,       \
                                      hipStream_t);                                                              \
    template void nn_dense_bwd_w<AT>(int64_t, const AT*, const AT*, const float*, const AT*, float*, hipStream_t); \
    template void nn_dense_in<AT, kNnFR>(int64_t, const float*, const float*, const float*, AT*, hipStream_t);    \
    template void nn_dense_in<AT, kNnFC>(int64_t, const float*, const float*, const float*, AT*, hipStream_t);    \
    template void nn_dense_bwd_w_in<AT, kNnFR>(int64_t, const float*, const float*, const AT*, float*, hipStream_t); \
    template void nn_dense_bwd_w_in<AT, kNnFC>(int64_t, const float*, const float*, const AT*, float*, hipStream_t);
NN_INST(float)
NN_INST(Bf16)
#undef NN_INST

}  // namespace help
