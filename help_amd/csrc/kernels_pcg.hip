// Kernels of the matrix-free PCG path (HELP PCG.cpp:38-395).
//
// * Row-split CSR products: A has rows of wildly different lengths (Zipf row
//   popularity gives rows with millions of nonzeros), so rows up to
//   kLightRow nonzeros take a thread, rows up to kHeavyRow a wave, and
//   longer rows are cut into chunks, a workgroup each, combined in chunk order:
//   deterministic.
// * Greedy partial Cholesky (PCG.cpp:38-103): per pivot an argmax over the
//   Schur diagonal; the candidates' rows of A scattered into n-vectors, their
//   columns of ADA^T and their left-looking updates against the previous
//   columns, in blocks of kPcBlk or pivot by pivot (column-major m x K factor,
//   so the thread-per-row update reads coalesced).
// * Preconditioner apply (PCG.cpp:183-196) with the factor in FP32: the
//   product and the transposed product, a pass over the m x K factor each.
#include <algorithm>
#include <climits>
#include <cmath>

#include "device.h"
#include "launch.h"
#include "pcg.h"

namespace help {

namespace {

constexpr int kB = 256;
inline int grid_for(int64_t n) { return (int)std::max<int64_t>(1, (n + kB - 1) / kB); }

__device__ inline double block_sum(double v, double* red) {
    const int t = threadIdx.x;
    red[t] = v;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) red[t] += red[t + w];
        __syncthreads();
    }
    const double s = red[0];
    __syncthreads();
    return s;
}

__device__ inline double wave_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// ------------------------------------------------------ row-split products
template <bool SQ>
__global__ __launch_bounds__(256) void k_csr_light(int32_t m, const int64_t* __restrict__ rowptr,
                                                   const int32_t* __restrict__ colind,
                                                   const double* __restrict__ val,
                                                   const double* __restrict__ x, double* __restrict__ y) {
    const int32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= m) return;
    const int64_t b = rowptr[i], e = rowptr[i + 1];
    if (e - b > kLightRow) return;
    // 8 terms' loads in flight (indices past the row clamped, terms dropped)
    double acc = 0.0;
    for (int64_t p = b; p < e; p += 8) {
        double t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int64_t q = p + u < e ? p + u : e - 1;
            const double v = val[q];
            t[u] = (SQ ? v * v : v) * x[colind[q]];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) acc = (p + u < e) ? acc + t[u] : acc;
    }
    y[i] = acc;
}

// a wave per medium row: lane-strided partial sums with four terms in
// flight, combined by a fixed butterfly
template <bool SQ>
__global__ __launch_bounds__(256) void k_csr_medium(int32_t nmed, const int32_t* __restrict__ mrow,
                                                    const int64_t* __restrict__ rowptr,
                                                    const int32_t* __restrict__ colind,
                                                    const double* __restrict__ val,
                                                    const double* __restrict__ x, double* __restrict__ y) {
    const int32_t h = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (h >= nmed) return;
    const int32_t i = mrow[h];
    const int64_t b = rowptr[i], e = rowptr[i + 1];
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    for (int64_t p0 = b + lane; p0 < e; p0 += 256) {
        double t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t q = p0 + 64 * u < e ? p0 + 64 * u : e - 1;
            const double v = val[q];
            t[u] = (SQ ? v * v : v) * x[colind[q]];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) a[u] = (p0 + 64 * u < e) ? a[u] + t[u] : a[u];
    }
    const double s = wave_sum((a[0] + a[1]) + (a[2] + a[3]));
    if (lane == 0) y[i] = s;
}

// A workgroup per chunk of a heavy row, eight terms per thread in flight.
// Bound by the gathers of x; the chunks are listed by column and XCD
// (RowSplitDev).  12.1 million nonzeros of 1,181 rows, x of 32 MB: 123 us; in
// row order with one term per thread in flight, 150 us.  (A wave per chunk,
// cut at blocks of 262,144 columns, took 70 us, and rounds differently: a solve
// that stops at 1e-10 then ends up to 1e-7 of an entry away.)
template <bool SQ>
__global__ __launch_bounds__(256) void k_csr_chunk(const RowChunk* __restrict__ chunks,
                                                   const int32_t* __restrict__ colind,
                                                   const double* __restrict__ val,
                                                   const double* __restrict__ x, double* __restrict__ part) {
    __shared__ double red[4][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const RowChunk c = chunks[blockIdx.x];
    if (c.e <= c.b) return;   // padding
    double a = 0.0;
    for (int64_t p0 = c.b + tid; p0 < c.e; p0 += 2048) {
        double v[8], g[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int64_t q = p0 + 256 * u < c.e ? p0 + 256 * u : c.e - 1;
            v[u] = val[q];
            g[u] = x[colind[q]];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double t = (SQ ? v[u] * v[u] : v[u]) * g[u];
            a = (p0 + 256 * u < c.e) ? a + t : a;
        }
    }
    red[wave][lane] = a;
    __syncthreads();
    if (wave != 0) return;
    const double s = wave_sum((red[0][lane] + red[2][lane]) + (red[1][lane] + red[3][lane]));
    if (lane == 0) part[c.slot] = s;
}

// a wave per heavy row: its chunk partials summed lane-strided, fixed tree
__global__ __launch_bounds__(256) void k_csr_heavy(int32_t nheavy, const int32_t* __restrict__ hrow,
                                                   const int32_t* __restrict__ hptr,
                                                   const double* __restrict__ part, double* __restrict__ y) {
    const int32_t h = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (h >= nheavy) return;
    double acc = 0.0;
    for (int32_t c = hptr[h] + lane; c < hptr[h + 1]; c += 64) acc += part[c];
    const double s = wave_sum(acc);
    if (lane == 0) y[hrow[h]] = s;
}

// t_j = dinv_j times the sum of column j's products, row after row.  The
// workgroup loads the values and their x kCscChunk at a time with the lanes
// along them, and each thread adds its column's from LDS (one position in 17
// left free, so that columns of equal length do not start in the same banks).
// Bound by the gathers of x.  19 million nonzeros in columns of 6 and 1, x of
// 8 MB: 96 us, 119 us when each thread read its own column.
constexpr int kCscChunk = 1024;
// place of nonzero p in the chunk that starts at c0, or its nearer end
__device__ inline int chunk_place(int64_t p, int64_t c0) {
    const int64_t q = p - c0;
    return (int)(q < 0 ? 0 : q < kCscChunk ? q : kCscChunk);
}
__global__ __launch_bounds__(256) void k_csc_ts(int32_t n, const int64_t* __restrict__ colptr,
                                                const int32_t* __restrict__ rowind, const double* __restrict__ val,
                                                const double* __restrict__ dinv, const double* __restrict__ x,
                                                double* __restrict__ t) {
    __shared__ double bv[kCscChunk + kCscChunk / 16], bx[kCscChunk + kCscChunk / 16];
    const int tid = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * kB, j = first + tid;
    const int64_t gb = colptr[first], ge = colptr[first + kB < n ? first + kB : n];
    const int64_t b = colptr[j < n ? j : n], e = colptr[j + 1 < n ? j + 1 : n];
    auto pos = [](int q) { return q + (q >> 4); };
    double acc = 0.0;
    for (int64_t c0 = gb; c0 < ge; c0 += kCscChunk) {
        double v[kCscChunk / kB], g[kCscChunk / kB];
#pragma unroll
        for (int u = 0; u < kCscChunk / kB; ++u) {
            if (c0 + u * kB < ge) {
                const int64_t q = c0 + u * kB + tid < ge ? c0 + u * kB + tid : ge - 1;
                v[u] = val[q];
                g[u] = x[rowind[q]];
            }
        }
        if (c0 > gb) __syncthreads();   // the last chunk has been added
#pragma unroll
        for (int u = 0; u < kCscChunk / kB; ++u)
            if (c0 + u * kB < ge) {
                bv[pos(u * kB + tid)] = v[u];
                bx[pos(u * kB + tid)] = g[u];
            }
        __syncthreads();
        const int lo = chunk_place(b, c0), hi = chunk_place(e, c0);
        for (int q = lo; q < hi; q += 4) {
            double w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int p = pos(q + u < hi ? q + u : hi - 1);
                w[u] = bv[p] * bx[p];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) acc = (q + u < hi) ? acc + w[u] : acc;
        }
    }
    if (j < n) t[j] = acc * dinv[j];
}

// ---------------------------------------------------- partial Cholesky build
__device__ inline bool better(double v, int32_t i, double bv, int32_t bi) {
    return v > bv || (v == bv && i < bi);
}

// A group of pivots starts with kPcBlk candidates, the largest Schur diagonals
// (ties to the lowest position), and is formed in one of two ways:
// * as a block: the candidates' columns of A D^-1 A^T and their left-looking
//   sums over all finished factor columns together, so the m x k factor and A
//   are read once per block instead of once per pivot.  Each step then takes the
//   largest Schur diagonal of all and adds the block's own columns; when that
//   pivot is none of the candidates the block ends there.
// * pivot by pivot: each step takes the largest Schur diagonal, whatever row it
//   is, then forms its product with A and its sums.
// Either way the state counts the leading pivots that were candidates
// (PcState::taken), from which the host chooses the next group's form
// (pcg_renew).  Rows in groups of more than kPcBlk near-parallel ones with
// similar diagonals lose all other candidates to the first pivot, and a block of
// one pivot costs more than a single one (kPcFew).
// The order of the pivots is the greedy one whatever the groups, and a column's
// sum over the earlier ones keeps its four interleaved chains (PCG.cpp:85-102
// in that order), so every column rounds the same in both forms.  The state
// stays on the device: every kernel of a block returns at once when it has
// ended.
// m = 10^6, K = 500 (zipf): 63.4 ms per build, 328 ms with a search, a product
// and the sums per pivot (of which the factor reads take 178 ms and the
// products with A 136 ms).  Rows in groups of 20 near-parallel ones: 386 ms;
// 390 ms per pivot, 637 ms in blocks alone.  m = 30,000, K = 77: 2.1 ms; 2.2
// per pivot, 12.7 in blocks alone.
typedef PcBest Best;
__device__ inline bool ahead(const Best& a, const Best& b) { return better(a.v, a.pos, b.v, b.pos); }

__device__ inline Best block_best(Best x, Best (&red)[kB / 64]) {
    for (int off = 32; off > 0; off >>= 1) {
        const Best o = {__shfl_xor(x.v, off), __shfl_xor(x.pos, off), __shfl_xor(x.row, off)};
        if (ahead(o, x)) x = o;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
    __syncthreads();
    Best b = red[0];
#pragma unroll
    for (int w = 1; w < kB / 64; ++w)
        if (ahead(red[w], b)) b = red[w];
    __syncthreads();
    return b;
}

// the workgroup's kPcBlk best rows not yet pivoted, in order; the first one is also
// its argmax partial
__global__ __launch_bounds__(256) void k_pc_top_part(int32_t m, const int32_t* __restrict__ pos,
                                                     const double* __restrict__ S, const PcState* __restrict__ st,
                                                     PcBest* __restrict__ top, PcBest* __restrict__ arg) {
    __shared__ Best red[kB / 64];
    const int32_t k = st->k;
    const Best none = {-HUGE_VAL, INT_MAX, -1};
    // this thread's best row strictly behind `last`
    auto next = [&](const Best& last) {
        Best b = none;
        for (int64_t j = (int64_t)blockIdx.x * kB + threadIdx.x; j < m; j += (int64_t)gridDim.x * kB) {
            const Best c = {S[j], pos[j], (int32_t)j};
            if (c.pos >= k && ahead(last, c) && ahead(c, b)) b = c;
        }
        return b;
    };
    Best mine = next({HUGE_VAL, -1, -1});
    for (int r = 0; r < kPcBlk; ++r) {
        const Best b = block_best(mine, red);
        if (threadIdx.x == 0) {
            top[blockIdx.x * kPcBlk + r] = b;
            if (r == 0) arg[blockIdx.x] = b;
        }
        if (b.row >= 0 && b.row == mine.row) mine = next(b);
    }
}

// the candidates of the next group out of nb workgroups' best
__global__ __launch_bounds__(256) void k_pc_top_pick(int32_t nb, int32_t K, const PcBest* __restrict__ top,
                                                     PcState* __restrict__ st) {
    constexpr int kPer = kTopBlocks / kB;   // lists per thread, each in order
    __shared__ Best red[kB / 64];
    const Best none = {-HUGE_VAL, INT_MAX, -1};
    int at[kPer];
    Best head[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int b = threadIdx.x + u * kB;
        at[u] = 0;
        head[u] = b < nb ? top[b * kPcBlk] : none;
    }
    for (int r = 0; r < kPcBlk; ++r) {
        Best mine = none;
#pragma unroll
        for (int u = 0; u < kPer; ++u)
            if (head[u].row >= 0 && ahead(head[u], mine)) mine = head[u];
        const Best b = block_best(mine, red);
        if (threadIdx.x == 0) st->cand[r] = b.row;
#pragma unroll
        for (int u = 0; u < kPer; ++u)
            if (b.row >= 0 && head[u].row == b.row)
                head[u] = ++at[u] < kPcBlk ? top[(threadIdx.x + u * kB) * kPcBlk + at[u]] : none;
    }
    if (threadIdx.x == 0) {
        st->k0 = st->k;
        st->taken = 0;
        st->stop = st->k >= K;
    }
}

// sc[j][c] = A(cand_c, j) dinv_j on the candidates' rows (blockIdx.y = c), or 0;
// one: sc[j] on the pivot's row (k_pc_column clears it)
__global__ void k_pc_scatter(const PcState* __restrict__ st, int one, const int64_t* __restrict__ rowptr,
                             const int32_t* __restrict__ colind, const double* __restrict__ val,
                             const double* __restrict__ dinv, double* __restrict__ sc, int clear) {
    const int c = blockIdx.y;
    const int32_t col = one ? st->col : st->cand[c];
    if (st->stop || col < 0) return;
    const int stride = one ? 1 : kPcBlk;
    const int64_t b = rowptr[col], e = rowptr[col + 1];
    for (int64_t p = b + (int64_t)blockIdx.x * kB + threadIdx.x; p < e; p += (int64_t)gridDim.x * kB) {
        const int32_t j = colind[p];
        sc[(int64_t)j * stride + c] = clear ? 0.0 : val[p] * dinv[j];
    }
}

// g[c][i] = sum_p val[p] sc[colind[p]][c]: the products of A with all candidates'
// vectors, the candidate on the low lanes, so a nonzero's gather is one
// 64-byte line.  Rows by length as in the single products.
__global__ __launch_bounds__(256) void k_pc_csr_light(int32_t m, const PcState* __restrict__ st,
                                                      const int64_t* __restrict__ rowptr,
                                                      const int32_t* __restrict__ colind,
                                                      const double* __restrict__ val, const double* __restrict__ sc,
                                                      double* __restrict__ g) {
    const int64_t t = (int64_t)blockIdx.x * kB + threadIdx.x;
    const int64_t i = t / kPcBlk;
    const int c = (int)(t % kPcBlk);
    if (st->stop || i >= m) return;
    const int64_t b = rowptr[i], e = rowptr[i + 1];
    if (e - b > kLightRow) return;
    double acc = 0.0;
    for (int64_t p = b; p < e; p += 4) {
        double x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t q = p + u < e ? p + u : e - 1;
            x[u] = val[q] * sc[(int64_t)colind[q] * kPcBlk + c];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) acc = (p + u < e) ? acc + x[u] : acc;
    }
    g[(int64_t)c * m + i] = acc;
}

// sum of a run of terms of one row for the block's kPcBlk columns (sc: kPcBlk
// values per column of A), on lane c for column c: every column has the
// accumulators of k_csr_medium (kChunk: of k_csr_chunk), four per lane, and
// their combine order, so it rounds as a product of its own
template <bool kChunk>
__device__ __forceinline__ double wave_range(int64_t b, int64_t e, const int32_t* __restrict__ colind,
                                             const double* __restrict__ val, const double* __restrict__ sc, int lane) {
    double a[kPcBlk][4] = {};
    for (int64_t p0 = b + lane; p0 < e; p0 += 256) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t q = p0 + 64 * u;
            if (q < e) {
                const double v = val[q];
                const double* g = sc + (int64_t)colind[q] * kPcBlk;
#pragma unroll
                for (int c = 0; c < kPcBlk; ++c) a[c][u] += v * g[c];
            }
        }
    }
    double out = 0.0;
#pragma unroll
    for (int c = 0; c < kPcBlk; ++c) {
        const double s = kChunk ? wave_sum((a[c][0] + a[c][2]) + (a[c][1] + a[c][3]))
                                : wave_sum((a[c][0] + a[c][1]) + (a[c][2] + a[c][3]));
        out = lane == c ? s : out;
    }
    return out;
}

__global__ __launch_bounds__(256) void k_pc_csr_medium(int32_t m, int32_t nmed, const int32_t* __restrict__ mrow,
                                                       const PcState* __restrict__ st,
                                                       const int64_t* __restrict__ rowptr,
                                                       const int32_t* __restrict__ colind,
                                                       const double* __restrict__ val, const double* __restrict__ sc,
                                                       double* __restrict__ g) {
    const int32_t h = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (st->stop || h >= nmed) return;
    const int32_t i = mrow[h];
    const double s = wave_range<false>(rowptr[i], rowptr[i + 1], colind, val, sc, lane);
    if (lane < kPcBlk) g[(int64_t)lane * m + i] = s;
}

__global__ __launch_bounds__(256) void k_pc_csr_chunk(int32_t nchunk, const RowChunk* __restrict__ chunks,
                                                      const PcState* __restrict__ st,
                                                      const int32_t* __restrict__ colind,
                                                      const double* __restrict__ val, const double* __restrict__ sc,
                                                      double* __restrict__ part) {
    // workgroup b takes four chunks of XCD b mod 8's run
    const int32_t i = (blockIdx.x / kXcds * 4 + (threadIdx.x >> 6)) * kXcds + blockIdx.x % kXcds;
    const int lane = threadIdx.x & 63;
    if (st->stop || i >= nchunk) return;
    const RowChunk c = chunks[i];
    if (c.e <= c.b) return;   // padding
    const double s = wave_range<true>(c.b, c.e, colind, val, sc, lane);
    if (lane < kPcBlk) part[(int64_t)c.slot * kPcBlk + lane] = s;
}

// a workgroup per heavy row
__global__ __launch_bounds__(256) void k_pc_csr_heavy(int32_t m, const int32_t* __restrict__ hrow,
                                                      const int32_t* __restrict__ hptr,
                                                      const PcState* __restrict__ st,
                                                      const double* __restrict__ part, double* __restrict__ g) {
    // a wave per kPcBlk / 4 columns, as k_csr_heavy
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (st->stop) return;
#pragma unroll
    for (int k = 0; k < kPcBlk / 4; ++k) {
        const int c = wave * (kPcBlk / 4) + k;
        double acc = 0.0;
        for (int32_t q = hptr[blockIdx.x] + lane; q < hptr[blockIdx.x + 1]; q += 64)
            acc += part[(int64_t)q * kPcBlk + c];
        const double s = wave_sum(acc);
        if (lane == 0) g[(int64_t)c * m + hrow[blockIdx.x]] = s;
    }
}

// wb[r][c] = D_r L(cand_c, r) for the finished columns r
__global__ void k_pc_weights(int32_t m, const PcState* __restrict__ st, const double* __restrict__ D,
                             const double* __restrict__ L, double* __restrict__ wb) {
    const int32_t t = blockIdx.x * kB + threadIdx.x;
    const int32_t r = t / kPcBlk, c = t % kPcBlk;
    if (st->stop || r >= st->k0) return;
    const int32_t row = st->cand[c];
    wb[t] = row >= 0 ? D[r] * L[(int64_t)r * m + row] : 0.0;
}

// acc[c][q][j] = sum over r < k0 - k0 % 4, r = q (mod 4), of L(j,r) wb[r][c]:
// every finished column read once for all candidates, 4 kPcBlk chains per row in
// registers.  Bound by reading the factor.
__global__ __launch_bounds__(256) void k_pc_block(int32_t m, const PcState* __restrict__ st,
                                                  const int32_t* __restrict__ pos, const double* __restrict__ wb,
                                                  const double* __restrict__ L, double* __restrict__ acc) {
    const int32_t j = blockIdx.x * kB + threadIdx.x;
    if (st->stop || j >= m) return;
    const int32_t k0 = st->k0, kb = k0 & ~3;
    if (pos[j] < k0) return;
    double a[kPcBlk][4];
#pragma unroll
    for (int c = 0; c < kPcBlk; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) a[c][q] = 0.0;
    double l[2][4] = {};   // this group of four columns and the next one
    if (kb > 0) {          // (there may be fewer than four columns in all)
#pragma unroll
        for (int q = 0; q < 4; ++q) l[0][q] = L[(int64_t)q * m + j];
    }
    for (int32_t r = 0; r < kb; r += 8) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int32_t rr = r + 4 * h;
            if (rr >= kb) break;
            const int32_t nx = min(rr + 4, kb - 4);
#pragma unroll
            for (int q = 0; q < 4; ++q) l[h ^ 1][q] = L[(int64_t)(nx + q) * m + j];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int c = 0; c < kPcBlk; ++c) a[c][q] += l[h][q] * wb[(rr + q) * kPcBlk + c];
        }
    }
#pragma unroll
    for (int c = 0; c < kPcBlk; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[(int64_t)(4 * c + q) * m + j] = a[c][q];
}

// The next pivot: the best of np partials.  In a block (one = 0), done or none of
// the candidates: the block stops.  Else it is swapped to position k and
// w_r = D_r L(col, r) for r < k; s = sum_r w_r L(col, r).
__global__ __launch_bounds__(256) void k_pc_pivot(int32_t m, int32_t K, int one, int32_t np,
                                                  const PcBest* __restrict__ arg, PcState* __restrict__ st,
                                                  int32_t* __restrict__ perm, int32_t* __restrict__ pos,
                                                  const double* __restrict__ L, const double* __restrict__ D,
                                                  double* __restrict__ w) {
    __shared__ Best redb[kB / 64];
    __shared__ double red[kB];
    if (st->stop) return;
    const int32_t k = st->k, before = k - st->k0, taken = st->taken;
    Best mine = {-HUGE_VAL, INT_MAX, -1};
    for (int i = threadIdx.x; i < np; i += kB) {
        const Best c = arg[i];
        if (c.row >= 0 && ahead(c, mine)) mine = c;
    }
    Best b = block_best(mine, redb);
    // no row is ahead of none (every value left is NaN): the row at position k
    if (b.row < 0 && k < K) b = {0.0, k, perm[k]};
    int ci = -1;
#pragma unroll
    for (int c = 0; c < kPcBlk; ++c)
        if (k < K && st->cand[c] == b.row) ci = c;
    __syncthreads();   // every thread has read the state
    if (k >= K || (ci < 0 && !one)) {
        if (threadIdx.x == 0) st->stop = 1;
        return;
    }
    const int32_t col = b.row;
    double acc = 0.0;
    for (int32_t r = threadIdx.x; r < k; r += kB) {
        const double l = L[(int64_t)r * m + col];
        const double wr = D[r] * l;
        w[r] = wr;
        acc += wr * l;
    }
    const double s = block_sum(acc, red);
    if (threadIdx.x == 0) {
        const int32_t a = perm[k];
        perm[k] = col;
        perm[b.pos] = a;
        pos[a] = b.pos;
        pos[col] = k;
        st->col = col;
        st->ci = one ? 0 : ci;
        st->s = s;
        st->k = k + 1;
        if (ci >= 0 && taken == before) st->taken = taken + 1;
    }
}

// D_k = g(col) - s, and column k of L over all rows: 1 at the pivot, 0 at
// earlier pivots, else (g_j - sum_r L(j,r) w_r) / D_k; the Schur diagonal loses
// D_k L(j,k)^2; the best row left of every workgroup.  kBlock: the sums over the
// columns before the block are there (accs).  Else the pivot's vector is cleared.
template <bool kBlock>
__global__ __launch_bounds__(256) void k_pc_column(int32_t m, const PcState* __restrict__ st,
                                                   const int32_t* __restrict__ pos, const double* __restrict__ g,
                                                   const double* __restrict__ accs, const double* __restrict__ wg,
                                                   double* __restrict__ D, double* __restrict__ L,
                                                   float* __restrict__ L32, int64_t ld32, double* __restrict__ S,
                                                   PcBest* __restrict__ arg, const int64_t* __restrict__ rowptr,
                                                   const int32_t* __restrict__ colind, double* __restrict__ sc) {
    __shared__ Best red[kB / 64];
    if (st->stop) return;
    const int32_t k = st->k - 1, kb = kBlock ? st->k0 & ~3 : 0, col = st->col, ci = st->ci;
    const double dk = g[(int64_t)ci * m + col] - st->s;
    if (blockIdx.x == 0 && threadIdx.x == 0) D[k] = dk;
    if constexpr (!kBlock) {
        for (int64_t p = rowptr[col] + (int64_t)blockIdx.x * kB + threadIdx.x; p < rowptr[col + 1]; p += (int64_t)gridDim.x * kB)
            sc[colind[p]] = 0.0;
    }
    Best best = {-HUGE_VAL, INT_MAX, -1};
    for (int64_t j = (int64_t)blockIdx.x * kB + threadIdx.x; j < m; j += (int64_t)gridDim.x * kB) {
        double l = 0.0;
        const int32_t pj = pos[j];
        if (j == col) {
            l = 1.0;
        } else if (pj >= k) {
            double a[4] = {};
            if constexpr (kBlock) {
#pragma unroll
                for (int q = 0; q < 4; ++q) a[q] = accs[(int64_t)(4 * ci + q) * m + j];
            }
            int32_t r = kb;
            for (; r + 3 < k; r += 4)
#pragma unroll
                for (int q = 0; q < 4; ++q) a[q] += L[(int64_t)(r + q) * m + j] * wg[r + q];
            for (; r < k; ++r) a[0] += L[(int64_t)r * m + j] * wg[r];
            const double u = g[(int64_t)ci * m + j] - ((a[0] + a[1]) + (a[2] + a[3]));
            l = u / dk;
            const double sj = S[j] - dk * l * l;
            S[j] = sj;
            const Best c = {sj, pj, (int32_t)j};
            if (ahead(c, best)) best = c;
        }
        L[(int64_t)k * m + j] = l;
        if (L32) L32[(int64_t)k * ld32 + j] = (float)l;
    }
    const Best b = block_best(best, red);
    if (threadIdx.x == 0) arg[blockIdx.x] = b;
}

// L11 (row-major K x K, rows = pivots in order) and X = L11^-1 by columns:
// thread c solves L11 x = e_c forward (unit diagonal)
__global__ void k_pc_l11_gather(int32_t m, int32_t K, const int32_t* __restrict__ perm,
                                const double* __restrict__ L, double* __restrict__ L11) {
    const int64_t idx = (int64_t)blockIdx.x * kB + threadIdx.x;
    if (idx >= (int64_t)K * K) return;
    const int32_t i = (int32_t)(idx / K), c = (int32_t)(idx % K);
    L11[idx] = (c <= i) ? L[(int64_t)c * m + perm[i]] : 0.0;
}

// Column c of X = L11^-1 (unit lower) by forward substitution, a wave per
// column: the column lives in LDS, row i's dot over t in [c, i) has the
// lanes over t (coalesced reads of row i of L11) and a fixed reduction.
__global__ __launch_bounds__(256) void k_pc_l11_inv(int32_t K, const double* __restrict__ L11,
                                                    double* __restrict__ X) {
    __shared__ double xs[4][kPcgMaxK];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int32_t c = blockIdx.x * 4 + wave;
    if (c >= K) return;
    double* x = xs[wave];
    for (int32_t i = lane; i < K; i += 64) x[i] = (i == c) ? 1.0 : 0.0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int32_t i = c + 1; i < K; ++i) {
        const double* Li = L11 + (int64_t)i * K;
        double a0 = 0.0, a1 = 0.0;
        int32_t t = c + lane;
        for (; t + 64 < i; t += 128) {
            a0 += Li[t] * x[t];
            a1 += Li[t + 64] * x[t + 64];
        }
        if (t < i) a0 += Li[t] * x[t];
        const double s = wave_sum(a0 + a1);
        if (lane == 0) x[i] = -s;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    for (int32_t i = lane; i < K; i += 64) X[(int64_t)i * K + c] = x[i];
}

__global__ void k_vdiv(int64_t n, const double* __restrict__ a, const double* __restrict__ b,
                       double* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * kB + threadIdx.x;
    if (i < n) out[i] = a[i] / b[i];
}

// ------------------------------------------------------ preconditioner apply
// y1 = L11^-1 r(pivots)
__global__ __launch_bounds__(256) void k_pca_y1(int32_t K, const int32_t* __restrict__ perm,
                                                const double* __restrict__ X, const double* __restrict__ r,
                                                double* __restrict__ y1) {
    // a wave per row i of X (lanes over the columns, coalesced)
    const int32_t i = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (i >= K) return;
    double a0 = 0.0, a1 = 0.0;
    int32_t c = lane;
    for (; c + 64 <= i; c += 128) {
        a0 += X[(int64_t)i * K + c] * r[perm[c]];
        a1 += X[(int64_t)i * K + c + 64] * r[perm[c + 64]];
    }
    if (c <= i) a0 += X[(int64_t)i * K + c] * r[perm[c]];
    const double s = wave_sum(a0 + a1);
    if (lane == 0) y1[i] = s;
}

// z_j = (r_j - sum_c L(j,c) y1_c) / S_j off the pivots, 0 on them; the
// factor in FP32 (the default) or FP64, the sums in FP64
template <typename T>
__global__ __launch_bounds__(256) void k_pca_t2(int32_t m, int64_t ld, int32_t K, const int32_t* __restrict__ pos,
                                                const T* __restrict__ L32, const double* __restrict__ y1g,
                                                const double* __restrict__ S, const double* __restrict__ r,
                                                double* __restrict__ z) {
    __shared__ double y1[kPcgMaxK];
    for (int c = threadIdx.x; c < K; c += kB) y1[c] = y1g[c];
    __syncthreads();
    const int32_t j = blockIdx.x * kB + threadIdx.x;
    if (j >= m) return;
    if (pos[j] < K) { z[j] = 0.0; return; }
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    int32_t c = 0;
    for (; c + 3 < K; c += 4) {
        a0 += (double)L32[(int64_t)c * ld + j] * y1[c];
        a1 += (double)L32[(int64_t)(c + 1) * ld + j] * y1[c + 1];
        a2 += (double)L32[(int64_t)(c + 2) * ld + j] * y1[c + 2];
        a3 += (double)L32[(int64_t)(c + 3) * ld + j] * y1[c + 3];
    }
    for (; c < K; ++c) a0 += (double)L32[(int64_t)c * ld + j] * y1[c];
    z[j] = (r[j] - ((a0 + a1) + (a2 + a3))) / S[j];
}

// ltpart[c * nb + b] = sum over the kLtRows rows of block b of L(j,c) z_j
// (z is 0 on the pivots); a wave per column, 32 rows per lane in flight.
// gridDim.y workgroups share the columns of a block where that leaves at most
// kLtGroups (m = 31,415, K = 77, 16 blocks: 7.2 us, 35 us with one each;
// m = 10^6, K = 500, 489 blocks: 342 us with one each, 367 with four)
template <typename T>
__global__ __launch_bounds__(256) void k_pca_lt(int32_t m, int64_t ld, int32_t K, const T* __restrict__ L32,
                                                const double* __restrict__ z, double* __restrict__ ltpart) {
    __shared__ double zs[kLtRows];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t r0 = (int64_t)blockIdx.x * kLtRows;
    for (int t = threadIdx.x; t < kLtRows; t += kB) zs[t] = (r0 + t < m) ? z[r0 + t] : 0.0;
    __syncthreads();
    const int64_t last = (int64_t)m - 1;
    for (int c = wave + 4 * blockIdx.y; c < K; c += 4 * gridDim.y) {
        const T* Lc = L32 + (int64_t)c * ld;
        double a[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int u = 0; u < kLtRows / 64; ++u) {
            const int64_t j = r0 + lane + 64 * u;
            a[u & 3] += (double)Lc[j < m ? j : last] * zs[lane + 64 * u];
        }
        const double s = wave_sum((a[0] + a[1]) + (a[2] + a[3]));
        if (lane == 0) ltpart[(int64_t)c * gridDim.x + blockIdx.x] = s;
    }
}

// w_c = y1_c / S(pivot c) - sum_b ltpart[c][b]; a wave per column c
__global__ __launch_bounds__(256) void k_pca_w(int32_t K, int32_t nb, const int32_t* __restrict__ perm,
                                               const double* __restrict__ y1, const double* __restrict__ S,
                                               const double* __restrict__ ltpart, double* __restrict__ w) {
    const int32_t c = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (c >= K) return;
    double a0 = 0.0, a1 = 0.0;
    int32_t b = lane;
    for (; b + 64 < nb; b += 128) {
        a0 += ltpart[(int64_t)c * nb + b];
        a1 += ltpart[(int64_t)c * nb + b + 64];
    }
    if (b < nb) a0 += ltpart[(int64_t)c * nb + b];
    const double s = wave_sum(a0 + a1);
    if (lane == 0) w[c] = y1[c] / S[perm[c]] - s;
}

// z(pivot i) = sum_{c >= i} X[c][i] w_c   (L11^-T w): 64 pivots per workgroup
// on the lanes, one of the eight interleaved chains (c - i mod 8; the last,
// partial group of eight goes to chain 0) per wave.  K = 500: 28 us,
// 75 us with a pivot's chains in one thread.
__global__ __launch_bounds__(512) void k_pca_final(int32_t K, const int32_t* __restrict__ perm,
                                                   const double* __restrict__ X, const double* __restrict__ w,
                                                   double* __restrict__ z) {
    __shared__ double red[8][64];
    const int lane = threadIdx.x & 63, u = threadIdx.x >> 6;
    const int32_t i = blockIdx.x * 64 + lane, ic = min(i, K - 1);
    const int32_t end = ic + ((K - ic) & ~7);   // of the full groups
    double a = 0.0;
    for (int32_t c = ic + u; c < end; c += 64) {
        double x[8], v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int32_t q = min(c + 8 * t, K - 1);
            x[t] = X[(int64_t)q * K + ic];
            v[t] = w[q];
        }
#pragma unroll
        for (int t = 0; t < 8; ++t)
            if (c + 8 * t < end) a += x[t] * v[t];
    }
    if (u == 0)
        for (int32_t c = end; c < K; ++c) a += X[(int64_t)c * K + ic] * w[c];
    red[u][lane] = a;
    __syncthreads();
    if (u == 0 && i < K) {
        double r[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) r[t] = red[t][lane];
        z[perm[i]] = ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
    }
}

// ---- conjugate gradients with the scalars on the device ----
// s[kCgRR] = r.r, s[kCgPQ] = p.q, s[kCgRZ + 0/1] = r.z of alternate
// iterations, s[kCgState] = 0 running / 1 converged / 2 breakdown,
// s[kCgIters] = iterations started.  Every kernel of an iteration returns at
// once when the state is not 0, so iterations the host enqueued after the
// stop change nothing.  The block partition of the reductions is that of
// k_dot_partial (kDotPartials blocks, grid-stride), and products and sums are
// not contracted into FMAs, as in those kernels, so every value is the one
// the separate dot and axpy kernels form.
__device__ inline bool cg_stopped(const double* s) { return s[kCgState] != 0.0; }

__device__ inline void block_sum_to(double acc, double* __restrict__ dst) {
    __shared__ double red[256];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) *dst = red[0];
}

__global__ __launch_bounds__(256) void k_cg_dot_partial(const double* __restrict__ a, const double* __restrict__ b,
                                                        int64_t n, double* __restrict__ part,
                                                        const double* __restrict__ s) {
#pragma clang fp contract(off)
    if (cg_stopped(s)) return;
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        acc = acc + a[i] * b[i];
    block_sum_to(acc, part + blockIdx.x);
}

// s[slot] = sum of the partials; kind 1 (p.q): the iteration has started,
// and it breaks down unless p.q > 0 and the current r.z > 0; kind 2 (r.r):
// converged when sqrt(r.r) <= target
__global__ __launch_bounds__(256) void k_cg_final(const double* __restrict__ part, int np, double* __restrict__ s,
                                                  int slot, int kind, int rz_cur, double target) {
#pragma clang fp contract(off)
    if (cg_stopped(s)) return;
    double acc = 0.0;
    for (int i = threadIdx.x; i < np; i += 256) acc = acc + part[i];
    __shared__ double tot;
    block_sum_to(acc, &tot);
    __syncthreads();
    if (threadIdx.x != 0) return;
    const double v = tot;
    s[slot] = v;
    if (kind == 1) {
        s[kCgIters] += 1.0;
        if (!(v > 0) || !(s[rz_cur] > 0)) s[kCgState] = 2.0;
    } else if (kind == 2) {
        if (sqrt(v) <= target) s[kCgState] = 1.0;
    }
}

// alpha = r.z / p.q;  x += alpha p;  r -= alpha q;  partials of r.r
__global__ __launch_bounds__(256) void k_cg_update(int64_t n, const double* __restrict__ s, int rz_cur,
                                                   const double* __restrict__ p, const double* __restrict__ q,
                                                   double* __restrict__ x, double* __restrict__ r,
                                                   double* __restrict__ part) {
#pragma clang fp contract(off)
    if (cg_stopped(s)) return;
    const double alpha = s[rz_cur] / s[kCgPQ];
    const double nalpha = -alpha;
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        x[i] = x[i] + alpha * p[i];
        const double ri = r[i] + nalpha * q[i];
        r[i] = ri;
        acc = acc + ri * ri;
    }
    block_sum_to(acc, part + blockIdx.x);
}

// beta = r.z(new) / r.z(old);  p = z + beta p
__global__ void k_cg_xpby(int64_t n, const double* __restrict__ s, int rz_cur, int rz_next,
                          const double* __restrict__ z, double* __restrict__ p) {
#pragma clang fp contract(off)
    if (cg_stopped(s)) return;
    const double beta = s[rz_next] / s[rz_cur];
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = z[i] + beta * p[i];
}

__global__ void k_cg_init(double* __restrict__ s, double rr, double rz) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        s[kCgRR] = rr; s[kCgPQ] = 0.0; s[kCgRZ] = rz; s[kCgRZ + 1] = 0.0; s[kCgState] = 0.0; s[kCgIters] = 0.0;
    }
}

}  // namespace

void build_row_split(int32_t m, const std::vector<int64_t>& rowptr, const std::vector<int32_t>& colind,
                     std::vector<RowChunk>& chunks, std::vector<int32_t>& hrow, std::vector<int32_t>& hptr,
                     std::vector<int32_t>& mrow) {
    chunks.clear();
    hrow.clear();
    mrow.clear();
    hptr.assign(1, 0);
    int64_t heavy = 0;
    for (int32_t i = 0; i < m; ++i) {
        const int64_t len = rowptr[i + 1] - rowptr[i];
        if (len > kHeavyRow) heavy += len;
        else if (len > kLightRow) mrow.push_back(i);
    }
    if (heavy == 0) return;
    // partials numbered by row; the chunks listed by their middle column
    std::vector<RowChunk> all;
    int32_t slot = 0;
    for (int32_t i = 0; i < m; ++i) {
        const int64_t b = rowptr[i], e = rowptr[i + 1];
        if (e - b <= kHeavyRow) continue;
        hrow.push_back(i);
        for (int64_t p = b; p < e; p += kRowChunk) all.push_back({p, std::min(e, p + kRowChunk), slot++});
        hptr.push_back(slot);
    }
    std::stable_sort(all.begin(), all.end(), [&](const RowChunk& x, const RowChunk& y) {
        return colind[(x.b + x.e) / 2] < colind[(y.b + y.e) / 2];
    });
    // eight runs of columns with equal nonzeros, one per XCD, dealt out in turn
    std::vector<std::vector<RowChunk>> run(kXcds);
    int64_t seen = 0;
    for (const RowChunk& c : all) {
        run[std::min<int64_t>(kXcds - 1, seen * kXcds / heavy)].push_back(c);
        seen += c.e - c.b;
    }
    size_t most = 0;
    for (const auto& r : run) most = std::max(most, r.size());
    for (size_t k = 0; k < most; ++k)
        for (const auto& r : run) chunks.push_back(k < r.size() ? r[k] : RowChunk{0, 0, 0});
}

void launch_csr_split(const RowSplitDev& rs, const int64_t* rowptr, const int32_t* colind, const double* val,
                      const double* x, double* y, bool square, hipStream_t st) {
    if (rs.m <= 0) return;
    if (rs.nmed) {
        const int nbm = (rs.nmed + 3) / 4;
        if (square) help::launch_kernel(k_csr_medium<true>, nbm, kB, 0, st, rs.nmed, rs.mrow, rowptr, colind, val, x, y);
        else help::launch_kernel(k_csr_medium<false>, nbm, kB, 0, st, rs.nmed, rs.mrow, rowptr, colind, val, x, y);
    }
    if (square) {
        help::launch_kernel(k_csr_light<true>, grid_for(rs.m), kB, 0, st, rs.m, rowptr, colind, val, x, y);
        if (rs.nchunk) help::launch_kernel(k_csr_chunk<true>, rs.nchunk, kB, 0, st, rs.chunks, colind, val, x, rs.part);
    } else {
        help::launch_kernel(k_csr_light<false>, grid_for(rs.m), kB, 0, st, rs.m, rowptr, colind, val, x, y);
        if (rs.nchunk) help::launch_kernel(k_csr_chunk<false>, rs.nchunk, kB, 0, st, rs.chunks, colind, val, x, rs.part);
    }
    if (rs.nheavy) help::launch_kernel(k_csr_heavy, (rs.nheavy + 3) / 4, kB, 0, st, rs.nheavy, rs.hrow, rs.hptr, rs.part, y);
}

void launch_csc_t_scaled(int32_t n, const int64_t* colptr, const int32_t* rowind, const double* val,
                         const double* dinv, const double* x, double* t, hipStream_t st) {
    if (n > 0) help::launch_kernel(k_csc_ts, grid_for(n), kB, 0, st, n, colptr, rowind, val, dinv, x, t);
}

namespace {
int pc_blocks(const PcBuild& B, int most) { return (int)std::min<int64_t>(most, ((int64_t)B.rows.m + kB - 1) / kB); }
void pc_candidates(const PcBuild& B, hipStream_t st) {
    const int nbt = pc_blocks(B, kTopBlocks);
    help::launch_kernel(k_pc_top_part, nbt, kB, 0, st, B.rows.m, B.pos, B.S, B.state, B.top, B.arg);
    help::launch_kernel(k_pc_top_pick, 1, kB, 0, st, nbt, B.K, B.top, B.state);
}
void pc_scatter(const PcBuild& B, int one, int clear, hipStream_t st) {
    const int nb = (int)std::min<int64_t>(2048, std::max<int64_t>(1, ((int64_t)B.max_row_nnz + kB - 1) / kB));
    help::launch_kernel(k_pc_scatter, dim3(nb, one ? 1 : kPcBlk), kB, 0, st, B.state, one, B.rowptr, B.colind, B.val, B.dinv, B.sc, clear);
}
// top: the partials of the search are the candidates', else the last column's
void pc_pivot(const PcBuild& B, int one, bool top, hipStream_t st) {
    const int np = pc_blocks(B, top ? kTopBlocks : kColumnBlocks);
    help::launch_kernel(k_pc_pivot, 1, kB, 0, st, B.rows.m, B.K, one, np, B.arg, B.state, B.perm, B.pos, B.L, B.D, B.w);
}
template <bool kBlock>
void pc_column(const PcBuild& B, hipStream_t st) {
    help::launch_kernel(k_pc_column<kBlock>, pc_blocks(B, kColumnBlocks), kB, 0, st, B.rows.m, B.state, B.pos, B.g, B.acc, B.w, B.D, B.L, B.L32, B.ld32, B.S, B.arg, B.rowptr, B.colind, B.sc);
}
}  // namespace

void launch_pc_block(const PcBuild& B, hipStream_t st) {
    const int32_t m = B.rows.m;
    const RowSplitDev& rs = B.rows;
    pc_candidates(B, st);
    pc_scatter(B, 0, 0, st);
    if (rs.nchunk)
        help::launch_kernel(k_pc_csr_chunk, (rs.nchunk + 4 * kXcds - 1) / (4 * kXcds) * kXcds, kB, 0, st, rs.nchunk, rs.chunks, B.state, B.colind, B.val, B.sc, B.part);
    if (rs.nmed)
        help::launch_kernel(k_pc_csr_medium, (rs.nmed + 3) / 4, kB, 0, st, m, rs.nmed, rs.mrow, B.state, B.rowptr, B.colind, B.val, B.sc, B.g);
    help::launch_kernel(k_pc_csr_light, grid_for((int64_t)m * kPcBlk), kB, 0, st, m, B.state, B.rowptr, B.colind, B.val, B.sc, B.g);
    if (rs.nheavy)
        help::launch_kernel(k_pc_csr_heavy, rs.nheavy, kB, 0, st, m, rs.hrow, rs.hptr, B.state, B.part, B.g);
    pc_scatter(B, 0, 1, st);
    help::launch_kernel(k_pc_weights, grid_for((int64_t)B.K * kPcBlk), kB, 0, st, m, B.state, B.D, B.L, B.wb);
    help::launch_kernel(k_pc_block, grid_for(m), kB, 0, st, m, B.state, B.pos, B.wb, B.L, B.acc);
    for (int s = 0; s < kPcBlk; ++s) {
        pc_pivot(B, 0, s == 0, st);
        pc_column<true>(B, st);
    }
}

void launch_pc_pivots(const PcBuild& B, int32_t steps, bool candidates, hipStream_t st) {
    if (candidates) pc_candidates(B, st);
    for (int s = 0; s < steps; ++s) {
        pc_pivot(B, 1, s == 0 && candidates, st);
        pc_scatter(B, 1, 0, st);
        launch_csr_split(B.rows, B.rowptr, B.colind, B.val, B.sc, B.g, false, st);
        pc_column<false>(B, st);
    }
}

void launch_pc_l11(int32_t m, int32_t K, const int32_t* perm, const double* L, double* L11, double* X,
                   hipStream_t st) {
    if (K <= 0) return;
    help::launch_kernel(k_pc_l11_gather, grid_for((int64_t)K * K), kB, 0, st, m, K, perm, L, L11);
    help::launch_kernel(k_pc_l11_inv, (K + 3) / 4, kB, 0, st, K, L11, X);
}

void launch_vdiv(int64_t n, const double* a, const double* b, double* out, hipStream_t st) {
    if (n > 0) help::launch_kernel(k_vdiv, grid_for(n), kB, 0, st, n, a, b, out);
}

template <typename T>
void launch_pc_apply(int32_t m, int32_t K, int64_t ld, const int32_t* perm, const int32_t* pos, const T* L32,
                     const double* X, const double* S, const double* r, double* y1, double* ltpart, double* z,
                     hipStream_t st) {
    // K = 0: z = r / S
    if (K <= 0) {
        help::launch_kernel(k_pca_t2<T>, grid_for(m), kB, 0, st, m, ld, K, pos, L32, y1, S, r, z);
        return;
    }
    const int nb = (int)(((int64_t)m + kLtRows - 1) / kLtRows);
    help::launch_kernel(k_pca_y1, (K + 3) / 4, kB, 0, st, K, perm, X, r, y1);
    help::launch_kernel(k_pca_t2<T>, grid_for(m), kB, 0, st, m, ld, K, pos, L32, y1, S, r, z);
    const int share = std::max(1, std::min((K + 3) / 4, kLtGroups / nb));
    help::launch_kernel(k_pca_lt<T>, dim3(nb, share), kB, 0, st, m, ld, K, L32, z, ltpart);
    double* w = y1 + kPcgMaxK;
    help::launch_kernel(k_pca_w, (K + 3) / 4, kB, 0, st, K, nb, perm, y1, S, ltpart, w);
    help::launch_kernel(k_pca_final, (K + 63) / 64, 512, 0, st, K, perm, X, w, z);
}

#define HELP_INST(T)                                                                                         \
    template void launch_pc_apply<T>(int32_t, int32_t, int64_t, const int32_t*, const int32_t*, const T*,     \
                                     const double*, const double*, const double*, double*, double*, double*,  \
                                     hipStream_t);
HELP_INST(float)
HELP_INST(double)
#undef HELP_INST

void launch_cg_init(double* s, double rr, double rz, hipStream_t st) {
    help::launch_kernel(k_cg_init, 1, 64, 0, st, s, rr, rz);
}

// one CG iteration after the matrix product q = M p and before the
// preconditioner: p.q (breakdown test), the x/r update with r.r
// (convergence test); then, after z = P^-1 r, r.z and the new direction
void launch_cg_step1(int64_t n, double* s, int rz_cur, double target, const double* p, const double* q, double* x,
                     double* r, double* part, hipStream_t st) {
    const int nb = (int)std::min<int64_t>(kDotPartials, std::max<int64_t>(1, (n + 255) / 256));
    help::launch_kernel(k_cg_dot_partial, nb, 256, 0, st, p, q, n, part, (const double*)s);
    help::launch_kernel(k_cg_final, 1, 256, 0, st, (const double*)part, nb, s, (int)kCgPQ, 1, rz_cur, target);
    help::launch_kernel(k_cg_update, nb, 256, 0, st, n, (const double*)s, rz_cur, p, q, x, r, part);
    help::launch_kernel(k_cg_final, 1, 256, 0, st, (const double*)part, nb, s, (int)kCgRR, 2, rz_cur, target);
}
void launch_cg_step2(int64_t n, double* s, int rz_cur, int rz_next, const double* r, const double* z, double* p,
                     double* part, hipStream_t st) {
    const int nb = (int)std::min<int64_t>(kDotPartials, std::max<int64_t>(1, (n + 255) / 256));
    help::launch_kernel(k_cg_dot_partial, nb, 256, 0, st, r, z, n, part, (const double*)s);
    help::launch_kernel(k_cg_final, 1, 256, 0, st, (const double*)part, nb, s, rz_next, 0, rz_cur, 0.0);
    help::launch_kernel(k_cg_xpby, (unsigned)((n + 255) / 256), 256, 0, st, n, (const double*)s, rz_cur, rz_next, z, p);
}

}  // namespace help
