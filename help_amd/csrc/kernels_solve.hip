// Supernodal triangular solves L y = b and L^T x = y, level by level.
//
// Forward (leaves to root): each supernode gathers its children's update
// vectors (the multifrontal analogue of extend-add, children in fixed
// order), solves with its diagonal block L11 and forms its own update vector
// W_s = L21 y_s + (children's rows beyond s).  Backward (root to leaves):
// each supernode subtracts L21^T x(rows) and solves with L11^T; the rows are
// ancestors, already final.  Within L11 the solve walks 64-column blocks and
// applies the stored inverse of each diagonal block as a parallel product,
// so a block costs a few barriers instead of 64 dependent steps.  Vectors
// are FP64 whatever the factor type.  Big supernodes hand the L21 products
// to separate many-workgroup kernels.
//
// The solves are bound by load latency, not bandwidth: a level is one
// dependent chain, so whatever does not depend on the level before is on its
// way before the gather (a task carries its supernode's sizes and offsets,
// the first values of the factor go to registers), every inner loop keeps
// several independent loads in flight, and levels of few blocks take more
// waves per block.  An update vector is stored by its parent's rows: the
// entries that land on row r of supernode s, in child order, are
// W[gptr[rowoff[s] + r] .. gptr[rowoff[s] + r + 1]), so a row adds up its
// children's entries without walking the children (their sizes, their maps
// and a barrier for each).  Supernodes with at most 64 rows (the large
// majority, near the leaves) take one wave each, with the rows on the lanes
// and no workgroup barrier.  The order of every sum is fixed, and the same
// for every number of waves.
#include <type_traits>

#include "device.h"

namespace help {

namespace {

constexpr int kMaxLdsCols = kMaxSnCols;   // x segment of a supernode held in LDS
constexpr int kMaxGemvRows = 4096;        // gathered x(rows) held in LDS by k_bwd_gemv
constexpr int kLdT = 65;                  // leading dimension of a 64x64 block in LDS

// orders this wave's LDS accesses before and after (lanes exchange data
// through LDS without a workgroup barrier)
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline double wave_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// sum_{k<cnt} a[k*stride] * v[k] with two accumulators (even and odd k),
// eight loads in flight, the tail's too
template <typename T>
__device__ inline double dot_strided(const T* __restrict__ a, int64_t stride, const double* v, int32_t cnt) {
    double a0 = 0.0, a1 = 0.0;
    for (int32_t k0 = 0; k0 < cnt; k0 += 8) {
        T av[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) av[u] = a[(int64_t)min(k0 + u, cnt - 1) * stride];
#pragma unroll
        for (int u = 0; u < 8; u += 2) {
            if (k0 + u < cnt) a0 += (double)av[u] * v[k0 + u];
            if (k0 + u + 1 < cnt) a1 += (double)av[u + 1] * v[k0 + u + 1];
        }
    }
    return a0 + a1;
}

// dst[i] = src[idx[i]] for i < cnt, kQ per thread in flight (the index
// loads first, then the value loads)
template <int kQ>
__device__ inline void gather_idx(double* dst, const double* __restrict__ src, const int32_t* __restrict__ idx,
                                  int32_t cnt, int tid, int nt) {
    for (int32_t i0 = tid; i0 < cnt; i0 += kQ * nt) {
        int32_t ii[kQ];
        double v[kQ];
#pragma unroll
        for (int q = 0; q < kQ; ++q) ii[q] = idx[min(i0 + q * nt, cnt - 1)];
#pragma unroll
        for (int q = 0; q < kQ; ++q) v[q] = src[ii[q]];
#pragma unroll
        for (int q = 0; q < kQ; ++q)
            if (i0 + q * nt < cnt) dst[i0 + q * nt] = v[q];
    }
}

// a -+ the children's entries W[g0..g1) of one row, in child order: a row of
// the supernode's own columns (own) subtracts them, an update row adds them
__device__ __forceinline__ double gather_row(const double* W, int64_t g0, int64_t g1, double a, bool own) {
    for (; g0 < g1; g0 += 4) {
        double v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = W[min(g0 + q, g1 - 1)];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (g0 + q < g1) a += own ? -v[q] : v[q];
    }
    return a;
}

// ------------------------------------------------------------- tiny (c <= 64)
// The forward solve reads the right-hand side b and writes y; the backward
// solve reads y and writes x (x may be b's storage).  Keeping input and
// output apart lets the blocks of one wide supernode run in parallel
// without reading entries another block is writing.
template <typename T, int G>
__device__ __forceinline__ void fwd_tiny(const SolveTask& tk, const SolveMaps& mp, const T* __restrict__ L,
                         const T* __restrict__ Dinv, const double* __restrict__ b, double* __restrict__ y,
                         double* W, double* xw) {
    const int lane = threadIdx.x & (G - 1);   // G lanes per supernode (c <= G)
    const int32_t f = tk.f, n = tk.n, c = tk.c;
    const T* Lp = L + tk.loff;
    const bool own = lane < n, live = lane < c;
    const int64_t* gp = mp.gptr + tk.rowoff + min(lane, c - 1);
    const int64_t g0 = gp[0], g1 = gp[1];
    int64_t ws = 0;
    if (live && !own) ws = mp.wslot[tk.reloff + lane - n];
    const double v0 = own ? b[f + lane] : 0.0;
    const double gv = gather_row(W, g0, g1, v0, own);
    xw[lane] = gv;
    wave_sync();
    // one diagonal block: x1 = Dinv x1
    const T* Db = Dinv + tk.dinvoff;
    const double v = own ? dot_strided<T>(Db + lane, n, xw, n) : 0.0;
    wave_sync();
    if (own) xw[lane] = v;
    wave_sync();
    if (own) {
        y[f + lane] = v;
    } else if (live) {
        const double a = dot_strided<T>(Lp + lane, c, xw, n);
        W[ws] = gv + a;
    }
}

template <typename T, int G>
__device__ __forceinline__ void bwd_tiny(const SolveTask& tk, const SolveMaps& mp, const T* __restrict__ L,
                         const T* __restrict__ Dinv, const double* __restrict__ y, double* __restrict__ x,
                         double* xw) {
    const int lane = threadIdx.x & (G - 1);   // G lanes per supernode (c <= G)
    const int32_t f = tk.f, n = tk.n, c = tk.c;
    const T* Lp = L + tk.loff;
    const int32_t* rows = mp.rowidx + tk.rowoff;
    xw[lane] = (lane >= n && lane < c) ? x[rows[lane]] : 0.0;
    wave_sync();
    double v = 0.0;
    if (lane < n) {
        const T* col = Lp + (int64_t)lane * c;
        v = y[f + lane] - dot_strided<T>(col + n, 1, xw + n, c - n);
    }
    wave_sync();
    if (lane < n) xw[lane] = v;
    wave_sync();
    if (lane < n) {
        const T* Db = Dinv + tk.dinvoff;
        x[f + lane] = dot_strided<T>(Db + (int64_t)lane * n, 1, xw, n);
    }
}

// ------------------------------------------------- one workgroup per supernode
// x1 = Dinv x1 for a 64-column block: thread (r, part) of the first four
// waves sums the columns k = part (mod 4), u = 0..15 -> k = part + 4 u (a
// full block: even and odd u apart), the parts combine in a fixed order.
// val(u) is the inverse's entry (r, part + 4 u).
template <typename F>
__device__ __forceinline__ void apply_dinv(F val, int32_t nb, double* xs, double (*red)[64]) {
    const int r = threadIdx.x & 63, part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (part < 4) {
        double a0 = 0.0, a1 = 0.0;
        if (nb == 64) {
#pragma unroll
            for (int u = 0; u < 16; u += 2) {
                a0 += val(u) * xs[part + 4 * u];
                a1 += val(u + 1) * xs[part + 4 * u + 4];
            }
        } else if (r < nb) {
#pragma unroll
            for (int u = 0; u < 16; ++u)
                if (part + 4 * u < nb) a0 += val(u) * xs[part + 4 * u];
        }
        red[part][r] = a0 + a1;
    }
    __syncthreads();
    if (part == 0 && r < nb) xs[r] = (red[0][r] + red[1][r]) + (red[2][r] + red[3][r]);
    __syncthreads();
}

// Forward for a supernode that is not wide: gather the children's update
// vectors, walk the 64-column blocks with the diagonal-block inverses and
// (big == 0) apply L21 here; big supernodes leave the update rows to
// k_fwd_gemv.
template <typename T, int NT>
__device__ __forceinline__ void fwd_sn(const SolveTask& tk, const SolveMaps& mp, const T* __restrict__ L,
                       const T* __restrict__ Dinv, const double* __restrict__ b, double* __restrict__ y,
                       double* W, double* xs, double (*red)[64]) {
    const int32_t f = tk.f, n = tk.n, c = tk.c;
    const T* Lp = L + tk.loff;
    const int64_t* gp = mp.gptr + tk.rowoff;
    const int64_t* wp = mp.wslot + tk.reloff;
    const int tid = threadIdx.x, r = tid & 63, part = __builtin_amdgcn_readfirstlane(tid >> 6);
    T dv[16];
    auto load_dinv = [&](int32_t jb) {
        const int32_t nb = min(64, n - jb);
        const T* Db = Dinv + tk.dinvoff + (int64_t)jb * 64;
        if (part < 4)
#pragma unroll
            for (int u = 0; u < 16; ++u) dv[u] = Db[min(part + 4 * u, nb - 1) * nb + min(r, nb - 1)];
    };
    load_dinv(0);
    for (int32_t i = tid; i < n; i += NT) xs[i] = gather_row(W, gp[i], gp[i + 1], b[f + i], true);
    __syncthreads();
    const int32_t rend = tk.big ? n : c;
    for (int32_t jb = 0; jb < n; jb += 64) {
        const int32_t nb = min(64, n - jb);
        apply_dinv([&](int u) { return (double)dv[u]; }, nb, xs + jb, red);
        // rows below the block: a row per thread; an update row starts from
        // its children's entries
        const double* xv = xs + jb;
        auto rows = [&](auto count) {
            constexpr int kP = decltype(count)::value;
            for (int32_t i0 = jb + nb + tid; i0 < rend; i0 += kP * NT) {
                // kP rows' loads in flight: slots and entries of the children,
                // kL columns of L; four accumulators (k mod 4) on a full block,
                // else two (even and odd k)
                int32_t i[kP];
                bool own[kP];
                int64_t ws[kP] = {}, g0[kP] = {}, g1[kP] = {};
                uint32_t ib[kP];   // byte offset of the row in a column
#pragma unroll
                for (int p = 0; p < kP; ++p) {
                    i[p] = min(i0 + p * NT, rend - 1);
                    own[p] = i[p] < n;
                    ib[p] = (uint32_t)i[p] * (uint32_t)sizeof(T);
                    if (!own[p]) {
                        ws[p] = wp[i[p] - n];
                        if (jb == 0) {
                            g0[p] = gp[i[p]];
                            g1[p] = gp[i[p] + 1];
                        }
                    }
                }
                constexpr int kL = sizeof(T) == 4 ? 16 : 8;
                T lv[kP][kL];
                auto next = [&](int32_t k0) {
#pragma unroll
                    for (int u = 0; u < kL; ++u) {
                        const char* col = (const char*)(Lp + (int64_t)(jb + min(k0 + u, nb - 1)) * c);
#pragma unroll
                        for (int p = 0; p < kP; ++p) lv[p][u] = *(const T*)(col + ib[p]);
                    }
                };
                next(0);
                double base[kP] = {}, cv[kP][2];
#pragma unroll
                for (int p = 0; p < kP; ++p)
#pragma unroll
                    for (int q = 0; q < 2; ++q) cv[p][q] = W[jb == 0 ? max(min(g0[p] + q, g1[p] - 1), (int64_t)0) : ws[p]];
#pragma unroll
                for (int p = 0; p < kP; ++p) {
                    if (own[p]) continue;
                    if (jb == 0) {
#pragma unroll
                        for (int q = 0; q < 2; ++q)
                            if (g0[p] + q < g1[p]) base[p] += cv[p][q];
                        base[p] = gather_row(W, g0[p] + 2, g1[p], base[p], false);
                    } else {
                        base[p] = cv[p][0];
                    }
                }
                double a[kP];
                if (nb == 64) {
                    double a4[kP][4] = {};
#pragma unroll 1
                    for (int32_t k0 = 0; k0 < 64; k0 += kL) {
                        if (k0 > 0) next(k0);
#pragma unroll
                        for (int u = 0; u < kL; ++u) {
#pragma unroll
                            for (int p = 0; p < kP; ++p) a4[p][u & 3] += (double)lv[p][u] * xv[k0 + u];
                        }
                    }
#pragma unroll
                    for (int p = 0; p < kP; ++p) a[p] = (a4[p][0] + a4[p][1]) + (a4[p][2] + a4[p][3]);
                } else {
                    double a2[kP][2] = {};
#pragma unroll 1
                    for (int32_t k0 = 0; k0 < nb; k0 += kL) {
                        if (k0 > 0) next(k0);
#pragma unroll
                        for (int u = 0; u < kL; ++u)
                            if (k0 + u < nb) {
#pragma unroll
                                for (int p = 0; p < kP; ++p) a2[p][u & 1] += (double)lv[p][u] * xv[k0 + u];
                            }
                    }
#pragma unroll
                    for (int p = 0; p < kP; ++p) a[p] = a2[p][0] + a2[p][1];
                }
#pragma unroll
                for (int p = 0; p < kP; ++p) {
                    if (i0 + p * NT >= rend) continue;
                    if (own[p]) xs[i[p]] -= a[p];
                    else W[ws[p]] = base[p] + a[p];
                }
            }
        };
        if (rend - jb - nb > NT) rows(std::integral_constant<int, 2>{});
        else rows(std::integral_constant<int, 1>{});
        if (jb + 64 < n) load_dinv(jb + 64);
        __syncthreads();
    }
    for (int32_t t = tid; t < n; t += NT) y[f + t] = xs[t];
}

// Forward, wide supernode, kR rows (from row r0) of the 64-row block i with
// the explicit inverse:
// y[f+64i+r] = sum_{j<=i} sum_q X_ij[r][q] g[64j+q] (X_ii = Dinv_i), where g
// is the supernode's gathered right-hand side; every block gathers the g
// entries it needs itself.  Chain w = 0..3 takes q = 16w..16w+15 of every
// 64x64 block, its even and odd q in two accumulators (held apart, p = 0 and
// 1, with eight waves); the partial sums combine in a fixed order.
template <typename T, int NT, int kR>
__device__ __forceinline__ void fwd_xinv(const SolveTask& tk, int32_t r0, const SolveMaps& mp, const T* __restrict__ Dinv,
                         const T* __restrict__ X, const double* __restrict__ b, double* __restrict__ y,
                         const double* W, double* ys, double (*red)[64]) {
    constexpr int kSplit = NT >= 512 ? 2 : 1;   // threads per row and chain
    constexpr int kU = 16 / kSplit;             // entries of a block's row per thread
    constexpr int kB = kSplit == 1 ? 2 : sizeof(T) == 4 ? 4 : 3;   // blocks in flight
    const int32_t i = tk.blk, f = tk.f, n = tk.n;
    const int64_t* gp = mp.gptr + tk.rowoff;
    const int tid = threadIdx.x, rl = tid % kR, r = r0 + rl;
    const int cw = kR == 64 ? __builtin_amdgcn_readfirstlane(tid / kR) : tid / kR, w = cw / kSplit, p = cw % kSplit;
    const bool work = w < 4;
    const int32_t hi = min(n, 64 * (i + 1));
    const int32_t nb = min(64, n - 64 * i);
    if (r0 >= nb) return;   // (uniform)
    const T* Xi = X + tk.xoff + (int64_t)i * (i - 1) / 2 * 4096 + r;   // X_ij, j < i: 4096 entries each
    T xv[kB][kU];
    auto load = [&](int32_t j0) {
#pragma unroll
        for (int bb = 0; bb < kB; ++bb) {
            const T* Xb = Xi + (int64_t)min(j0 + bb, i - 1) * 4096;
#pragma unroll
            for (int u = 0; u < kU; ++u) xv[bb][u] = Xb[64 * (16 * w + kSplit * u + p)];
        }
    };
    T dv[16];
    if (work) {
        if (p == 0) {
            const T* Db = Dinv + tk.dinvoff + (int64_t)i * 4096;
            const int rr = min(r, nb - 1);
#pragma unroll
            for (int u = 0; u < 16; ++u) dv[u] = Db[min(16 * w + u, nb - 1) * nb + rr];
        }
        if (i > 0) load(0);
    }
    for (int32_t t = tid; t < hi; t += NT) ys[t] = gather_row(W, gp[t], gp[t + 1], b[f + t], true);
    __syncthreads();
    if (work) {
        double a0 = 0.0, a1 = 0.0;
        for (int32_t j0 = 0; j0 < i; j0 += kB) {
            if (j0 > 0) load(j0);
#pragma unroll
            for (int bb = 0; bb < kB; ++bb) {
                if (j0 + bb < i) {
                    const double* yj = ys + 64 * (j0 + bb) + 16 * w + p;
                    if (kSplit == 2) {
#pragma unroll
                        for (int u = 0; u < kU; ++u) a0 += (double)xv[bb][u] * yj[2 * u];
                    } else {
#pragma unroll
                        for (int u = 0; u < kU; u += 2) {
                            a0 += (double)xv[bb][u] * yj[u];
                            a1 += (double)xv[bb][u + 1] * yj[u + 1];
                        }
                    }
                }
            }
        }
        if (p == 0) {
            const double* yi = ys + 64 * i;
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const int q = 16 * w + u;
                const double yv = (r < nb && q < nb) ? yi[min(q, nb - 1)] : 0.0;
                a0 += (double)dv[u] * yv;
            }
        }
        if (kSplit == 2) red[4 * p + w][rl] = a0;
        else red[w][rl] = a0 + a1;
    }
    __syncthreads();
    if (tid < kR && 64 * i + r < n) {
        double s4[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) s4[q] = kSplit == 2 ? red[q][rl] + red[4 + q][rl] : red[q][rl];
        y[f + 64 * i + r] = (s4[0] + s4[1]) + (s4[2] + s4[3]);
    }
}

// One launch per level: blocks [0, ntb) solve a tiny supernode per wave
// (tasks[0, ntiny)), the next nrest blocks one supernode each
// (tasks[ntiny, ntiny + nrest)), the last blocks 64 / kS rows of a 64-row
// block of a wide supernode each.  Bound by the loads that one CU keeps in
// flight (some 30 GB/s: a block of a 950-column supernode is 0.5 MB), so
// levels of few blocks split them (kS = 4) and take eight waves (NT = 512);
// what lies where, below, at the launch.  A level of the staircase program
// with 250 narrow supernodes of some 2500 rows: 24 us; 42 us when each
// workgroup walked the children one after the other.
template <typename T, int NT, int kS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NT >= 512 ? 4 : 3))) void k_fwd_level(
    const SolveTask* __restrict__ tasks, int32_t ntiny, int32_t nrest, const SolveTask* __restrict__ xt, SolveMaps mp,
    const T* __restrict__ L, const T* __restrict__ Dinv, const T* __restrict__ X, const double* __restrict__ b,
    double* __restrict__ y, double* W, RhsStride rs) {
    constexpr int kWaves = NT / 64;
    __shared__ double xs[kMaxLdsCols];
    __shared__ double red[8][64];
    b += blockIdx.y * rs.v; y += blockIdx.y * rs.v; W += blockIdx.y * rs.w;
    const int32_t ntb = (ntiny + kWaves - 1) / kWaves;
    const int32_t bid = blockIdx.x;
    if (bid < ntb) {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int32_t idx = bid * kWaves + wave;
        if (idx < ntiny) fwd_tiny<T, 64>(tasks[idx], mp, L, Dinv, b, y, W, red[wave]);
    } else if (bid < ntb + nrest) {
        fwd_sn<T, NT>(tasks[ntiny + bid - ntb], mp, L, Dinv, b, y, W, xs, red);
    } else {
        const int32_t xb = bid - ntb - nrest;
        fwd_xinv<T, NT, 64 / kS>(xt[xb / kS], xb % kS * (64 / kS), mp, Dinv, X, b, y, W, xs, red);
    }
}

// levels made of tiny supernodes only (the leaves: many of them, and a
// kernel with a small register and LDS footprint)
template <typename T, int G>
__global__ __launch_bounds__(256) void k_fwd_tiny(const SolveTask* __restrict__ tasks, int32_t count, SolveMaps mp,
                                                  const T* __restrict__ L, const T* __restrict__ Dinv,
                                                  const double* __restrict__ b, double* __restrict__ y,
                                                  double* W, RhsStride rs) {
    __shared__ double xw[256 / G][G];
    b += blockIdx.y * rs.v; y += blockIdx.y * rs.v; W += blockIdx.y * rs.w;
    const int g = threadIdx.x / G;
    const int32_t idx = blockIdx.x * (256 / G) + g;
    if (idx < count) fwd_tiny<T, G>(tasks[idx], mp, L, Dinv, b, y, W, xw[g]);
}

// W(rows of L21) = the children's entries + L21 y_s for a 64-row block of a
// big supernode's L21.
// Every row sums its columns as four parts (columns j = part mod 4), each
// part as four interleaved chains a_q (columns part + 4q + 16t while the
// group start part + 16t has its 16 columns; the group tail's columns go to
// a_0 in order), a part as (a_0 + a_1) + (a_2 + a_3) and the row as
// (part 0 + part 1) + (part 2 + part 3).  A thread per row and chain, so a
// block keeps 16 chains' loads in flight; the first ones, and the children's
// entries, are asked for before y_s is staged.  kR: 64 rows per workgroup
// (a wave per chain), or 16 where that leaves CUs without work.
template <typename T, int kR>
__global__ __launch_bounds__(16 * kR) void k_fwd_gemv(const SolveTask* __restrict__ tasks, SolveMaps mp,
                                                   const T* __restrict__ L, const double* __restrict__ y,
                                                   double* W, RhsStride rs) {
    __shared__ double xs[kMaxLdsCols];
    __shared__ double red[16][kR];
    __shared__ double gs[kR];
    constexpr int kF = kR == 64 ? 8 : 32, kS = 64 / kR;
    y += blockIdx.y * rs.v; W += blockIdx.y * rs.w;
    const SolveTask tk = tasks[blockIdx.x / kS];
    const int32_t f = tk.f, n = tk.n, c = tk.c;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int32_t r = tid % kR, ch = kR == 64 ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid / kR;   // chain ch = part + 4 q
    const int32_t part = ch & 3, q = ch >> 2;
    const int32_t i0 = n + tk.blk * 64 + blockIdx.x % kS * kR, i = i0 + r, ic = min(i, c - 1);
    if (i0 >= c) return;   // (uniform)
    const T* lp = L + tk.loff + ic;
    const int32_t nfull = max(n - part + 3, 0) >> 4;   // groups with their 16 columns
    const T* l0 = lp + (int64_t)(part + 4 * q) * c;
    T lv[kF], tv[3];
    if (nfull > 0) {
#pragma unroll
        for (int u = 0; u < kF; ++u) lv[u] = l0[(int64_t)min(u, nfull - 1) * 16 * c];
    }
    const int32_t jt = part + 16 * nfull;   // the tail's columns jt, jt + 4, jt + 8
    if (q == 0) {
#pragma unroll
        for (int u = 0; u < 3; ++u) tv[u] = lp[(int64_t)min(jt + 4 * u, n - 1) * c];
    }
    for (int32_t t = tid; t < n; t += nt) xs[t] = y[f + t];
    if (ch == 15) {
        const int64_t* gp = mp.gptr + tk.rowoff + ic;
        gs[r] = gather_row(W, gp[0], gp[1], 0.0, false);
    }
    int64_t ws = 0;
    if (ch == 0) ws = mp.wslot[tk.reloff + ic - n];
    __syncthreads();
    double a = 0.0;
    const double* xq = xs + part + 4 * q;
    for (int32_t t0 = 0; t0 < nfull; t0 += kF) {
        if (t0 > 0) {
#pragma unroll
            for (int u = 0; u < kF; ++u) lv[u] = l0[(int64_t)min(t0 + u, nfull - 1) * 16 * c];
        }
#pragma unroll
        for (int u = 0; u < kF; ++u)
            if (t0 + u < nfull) a += (double)lv[u] * xq[16 * (t0 + u)];
    }
    if (q == 0) {
#pragma unroll
        for (int u = 0; u < 3; ++u)
            if (jt + 4 * u < n) a += (double)tv[u] * xs[jt + 4 * u];
    }
    red[ch][r] = a;
    __syncthreads();
    if (ch == 0 && i < c) {
        double pv[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) pv[p] = (red[p][r] + red[p + 4][r]) + (red[p + 8][r] + red[p + 12][r]);
        W[ws] = gs[r] + ((pv[0] + pv[1]) + (pv[2] + pv[3]));
    }
}

// t[f+j] = sum_{i>=n} L21(i,j) x[row_i] for 4 kC columns j of a big supernode:
// each wave kC columns at once, lanes over the rows, 16 loads in flight, the
// first of them before x is gathered.  kC: 4, or 1 where that leaves CUs
// without work.
template <typename T, int kC>
__global__ __launch_bounds__(256) void k_bwd_gemv(const SolveTask* __restrict__ tasks, SolveMaps mp,
                                                  const T* __restrict__ L, const double* __restrict__ x,
                                                  double* __restrict__ tout, RhsStride rs) {
    __shared__ double xr[kMaxGemvRows];
    constexpr int kI = 16 / kC, kS = 4 / kC;
    x += blockIdx.y * rs.v; tout += blockIdx.y * rs.v;
    const SolveTask tk = tasks[blockIdx.x / kS];
    const int32_t f = tk.f, n = tk.n, c = tk.c;
    const int32_t cu = c - n;
    const int32_t* rows = mp.rowidx + tk.rowoff;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool lds = cu <= kMaxGemvRows;
    const int32_t j0 = tk.blk * 16 + (blockIdx.x % kS * 4 + wave) * kC;
    const int32_t nq = min(kC, n - j0);   // (<= 0: no columns for this wave)
    // columns past the supernode's last repeat its last one (loads stay
    // unconditional); their sums are not stored
    const T* col[kC];
#pragma unroll
    for (int q = 0; q < kC; ++q) col[q] = L + tk.loff + (int64_t)min(j0 + q, n - 1) * c + n;
    T lv[kI][kC];
    auto load = [&](int32_t i0) {
#pragma unroll
        for (int e = 0; e < kI; ++e)
#pragma unroll
            for (int q = 0; q < kC; ++q) lv[e][q] = col[q][(uint32_t)min(i0 + 64 * e, cu - 1)];
    };
    if (cu > 0) load(lane);   // (a wide root has no rows below)
    if (lds)
        gather_idx<8>(xr, x, rows + n, cu, tid, 256);
    __syncthreads();
    if (nq <= 0) return;
    double acc[kC] = {};
    for (int32_t i0 = lane; i0 < cu; i0 += 64 * kI) {
        if (i0 != lane) load(i0);
#pragma unroll
        for (int e = 0; e < kI; ++e) {
            const int32_t i = i0 + 64 * e;
            if (i < cu) {
                const double xv = lds ? xr[i] : x[rows[n + i]];
#pragma unroll
                for (int q = 0; q < kC; ++q) acc[q] += (double)lv[e][q] * xv;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < kC; ++q) {
        const double v = wave_sum(acc[q]);
        if (lane == q && q < nq) tout[f + j0 + q] = v;
    }
}

// Backward for a supernode that is not wide: x_s = L11^-T (y_s - L21^T x(rows));
// big supernodes take the L21 product t from k_bwd_gemv.  With eight waves the
// 64x64 blocks that the lanes would read with a stride go through LDS (bs,
// which shares its storage with xr; xq holds the gathered x(rows) beside it
// when there are at most 64).  Four waves read them directly: the levels that
// take four are full of narrow supernodes, and want the LDS for more of them
// (45 us for 5285 workgroups, 65 us through LDS).
template <typename T, int NT>
__device__ __forceinline__ void bwd_sn(const SolveTask& tk, const SolveMaps& mp, const T* __restrict__ L,
                       const T* __restrict__ Dinv, const double* __restrict__ y, const double* __restrict__ tin,
                       double* __restrict__ x, double* xs, int32_t pool, double* xq, double (*red)[64]) {
    constexpr int kWaves = NT / 64, kCw = 64 / kWaves;   // columns of a block per wave
    constexpr bool kStage = NT >= 512;
    const int32_t f = tk.f, n = tk.n, c = tk.c;
    const int32_t cu = c - n;
    const T* Lp = L + tk.loff;
    const int32_t* rows = mp.rowidx + tk.rowoff;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int32_t nblk = (n + 63) / 64;
    // beside the n entries of xs: the gathered x(rows), then a 64x64 block
    double* xr = xs + n;
    T* bs = (T*)xr;
    // the inverse of a block: along its columns into LDS, or the entries of
    // apply_dinv straight to registers
    constexpr int kDv = kStage ? kCw : 16;
    T dv[kDv];
    auto load_dinv = [&](int32_t bi) {
        const int32_t nb = min(64, n - 64 * bi);
        const T* Db = Dinv + tk.dinvoff + (int64_t)bi * 4096;
#pragma unroll
        for (int u = 0; u < kDv; ++u) {
            const int along = min(lane, nb - 1), other = min(wave + (kStage ? kWaves : 4) * u, nb - 1);
            dv[u] = kStage ? Db[other * nb + along] : Db[along * nb + other];
        }
    };
    load_dinv(nblk - 1);
    if (tk.big) {
        for (int32_t t = tid; t < n; t += NT) xs[t] = y[f + t] - tin[f + t];
    } else if (cu <= 64) {
        // few rows below the diagonal block: a thread per column, two
        // accumulators (even and odd rows)
        if constexpr (!kStage) {
            if (tid < cu) xq[tid] = x[rows[n + tid]];
            __syncthreads();
            for (int32_t j = tid; j < n; j += NT)
                xs[j] = y[f + j] - dot_strided<T>(Lp + (int64_t)j * c + n, 1, xq, cu);
        } else {
        T lv[kCw];
        for (int32_t j0 = 0; j0 < n; j0 += 64) {
#pragma unroll
            for (int u = 0; u < kCw; ++u)
                lv[u] = Lp[(int64_t)min(j0 + wave + kWaves * u, n - 1) * c + min(n + lane, c - 1)];
            if (j0 == 0 && tid < cu) xq[tid] = x[rows[n + tid]];
            double yv = 0.0;
            if (tid < min(64, n - j0)) yv = y[f + j0 + tid];
            __syncthreads();   // (bs is free)
#pragma unroll
            for (int u = 0; u < kCw; ++u) bs[(wave + kWaves * u) * kLdT + lane] = lv[u];
            __syncthreads();
            if (tid < min(64, n - j0)) {
                const T* col = bs + tid * kLdT;
                double a0 = 0.0, a1 = 0.0;
                int32_t k = 0;
#pragma unroll 4
                for (; k + 1 < cu; k += 2) {
                    a0 += (double)col[k] * xq[k];
                    a1 += (double)col[k + 1] * xq[k + 1];
                }
                if (k < cu) a0 += (double)col[k] * xq[k];
                xs[j0 + tid] = yv - (a0 + a1);
            }
        }
        }
    } else {
        const bool lds = c <= pool;
        if (lds) gather_idx<4>(xr, x, rows + n, cu, tid, NT);
        __syncthreads();
        // two columns and two groups of 256 rows per wave in flight; each
        // column has four accumulators over the groups' 64-row quarters (the
        // last, partial group's rows all go to the first) and one combine order
        for (int32_t j0 = 2 * wave; j0 < n; j0 += 2 * kWaves) {
            const T* col[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) col[q] = Lp + (int64_t)min(j0 + q, n - 1) * c + n;
            double a[2][4] = {};
            for (int32_t i = lane; i < cu; i += 512) {
                T lv[2][8];
                double xv[8];
#pragma unroll
                for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int q = 0; q < 2; ++q) lv[q][e] = col[q][(uint32_t)min(i + 64 * e, cu - 1)];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int32_t ie = min(i + 64 * e, cu - 1);
                    xv[e] = lds ? xr[ie] : x[rows[n + ie]];
                }
#pragma unroll
                for (int g = 0; g < 8; g += 4) {
                    if (i + 64 * g + 192 < cu) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
#pragma unroll
                            for (int q = 0; q < 2; ++q) a[q][e] += (double)lv[q][g + e] * xv[g + e];
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (i + 64 * (g + e) < cu) {
#pragma unroll
                                for (int q = 0; q < 2; ++q) a[q][0] += (double)lv[q][g + e] * xv[g + e];
                            }
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const double acc = wave_sum((a[q][0] + a[q][1]) + (a[q][2] + a[q][3]));
                if (lane == 0 && j0 + q < n) xs[j0 + q] = y[f + j0 + q] - acc;
            }
        }
    }
    __syncthreads();
    for (int32_t bi = nblk - 1; bi >= 0; --bi) {
        const int32_t jb = bi * 64;
        const int32_t nb = min(64, n - jb);
        const int32_t below = jb + nb;
        if constexpr (kStage) {
#pragma unroll
            for (int u = 0; u < kCw; ++u) bs[(wave + kWaves * u) * kLdT + lane] = dv[u];
            if (bi > 0) load_dinv(bi - 1);
        }
        if (below < n) {
            // xs[jb+q] -= sum_{below <= i < n} L(i, jb+q) xs[i]; a wave takes
            // kCw columns, lanes over the rows
            // (only the last block can be partial, and nothing lies below it)
            const int32_t q0 = wave * kCw;
            const T* base = Lp + (int64_t)(jb + q0) * c;
            double acc[kCw];
#pragma unroll
            for (int u = 0; u < kCw; ++u) acc[u] = 0.0;
#pragma unroll 2
            for (int32_t i = below + lane; i < n; i += 64) {
                const double xv = xs[i];
#pragma unroll
                for (int u = 0; u < kCw; ++u) acc[u] += (double)base[(int64_t)u * c + i] * xv;
            }
#pragma unroll
            for (int u = 0; u < kCw; ++u) {
                const double v = wave_sum(acc[u]);
                if (lane == u) xs[jb + q0 + u] -= v;
            }
        }
        __syncthreads();
        if constexpr (kStage) {
            const T* bt = bs + lane * kLdT + wave;
            apply_dinv([&](int u) { return (double)bt[4 * u]; }, nb, xs + jb, red);
        } else {
            apply_dinv([&](int u) { return (double)dv[u]; }, nb, xs + jb, red);
            if (bi > 0) load_dinv(bi - 1);
        }
    }
    for (int32_t t = tid; t < n; t += NT) x[f + t] = xs[t];
}

// Backward, wide supernode, kC columns (from column q0) of the 64-column block
// j with the explicit inverse:
// x[f+64j+q] = sum_{i>=j} sum_r X_ij[r][q] (y - t)[f+64i+r].  A wave takes
// kC / waves columns q, lanes over r; the sum over blocks and lanes has a
// fixed order.
template <typename T, int NT, int kC>
__device__ __forceinline__ void bwd_xinv(const SolveTask& tk, int32_t q0, const T* __restrict__ Dinv, const T* __restrict__ X,
                         const double* __restrict__ y, const double* __restrict__ tin, double* __restrict__ x,
                         double* ys) {
    constexpr int kWaves = NT / 64, kCw = kC / kWaves;
    constexpr int kB = NT < 512 ? 2 : 32 / kCw;   // blocks in flight
    const int32_t j = tk.blk, f = tk.f, n = tk.n;
    const int32_t nblk = (n + 63) / 64;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int32_t nb = min(64, n - 64 * j);
    if (q0 >= nb) return;   // (uniform)
    const int qw = q0 + kCw * w;
    const T* Xj = X + tk.xoff + (int64_t)j * 4096 + lane + 64 * qw;
    T xv[kB][kCw], dv[kCw];
    auto load = [&](int32_t i0) {
#pragma unroll
        for (int bb = 0; bb < kB; ++bb) {
            const int64_t i = min(i0 + bb, nblk - 1);
            const T* Xb = Xj + i * (i - 1) / 2 * 4096;
#pragma unroll
            for (int u = 0; u < kCw; ++u) xv[bb][u] = Xb[64 * u];
        }
    };
    {
        const T* Db = Dinv + tk.dinvoff + (int64_t)j * 4096;
#pragma unroll
        for (int u = 0; u < kCw; ++u) dv[u] = Db[min(qw + u, nb - 1) * nb + min(lane, nb - 1)];
    }
    if (j + 1 < nblk) load(j + 1);
    for (int32_t t = 64 * j + tid; t < n; t += NT) ys[t] = y[f + t] - tin[f + t];
    __syncthreads();
    double acc[kCw];
#pragma unroll
    for (int u = 0; u < kCw; ++u) acc[u] = 0.0;
    {
        const double yv = lane < nb ? ys[64 * j + min(lane, nb - 1)] : 0.0;
#pragma unroll
        for (int u = 0; u < kCw; ++u) acc[u] += (double)dv[u] * yv;
    }
    for (int32_t i0 = j + 1; i0 < nblk; i0 += kB) {
        if (i0 > j + 1) load(i0);
#pragma unroll
        for (int bb = 0; bb < kB; ++bb) {
            const int32_t i = i0 + bb;
            if (i < nblk) {
                const int32_t nbi = min(64, n - 64 * i);
                const double yv = lane < nbi ? ys[64 * i + min(lane, nbi - 1)] : 0.0;
#pragma unroll
                for (int u = 0; u < kCw; ++u) acc[u] += (double)xv[bb][u] * yv;
            }
        }
    }
#pragma unroll
    for (int u = 0; u < kCw; ++u) {
        const double v = wave_sum(acc[u]);
        const int32_t q = 64 * j + qw + u;
        if (lane == u && q < n) x[f + q] = v;
    }
}

// One launch per level, block kinds as in k_fwd_level (250 narrow supernodes
// of some 2500 rows: 17 us, 36 us when their x(rows) beyond 2048 were read
// again for every four columns).
template <typename T, int NT, int kS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_bwd_level(
    const SolveTask* __restrict__ tasks, int32_t ntiny, int32_t nrest, const SolveTask* __restrict__ xt, SolveMaps mp,
    const T* __restrict__ L, const T* __restrict__ Dinv, const T* __restrict__ X, const double* __restrict__ y,
    const double* __restrict__ tin, double* __restrict__ x, RhsStride rs) {
    constexpr int kWaves = NT / 64;
    // a supernode's columns, and its gathered rows or a 64x64 block
    constexpr int kPool = NT >= 512 ? kMaxLdsCols + 64 * kLdT * (int)sizeof(T) / 8 : 2 * kMaxLdsCols;
    __shared__ __attribute__((aligned(16))) double xs[kPool];
    __shared__ double red[8][64];
    __shared__ double xq[64];
    y += blockIdx.y * rs.v; tin += blockIdx.y * rs.v; x += blockIdx.y * rs.v;
    const int32_t ntb = (ntiny + kWaves - 1) / kWaves;
    const int32_t bid = blockIdx.x;
    if (bid < ntb) {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int32_t idx = bid * kWaves + wave;
        if (idx < ntiny) bwd_tiny<T, 64>(tasks[idx], mp, L, Dinv, y, x, red[wave]);
    } else if (bid < ntb + nrest) {
        bwd_sn<T, NT>(tasks[ntiny + bid - ntb], mp, L, Dinv, y, tin, x, xs, kPool, xq, red);
    } else {
        const int32_t xb = bid - ntb - nrest;
        bwd_xinv<T, NT, 64 / kS>(xt[xb / kS], xb % kS * (64 / kS), Dinv, X, y, tin, x, xs);
    }
}

template <typename T, int G>
__global__ __launch_bounds__(256) void k_bwd_tiny(const SolveTask* __restrict__ tasks, int32_t count, SolveMaps mp,
                                                  const T* __restrict__ L, const T* __restrict__ Dinv,
                                                  const double* __restrict__ y, double* __restrict__ x,
                                                  RhsStride rs) {
    __shared__ double xw[256 / G][G];
    y += blockIdx.y * rs.v; x += blockIdx.y * rs.v;
    const int g = threadIdx.x / G;
    const int32_t idx = blockIdx.x * (256 / G) + g;
    if (idx < count) bwd_tiny<T, G>(tasks[idx], mp, L, Dinv, y, x, xw[g]);
}

}  // namespace

// Where a launch leaves CUs without work.  Levels of at most kFewBlocks
// workgroups (two per CU, counting a wide supernode's blocks before the
// split) take eight waves per workgroup and split the blocks of wide
// supernodes four ways: 16 blocks of 950 columns in FP64 17.4 -> 10.8 us
// forward and 16.0 -> 7.2 backward, 106 blocks 19.5 -> 13.1 and 23.0 -> 10.9,
// 322 blocks 28.8 -> 22.0 and 30.9 -> 21.7; levels of more are small
// supernodes, and slower with eight waves (1894: 24 -> 46 us backward, 5285:
// 45 -> 51 us forward and 45 -> 96 us backward).  The L21
// products split only where they have fewer blocks still, as a split block
// reads the lines at its ends twice: forward, 16 rows instead of 64, 61
// blocks 17.8 -> 15.1 us but 90 blocks 18.5 -> 19.7 and 225 blocks
// 21.7 -> 31.5; backward, a column per wave instead of four, 216 blocks
// 20.6 -> 19.3 but 385 blocks 23.6 -> 25.9.
constexpr int32_t kFewBlocks = 512;
constexpr int32_t kFewFwd = 64;
constexpr int32_t kFewBwd = 256;

template <typename T>
void launch_fwd_level(const SolveTask* tasks, int32_t count, int32_t ntiny, const SolveTask* xt, int32_t nx,
                      SolveMaps mp, const T* L, const T* Dinv, const T* X, const double* b, double* y, double* W,
                      int nrhs, RhsStride rs, hipStream_t st, int tiny_lanes) {
    const int32_t nrest = count - ntiny;
    if (nrest == 0 && nx == 0) {
        if (ntiny > 0 && tiny_lanes == 32)
            help::launch_kernel(k_fwd_tiny<T, 32>, dim3((ntiny + 7) / 8, nrhs), 256, 0, st, tasks, ntiny, mp, L,
                                Dinv, b, y, W, rs);
        else if (ntiny > 0)
            help::launch_kernel(k_fwd_tiny<T, 64>, dim3((ntiny + 3) / 4, nrhs), 256, 0, st, tasks, ntiny, mp, L,
                                Dinv, b, y, W, rs);
        return;
    }
    const int64_t few = (ntiny + 7) / 8 + nrest;
    if (few * nrhs <= kFewBlocks && (int64_t)nx * nrhs <= kFewBlocks)
        help::launch_kernel(k_fwd_level<T, 512, 4>, dim3(few + 4 * nx, nrhs), 512, 0, st, tasks, ntiny, nrest, xt,
                            mp, L, Dinv, X, b, y, W, rs);
    else
        help::launch_kernel(k_fwd_level<T, 256, 1>, dim3((ntiny + 3) / 4 + nrest + nx, nrhs), 256, 0, st, tasks,
                            ntiny, nrest, xt, mp, L, Dinv, X, b, y, W, rs);
}
template <typename T>
void launch_bwd_level(const SolveTask* tasks, int32_t count, int32_t ntiny, const SolveTask* xt, int32_t nx,
                      SolveMaps mp, const T* L, const T* Dinv, const T* X, const double* y, const double* t,
                      double* x, int nrhs, RhsStride rs, hipStream_t st, int tiny_lanes) {
    const int32_t nrest = count - ntiny;
    if (nrest == 0 && nx == 0) {
        if (ntiny > 0 && tiny_lanes == 32)
            help::launch_kernel(k_bwd_tiny<T, 32>, dim3((ntiny + 7) / 8, nrhs), 256, 0, st, tasks, ntiny, mp, L,
                                Dinv, y, x, rs);
        else if (ntiny > 0)
            help::launch_kernel(k_bwd_tiny<T, 64>, dim3((ntiny + 3) / 4, nrhs), 256, 0, st, tasks, ntiny, mp, L,
                                Dinv, y, x, rs);
        return;
    }
    const int64_t few = (ntiny + 7) / 8 + nrest;
    if (few * nrhs <= kFewBlocks && (int64_t)nx * nrhs <= kFewBlocks)
        help::launch_kernel(k_bwd_level<T, 512, 4>, dim3(few + 4 * nx, nrhs), 512, 0, st, tasks, ntiny, nrest, xt,
                            mp, L, Dinv, X, y, t, x, rs);
    else
        help::launch_kernel(k_bwd_level<T, 256, 1>, dim3((ntiny + 3) / 4 + nrest + nx, nrhs), 256, 0, st, tasks,
                            ntiny, nrest, xt, mp, L, Dinv, X, y, t, x, rs);
}
template <typename T>
void launch_fwd_gemv(const SolveTask* tasks, int32_t count, SolveMaps mp, const T* L, const double* y, double* W,
                     int nrhs, RhsStride rs, hipStream_t st) {
    if (count <= 0) return;
    if ((int64_t)count * nrhs <= kFewFwd)
        help::launch_kernel(k_fwd_gemv<T, 16>, dim3(4 * count, nrhs), 256, 0, st, tasks, mp, L, y, W, rs);
    else
        help::launch_kernel(k_fwd_gemv<T, 64>, dim3(count, nrhs), 1024, 0, st, tasks, mp, L, y, W, rs);
}
template <typename T>
void launch_bwd_gemv(const SolveTask* tasks, int32_t count, SolveMaps mp, const T* L, const double* x, double* t,
                     int nrhs, RhsStride rs, hipStream_t st) {
    if (count <= 0) return;
    if ((int64_t)count * nrhs <= kFewBwd)
        help::launch_kernel(k_bwd_gemv<T, 1>, dim3(4 * count, nrhs), 256, 0, st, tasks, mp, L, x, t, rs);
    else
        help::launch_kernel(k_bwd_gemv<T, 4>, dim3(count, nrhs), 256, 0, st, tasks, mp, L, x, t, rs);
}

#define HELP_INST(T)                                                                                            \
    template void launch_fwd_level<T>(const SolveTask*, int32_t, int32_t, const SolveTask*, int32_t, SolveMaps, \
                                      const T*, const T*, const T*, const double*, double*, double*, int,       \
                                      RhsStride, hipStream_t, int);                                             \
    template void launch_bwd_level<T>(const SolveTask*, int32_t, int32_t, const SolveTask*, int32_t, SolveMaps, \
                                      const T*, const T*, const T*, const double*, const double*, double*, int, \
                                      RhsStride, hipStream_t, int);                                             \
    template void launch_fwd_gemv<T>(const SolveTask*, int32_t, SolveMaps, const T*, const double*, double*,    \
                                     int, RhsStride, hipStream_t);                                              \
    template void launch_bwd_gemv<T>(const SolveTask*, int32_t, SolveMaps, const T*, const double*, double*,    \
                                     int, RhsStride, hipStream_t);
HELP_INST(double)
HELP_INST(float)
#undef HELP_INST

}  // namespace help
