// Host side of the matrix-free PCG mode (HELP UsePCG_CPU.cpp:91-178 and
// PCG.cpp:38-395): the partial-Cholesky preconditioner is built once per
// renew (d is the same for the three solves of an iteration; the reference
// rebuilds it inside every solve, PCG.cpp:301), then each solve runs FP64
// conjugate gradients on A D^-1 A^T (gamma = delta = 0, UsePCG_CPU.cpp:154-155)
// with the preconditioner applied from the FP32 copy of the factor.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>

#include "handle.h"
#include "pcg.h"

namespace {
// Scratch of the allocation-free preconditioner apply
// (help_gpu_pcg_apply_noalloc): the apply's y1/w vectors (2 * kPcgMaxK) and
// its per-block partial sums (K * ceil(m / kLtRows)).  Every GPU holds one
// copy until the process ends; calls that overlap on one GPU share it and
// race.  The kernels write every entry they read, so nothing needs clearing.
constexpr int64_t kNoAllocScratch = int64_t(1) << 20;   // doubles, 8 MiB
__device__ __align__(256) double scratch[kNoAllocScratch];
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_dev[kMaxDevices] = {};

// device address of `scratch` on the current device, looked up once per
// device (the host-side name of the array is not a device address)
double* scratch_ptr() {
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) throw help::HipError("device index out of range", HELP_ERR_HIP);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void* p = nullptr;
        HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_dev[dev] = (double*)p;
    }
    return g_scratch_dev[dev];
}
}  // namespace

namespace help {

struct PcgState {
    int32_t K = 0;
    int64_t ld32 = 0;                // column stride of the FP32 factor: whole 128-byte lines
    DBuf<double> cg, part;           // CG scalars (kCgSlots) and reduction partials
    double* hpin = nullptr;          // pinned: the scalars of the last two iterations
    hipEvent_t ev[2] = {nullptr, nullptr};
    ~PcgState() {
        for (auto& e : ev)
            if (e) (void)hipEventDestroy(e);
        if (hpin) (void)hipHostFree(hpin);
        if (hstate) (void)hipHostFree(hstate);
    }
    DBuf<double> L, D, S, w, g, sc, acc, wb, bpart, L11, X, y1, ltpart;
    DBuf<float> L32;
    DBuf<int32_t> perm, pos;
    DBuf<PcState> state;
    DBuf<PcBest> top, arg;
    PcState* hstate = nullptr;       // pinned: the state after the last two groups of the build
    double build_bytes = 0;          // algorithmic bytes of the last build
    bool blocks = false;             // the build may take its pivots in blocks
    DBuf<double> x, r, z, p, q, t;
    std::vector<int32_t> iota;
};

void pcg_free(PcgState* p) { delete p; }

void pcg_setup(help_gpu* h) {
    auto* P = new PcgState();
    h->pcg = P;
    hipStream_t st = h->st;
    const int32_t m = h->m, n = h->n;
    P->K = std::max(0, std::min<int32_t>(std::min(h->opts.pcg_k, kPcgMaxK), m));
    const int64_t K = std::max<int32_t>(P->K, 1);
    P->L.alloc((size_t)m * K);
    P->ld32 = ((int64_t)m + 31) / 32 * 32;
    if (h->opts.pcg_fp32_precond) P->L32.alloc((size_t)P->ld32 * K);
    P->D.alloc(K);
    P->w.alloc(K);
    P->S.alloc(m);
    P->L11.alloc((size_t)K * K);
    P->X.alloc((size_t)K * K);
    P->y1.alloc(2 * kPcgMaxK);
    P->ltpart.alloc((size_t)K * (((int64_t)m + kLtRows - 1) / kLtRows));
    P->perm.alloc(m);
    P->pos.alloc(m);
    P->x.alloc(m); P->r.alloc(m); P->z.alloc(m); P->p.alloc(m); P->q.alloc(m);
    P->t.alloc(n);
    P->cg.alloc(kCgSlots);
    P->part.alloc(kDotPartials);
    HIPCHK(hipHostMalloc((void**)&P->hpin, 2 * kCgSlots * sizeof(double), hipHostMallocDefault));
    for (auto& e : P->ev) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    P->iota.resize(m);
    for (int32_t i = 0; i < m; ++i) P->iota[i] = i;
    if (P->K > 0) {
        P->state.alloc(1);
        P->top.alloc(kTopBlocks * kPcBlk);
        P->arg.alloc(std::max(kTopBlocks, kColumnBlocks));
        HIPCHK(hipHostMalloc((void**)&P->hstate, 2 * sizeof(PcState), hipHostMallocDefault));
        // the build's blocks: the candidates' vectors over the columns, the
        // columns of A D^-1 A^T and their left-looking sums (8 (16 n + 80 m)
        // bytes).  Where they do not fit, or no block could pay (the first group
        // of K < 2 kPcFew leaves fewer than kPcFew pivots), the build goes pivot
        // by pivot.
        P->blocks = P->K >= 2 * kPcFew;
        if (P->blocks) {
            try {
                P->sc.alloc((size_t)n * kPcBlk);
                P->g.alloc((size_t)m * kPcBlk);
                P->acc.alloc((size_t)m * kPcBlk * 4);
                P->wb.alloc((size_t)K * kPcBlk);
                P->bpart.alloc(std::max<size_t>(1, (size_t)h->rows.nparts * kPcBlk));
            } catch (const HipError&) {
                (void)hipGetLastError();
                for (auto* b : {&P->sc, &P->g, &P->acc, &P->wb, &P->bpart}) b->free();
                P->blocks = false;
            }
        }
        if (!P->blocks) {
            P->sc.alloc(n);
            P->g.alloc(m);
        }
        HIPCHK(hipMemsetAsync(P->sc.p, 0, sizeof(double) * P->sc.n, st));
    }
    HIPCHK(hipStreamSynchronize(st));
}

// Greedy partial LDL^T of A D^-1 A^T with K pivots (PCG.cpp:38-103), the
// inverse of its unit-lower leading block (PCG.cpp:119-133), and the FP32
// copy of the factor for the apply.  d_dinv must hold 1/d.
void pcg_renew(help_gpu* h) {
    PcgState* P = h->pcg;
    hipStream_t st = h->st;
    const int32_t m = h->m;
    const int32_t K = P->K;
    // Schur diagonal: diag(A D^-1 A^T) (PCG.cpp:40-46)
    launch_csr_split(h->rows, h->d_rowptr.p, h->d_colind.p, h->d_csrval.p, h->d_dinv.p, P->S.p, true, st);
    HIPCHK(hipMemcpyAsync(P->perm.p, P->iota.data(), sizeof(int32_t) * m, hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(P->pos.p, P->iota.data(), sizeof(int32_t) * m, hipMemcpyHostToDevice, st));
    PcBuild B;
    B.rows = h->rows;
    B.rowptr = h->d_rowptr.p; B.colind = h->d_colind.p; B.val = h->d_csrval.p; B.dinv = h->d_dinv.p;
    B.K = K; B.max_row_nnz = h->max_row_nnz; B.ld32 = P->ld32;
    B.state = P->state.p; B.top = P->top.p; B.arg = P->arg.p;
    B.perm = P->perm.p; B.pos = P->pos.p;
    B.S = P->S.p; B.D = P->D.p; B.L = P->L.p; B.w = P->w.p; B.L32 = h->opts.pcg_fp32_precond ? P->L32.p : nullptr;
    B.sc = P->sc.p; B.part = P->bpart.p; B.g = P->g.p; B.acc = P->acc.p; B.wb = P->wb.p;
    if (K > 0) HIPCHK(hipMemsetAsync(P->state.p, 0, sizeof(PcState), st));
    // Groups of pivots: a block as long as the last group's leading candidates
    // were enough for one to pay, else pivot by pivot in groups of 4, 16 and then
    // 64 until they are again (a block that pays starts over at 4; the last group
    // needs no candidates).  A block that fails costs as much as a few pivots, so
    // small K starts without one.  The state comes back after every group; after
    // a block that paid, the next one is queued before its state is read.
    // m = 30,000, K = 16: 0.37 ms, 0.40 where no block pays; 0.30 and 2.65 in
    // blocks alone, 0.41 pivot by pivot.
    const double nnz = (double)h->nnz, N = h->n, M = m;
    int32_t k = 0, steps = P->blocks ? kPcFew : K;
    bool block = P->blocks && K > 2 * kPcBlk, paid = false, single = false;   // single: the last group went pivot by pivot
    int64_t launched = 0, read = 0;
    bool form[2] = {false, false};   // of the groups in flight: block?
    P->build_bytes = 12.0 * nnz + 8.0 * (N + M);   // the Schur diagonal
    while (k < K) {
        const bool blk = block && P->blocks && K - k >= kPcFew;
        if (launched == read || (launched == read + 1 && paid && form[read & 1] && K - k >= kPcBlk + kPcFew)) {
            if (blk) {
                launch_pc_block(B, st);
            } else {
                launch_pc_pivots(B, std::min(steps, K - k), steps < K - k || !single, st);
                steps = std::min(4 * steps, 4 * kPcBlk);
            }
            form[launched & 1] = blk;
            HIPCHK(hipMemcpyAsync(P->hstate + (launched & 1), P->state.p, sizeof(PcState), hipMemcpyDeviceToHost, st));
            HIPCHK(hipEventRecord(P->ev[launched & 1], st));
            ++launched;
            continue;
        }
        HIPCHK(hipEventSynchronize(P->ev[read & 1]));
        const PcState& s = P->hstate[read & 1];
        const bool was = form[read & 1];
        // A block reads A once, with kPcBlk vectors (8 (n + m) each), the
        // finished columns once and the candidates' sums (32 m each), and per
        // pivot its sums and the block's own columns; pivot by pivot, each reads
        // A with one vector and the columns before it.  Either way a pivot takes
        // the Schur diagonal and a column in FP64 and FP32.
        const double k0 = was ? s.k0 : k, got = s.k - k0, own = 4.0 * got * (got - 1);   // own columns: 8 m got (got - 1) / 2
        P->build_bytes += was ? 12.0 * nnz + kPcBlk * (8.0 * (N + M) + 32.0 * M) + 8.0 * M * k0 + got * 32.0 * M
                              : got * (12.0 * nnz + 8.0 * (N + M) + 8.0 * M * k0);
        P->build_bytes += M * (own + 36.0 * got);
        k = s.k;
        block = s.taken >= kPcFew;
        paid = was && block;
        single = !was;
        if (paid) steps = kPcFew;
        ++read;
    }
    launch_pc_l11(m, K, P->perm.p, P->L.p, P->L11.p, P->X.p, st);
    HIPCHK(hipGetLastError());
}

double pcg_build_bytes(const help_gpu* h) { return h->pcg ? h->pcg->build_bytes : 0.0; }

// per iteration: A^T p scaled (12 nnz + 8 m + 16 n), A t (12 nnz + 8 n + 8 m),
// the preconditioner (two passes over the m x K factor: 8 m K in FP32,
// 16 m K in FP64) and about ten m-vector streams
double pcg_iteration_bytes(const help_gpu* h) {
    const double nnz = (double)h->nnz, m = h->m, n = h->n, K = h->pcg ? h->pcg->K : 0;
    const double w = h->opts.pcg_fp32_precond ? 4.0 : 8.0;
    return 24.0 * nnz + 24.0 * n + 16.0 * m + 2.0 * w * m * K + 80.0 * m;
}

static double dot(help_gpu* h, const double* a, const double* b, int64_t n) {
    launch_dot(a, b, n, h->d_part.p, h->d_scal.p, h->st);
    double v = 0;
    HIPCHK(hipMemcpyAsync(&v, h->d_scal.p, sizeof(double), hipMemcpyDeviceToHost, h->st));
    HIPCHK(hipStreamSynchronize(h->st));
    return v;
}

// Conjugate gradients (PCG.cpp:296-395) on A D^-1 A^T x = rhs from x0 (or
// zero), all vectors on the device in the original row order.  Stops at
// ||r|| <= pcg_tol ||r0|| or pcg_max_iter iterations; x2 <- x.  Returns the
// iteration count; rel is the final ||r|| / ||r0||.
//
// The scalars of the iteration (p.q, r.r, r.z, alpha, beta) stay on the
// device (launch_cg_step1/2): no host round trip inside an iteration.  The
// host copies the state of every iteration to pinned memory and reads it one
// iteration later, while the next one is already queued, and stops queueing
// once it sees convergence or breakdown; the one extra iteration in flight
// then changes nothing (its kernels see the stopped state and return).
int pcg_solve(help_gpu* h, const double* rhs, const double* x0, double* x2, double& rel) {
    PcgState* P = h->pcg;
    hipStream_t st = h->st;
    const int32_t m = h->m, n = h->n;
    double *x = P->x.p, *r = P->r.p, *z = P->z.p, *p = P->p.p, *q = P->q.p, *t = P->t.p;
    auto matvec = [&](const double* v, double* out) {   // out = A D^-1 A^T v
        launch_csc_t_scaled(n, h->d_colptr.p, h->d_rowind.p, h->d_val.p, h->d_dinv.p, v, t, st);
        launch_csr_split(h->rows, h->d_rowptr.p, h->d_colind.p, h->d_csrval.p, t, out, false, st);
    };
    auto precond = [&](const double* v, double* out) { pcg_precond(h, v, out); };
    const double bb = dot(h, rhs, rhs, m);
    if (x0) {
        HIPCHK(hipMemcpyAsync(x, x0, sizeof(double) * m, hipMemcpyDeviceToDevice, st));
        matvec(x, q);
        launch_sub(m, rhs, q, r, st);
    } else {
        HIPCHK(hipMemsetAsync(x, 0, sizeof(double) * m, st));
        HIPCHK(hipMemcpyAsync(r, rhs, sizeof(double) * m, hipMemcpyDeviceToDevice, st));
    }
    double rr = dot(h, r, r, m);
    if (x0 && !(rr <= bb)) {   // a guess worse than zero (or not finite): start from zero
        HIPCHK(hipMemsetAsync(x, 0, sizeof(double) * m, st));
        HIPCHK(hipMemcpyAsync(r, rhs, sizeof(double) * m, hipMemcpyDeviceToDevice, st));
        rr = bb;
    }
    // the reference's stop is relative to ||r0|| (PCG.cpp:328); with a
    // warm start the relative target is taken against ||rhs|| so that a
    // good guess cannot loosen it
    const double r0 = std::sqrt(x0 ? std::max(bb, 0.0) : rr);
    const double target = h->opts.pcg_tol * r0;
    int it = 0;
    if (r0 == 0.0) {
        rel = 0;
    } else if (!(std::sqrt(rr) > target) || h->opts.pcg_max_iter <= 0) {
        rel = std::sqrt(rr) / r0;
    } else {
        precond(r, z);
        HIPCHK(hipMemcpyAsync(p, z, sizeof(double) * m, hipMemcpyDeviceToDevice, st));
        const double rz = dot(h, r, z, m);
        double* sc = P->cg.p;
        launch_cg_init(sc, rr, rz, st);
        const int maxit = h->opts.pcg_max_iter;
        int queued = 0;
        for (; queued < maxit; ++queued) {
            const int cur = kCgRZ + (queued & 1), next = kCgRZ + ((queued + 1) & 1);
            matvec(p, q);
            launch_cg_step1(m, sc, cur, target, p, q, x, r, P->part.p, st);
            precond(r, z);
            launch_cg_step2(m, sc, cur, next, r, z, p, P->part.p, st);
            double* hp = P->hpin + kCgSlots * (queued & 1);
            HIPCHK(hipMemcpyAsync(hp, sc, sizeof(double) * kCgSlots, hipMemcpyDeviceToHost, st));
            HIPCHK(hipEventRecord(P->ev[queued & 1], st));
            if (queued >= 1) {   // the state after the previous iteration
                HIPCHK(hipEventSynchronize(P->ev[(queued - 1) & 1]));
                if (P->hpin[kCgSlots * ((queued - 1) & 1) + kCgState] != 0.0) { ++queued; break; }
            }
        }
        HIPCHK(hipStreamSynchronize(st));
        const double* fin = P->hpin + kCgSlots * ((queued - 1) & 1);
        it = (int)fin[kCgIters];
        rel = std::sqrt(fin[kCgRR]) / r0;
    }
    HIPCHK(hipMemcpyAsync(x2, x, sizeof(double) * m, hipMemcpyDeviceToDevice, st));
    HIPCHK(hipGetLastError());
    return it;
}

// z = M^-1 v with the preconditioner of the last renew (device vectors,
// original row order), as pcg_solve applies it
void pcg_precond(help_gpu* h, const double* v, double* out) {
    PcgState* P = h->pcg;
    if (h->opts.pcg_fp32_precond)
        launch_pc_apply<float>(h->m, P->K, P->ld32, P->perm.p, P->pos.p, P->L32.p, P->X.p, P->S.p, v, P->y1.p,
                               P->ltpart.p, out, h->st);
    else
        launch_pc_apply<double>(h->m, P->K, h->m, P->perm.p, P->pos.p, P->L.p, P->X.p, P->S.p, v, P->y1.p,
                                P->ltpart.p, out, h->st);
}

// pcg_precond with its scratch in the file-scope `scratch` array: no
// allocation, device vectors only
void pcg_precond_noalloc(help_gpu* h, const double* v, double* out) {
    PcgState* P = h->pcg;
    const int64_t nb = ((int64_t)h->m + kLtRows - 1) / kLtRows;
    const int64_t need = 2 * (int64_t)kPcgMaxK + (int64_t)std::max(P->K, 1) * nb;
    if (need > kNoAllocScratch)
        throw std::runtime_error("pcg_apply_noalloc: needs " + std::to_string(need) +
                                 " scratch doubles (2 * 1024 + K * ceil(m / 2048)), above the maximum " +
                                 std::to_string(kNoAllocScratch));
    double* s = scratch_ptr();
    if (h->opts.pcg_fp32_precond)
        launch_pc_apply<float>(h->m, P->K, P->ld32, P->perm.p, P->pos.p, P->L32.p, P->X.p, P->S.p, v, s,
                               s + 2 * kPcgMaxK, out, h->st);
    else
        launch_pc_apply<double>(h->m, P->K, h->m, P->perm.p, P->pos.p, P->L.p, P->X.p, P->S.p, v, s,
                                s + 2 * kPcgMaxK, out, h->st);
}

void pcg_download(help_gpu* h, int32_t* K, int32_t* perm, double* D, double* S, double* L) {
    PcgState* P = h->pcg;
    hipStream_t st = h->st;
    const int32_t m = h->m;
    if (K) *K = P->K;
    if (perm) HIPCHK(hipMemcpyAsync(perm, P->perm.p, sizeof(int32_t) * m, hipMemcpyDeviceToHost, st));
    if (D && P->K) HIPCHK(hipMemcpyAsync(D, P->D.p, sizeof(double) * P->K, hipMemcpyDeviceToHost, st));
    if (S) HIPCHK(hipMemcpyAsync(S, P->S.p, sizeof(double) * m, hipMemcpyDeviceToHost, st));
    if (L && P->K) HIPCHK(hipMemcpyAsync(L, P->L.p, sizeof(double) * (size_t)m * P->K, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
}

}  // namespace help
