"""Workloads that time the backend through its public entry points.

Four families of linear programs, with the shapes of the benchmark's and the
tests' instances (help_amd/instances.py), generated here with numpy:

* random     A = [B | I], k N(0,1) nonzeros per column of B (small, launch-bound)
* mcf        multicommodity flow on a side x side grid (sparse factor, deep tree)
* staircase  periods of rows x 3 rows blocks, 5 nonzeros per column and a link
             into the next period (large dense fronts)
* zipf       A = [B | I], 6 nonzeros per column, Zipf(1.1) row popularity (PCG mode)

and what a user of the backend does with one:

* iteration  one interior-point iteration's linear algebra: renew with a new
             d, the two systems that share a call (solve2), the corrector's
             system (solve)
* solves     the three systems alone, on a factor that is already there
* build      PCG mode: the preconditioner of a new d, and one apply of it
* pcg        PCG mode: one system solved by conjugate gradients to 1e-10
* predict    the warm-start network's guess for one system
* train      the network's loss and weight gradient on one (d, r, dy) tuple

The sparsity of an instance is fixed by its sizes; the values of A (but the
grid's +-1), d and the right-hand sides come from the seed.  d is log-uniform
over +-`decades`, as it spreads along an interior-point run.
"""
import ctypes as C
import functools
import os

import numpy as np
import torch

import help_amd
from help_amd import LinearEquation
from help_amd import _lib as L
from help_amd.backend import HelpError, Instance
from help_amd.warmstart import Mpnn

NET = os.path.join(os.path.dirname(os.path.abspath(help_amd.__file__)), "data", "warmstart_net_mcf.npz")
BETA = 1e-5          # the factor's diagonal shift (the library's default)
HIDDEN = 64          # the network's width


# ----------------------------------------------------------------- instances
def _distinct(rng, count, k, draw):
    """count x k row numbers, distinct and ascending in each line"""
    rows = np.sort(draw(rng, (count, k)), axis=1)
    while True:
        bad = np.nonzero((rows[:, 1:] == rows[:, :-1]).any(axis=1))[0]
        if bad.size == 0:
            return rows
        rows[bad] = np.sort(draw(rng, (bad.size, k)), axis=1)


def _columns(m, counts, rows):
    colptr = np.zeros(len(counts) + 1, np.int64)
    np.cumsum(counts, out=colptr[1:])
    return m, len(counts), colptr, np.ascontiguousarray(rows, np.int32)


@functools.lru_cache(maxsize=4)
def _pattern(family, size, size2):
    """(m, n, colptr, rowind, +-1 values or None) of an instance"""
    rng = np.random.default_rng(7)
    if family == "random":            # size rows, size2 nonzeros per column, 2 size columns and the identity
        m, k = size, size2
        rows = _distinct(rng, 2 * m, k, lambda g, s: g.integers(0, m, s))
        return _columns(m, np.r_[np.full(2 * m, k), np.ones(m, int)], np.r_[rows.ravel(), np.arange(m)]) + (None,)
    if family == "staircase":         # size periods of size2 rows
        T, R, C, k = size, size2, 3 * size2, 5
        rows = _distinct(rng, T * C, k, lambda g, s: g.integers(0, R, s))
        period = np.repeat(np.arange(T), C)
        rows += R * period[:, None]
        link = R * (period + 1) + rng.integers(0, R, T * C)
        body = np.concatenate([np.c_[rows, link][: (T - 1) * C].ravel(), rows[(T - 1) * C:].ravel()])
        counts = np.r_[np.full((T - 1) * C, k + 1), np.full(C, k), np.ones(T * R, int)]
        return _columns(T * R, counts, np.r_[body, np.arange(T * R)]) + (None,)
    if family == "zipf":              # size rows, 3 size columns of 6 and the identity
        m = size
        cdf = np.cumsum(np.arange(1, m + 1, dtype=np.float64) ** -1.1)
        cdf /= cdf[-1]
        rows = _distinct(rng, 3 * m, 6, lambda g, s: np.minimum(np.searchsorted(cdf, g.random(s), side="right"), m - 1))
        return _columns(m, np.r_[np.full(3 * m, 6), np.ones(m, int)], np.r_[rows.ravel(), np.arange(m)]) + (None,)
    G, K = size, size2                # mcf: a G x G grid, K commodities; the last node's row is dropped
    node = np.arange(G * G)
    r, c = node // G, node % G
    arcs = []
    for dr, dc in ((0, 1), (1, 0), (0, -1), (-1, 0)):
        ok = (r + dr >= 0) & (r + dr < G) & (c + dc >= 0) & (c + dc < G)
        arcs.append(np.c_[node[ok], node[ok] + dr * G + dc])
    arcs = np.concatenate(arcs)
    arcs = arcs[np.lexsort((arcs[:, 1], arcs[:, 0]))]
    na, nc = len(arcs), G * G - 1
    tri = np.empty((K, na, 3), np.int64)
    sgn = np.empty((K, na, 3))
    lo_tail = arcs[:, 0] < arcs[:, 1]
    for q in range(K):
        tri[q, :, 0] = arcs.min(axis=1) + q * nc
        tri[q, :, 1] = arcs.max(axis=1) + q * nc
        tri[q, :, 2] = K * nc + np.arange(na)
        sgn[q, :, 0] = np.where(lo_tail, 1.0, -1.0)
        sgn[q, :, 1] = -sgn[q, :, 0]
        sgn[q, :, 2] = 1.0
    keep = np.ones((K, na, 3), bool)
    keep[:, :, 1] = arcs.max(axis=1) < nc
    counts = np.r_[keep.sum(axis=2).ravel(), np.ones(na, int)]
    rows = np.r_[tri[keep], K * nc + np.arange(na)]
    return _columns(K * nc + na, counts, rows) + (np.r_[sgn[keep], np.ones(na)],)


def _instance(case, rng):
    m, n, colptr, rowind, val = _pattern(case["family"], case["size"], case["size2"])
    if val is None:
        val = rng.standard_normal(len(rowind))
        val[colptr[n - m]:] = 1.0     # the identity's columns
    return Instance(m, n, colptr, rowind, val, np.zeros(m), np.zeros(n))


def _inputs(case, seed):
    """The instance, d and the vectors of the case's operation (host arrays)."""
    rng = np.random.default_rng([int(seed), 11])
    inst = _instance(case, rng)
    m, n = inst.m, inst.n
    dec = case["decades"]
    d = np.exp(rng.uniform(-dec, dec, n) * np.log(10.0))
    op = case["op"]
    if op in ("iteration", "solves"):
        vec = [v for _ in range(3) for v in (rng.standard_normal(n), rng.standard_normal(m))]
    elif op == "build":
        vec = [rng.standard_normal(m)]
    elif op == "pcg":
        vec = [rng.standard_normal(n), rng.standard_normal(m)]
    else:
        # r and a target whose scaled values are of order one, as dy g / rms(r) is
        r = rng.standard_normal(m)
        g = np.bincount(inst.rowind, inst.val ** 2 / np.repeat(d, np.diff(inst.colptr)), m)
        vec = [r, rng.standard_normal(m) / g]
    return inst, d, vec


# --------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest LP: the host driver's calls (host arrays), launches and latency
        dict(name="ipm_random2000_fp64_amd", op="iteration", family="random", size=2000, size2=4,
             mode="fp64", order="amd", decades=2.0, host=True),
        # the grid LP with HELP's default ordering, driven from the GPU
        dict(name="ipm_mcf150x8_fp64_amd", op="iteration", family="mcf", size=150, size2=8,
             mode="fp64", order="amd", decades=1.0, host=False),
        # an odd-sized grid in the mixed-precision mode
        dict(name="ipm_mcf61x3_fp32_amd", op="iteration", family="mcf", size=61, size2=3,
             mode="fp32", order="amd", decades=1.0, host=False),
        # the headline LP: dense fronts, nested dissection, both precisions
        dict(name="ipm_staircase200_fp64_nd", op="iteration", family="staircase", size=200, size2=1000,
             mode="fp64", order="nd", decades=2.0, host=False),
        dict(name="ipm_staircase200_fp32_nd", op="iteration", family="staircase", size=200, size2=1000,
             mode="fp32", order="nd", decades=2.0, host=False),
        # the staircase as HELP runs it by default: AMD, a long chain of panels
        dict(name="ipm_staircase25_fp64_amd", op="iteration", family="staircase", size=25, size2=1000,
             mode="fp64", order="amd", decades=2.0, host=False),
        # triangular solves alone: every further right-hand side of a factor
        dict(name="solves_staircase200_fp64_nd", op="solves", family="staircase", size=200, size2=1000,
             mode="fp64", order="nd", decades=2.0, host=False),
        # PCG mode at the size it is for: the preconditioner, and one system
        dict(name="build_zipf1e6_k500", op="build", family="zipf", size=1000000, size2=0, k=500, fp32=1,
             decades=1.0, host=False),
        dict(name="pcg_zipf1e6_k500", op="pcg", family="zipf", size=1000000, size2=0, k=500, fp32=1,
             decades=0.5, host=False),
        # ... and a small odd one with the FP64 apply
        dict(name="pcg_zipf31415_k77_fp64", op="pcg", family="zipf", size=31415, size2=0, k=77, fp32=0,
             decades=0.5, host=False),
        # the warm start: a guess per solve, and the training step that makes it
        dict(name="predict_mcf150x8_bf16", op="predict", family="mcf", size=150, size2=8, bf16=1, decades=1.0,
             host=True),
        dict(name="train_mcf105x5_bf16", op="train", family="mcf", size=105, size2=5, bf16=1, decades=1.0,
             host=True),
    ]


def _between(rng, lo, hi):
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))


def draw(rng):
    kind = rng.choice(["random", "mcf", "staircase", "staircase", "build", "pcg", "net", "net"])
    host = rng.random() < 0.3
    direct = dict(op=rng.choice(["iteration", "iteration", "solves"]), mode=rng.choice(["fp64", "fp32"]),
                  order=rng.choice(["amd", "nd"]), host=host)
    if kind == "random":
        return dict(direct, family="random", size=_between(rng, 300, 5000), size2=rng.randint(3, 6),
                    decades=rng.choice([1.0, 2.0]))
    if kind == "mcf":
        return dict(direct, family="mcf", size=_between(rng, 20, 150), size2=rng.randint(2, 8), decades=1.0)
    if kind == "staircase":
        return dict(direct, family="staircase", size=_between(rng, 4, 120), size2=_between(rng, 250, 1000),
                    decades=rng.choice([1.0, 2.0]))
    if kind in ("build", "pcg"):
        return dict(op=kind, family="zipf", size=_between(rng, 20000, 900000), size2=0, k=_between(rng, 40, 500),
                    fp32=rng.choice([1, 1, 0]), decades=1.0 if kind == "build" else 0.5, host=host)
    return dict(op=rng.choice(["predict", "train"]), family="mcf", size=_between(rng, 30, 150),
                size2=rng.randint(2, 8), bf16=rng.choice([1, 1, 0]), decades=1.0, host=True)


def prepare(case, seed):
    inst, d, vec = _inputs(case, seed)
    op = case["op"]
    if op in ("iteration", "solves"):
        le = LinearEquation(mode=L.MODE_DIRECT_FP64 if case["mode"] == "fp64" else L.MODE_DIRECT_FP32,
                            ordering=L.ORDER_AMD if case["order"] == "amd" else L.ORDER_ND)
    elif op in ("build", "pcg"):
        le = LinearEquation(mode=L.MODE_PCG, pcg_k=case["k"], pcg_fp32_precond=case["fp32"])
    else:
        le = LinearEquation(mode=L.MODE_PCG, pcg_k=0)
    le.construct(inst)
    s = dict(op=op, le=le, host=case["host"], m=inst.m, n=inst.n)
    if op in ("predict", "train"):
        s["net"] = Mpnn(bf16=bool(case["bf16"]))
        s["net"].set_params(np.load(NET)["params"])
    if case["host"]:
        s["d"], s["v"] = d, vec
        if op in ("solves", "pcg"):
            le.renew(d)
        return s
    s["d"] = torch.from_numpy(d).cuda()
    s["v"] = [torch.from_numpy(v).cuda() for v in vec]
    sizes = {"iteration": (inst.n, inst.m) * 3, "solves": (inst.n, inst.m) * 3, "build": (inst.m,),
             "pcg": (inst.n, inst.m)}[op]
    s["x"] = [torch.empty(k, dtype=torch.float64, device="cuda") for k in sizes]
    torch.cuda.synchronize()
    if op in ("solves", "pcg"):
        _ok(L.lib().help_gpu_renew(le.h, _p(s["d"]), None), "renew")
    return s


def _p(t):
    return C.cast(t.data_ptr(), C.POINTER(C.c_double))


def _ok(st, what):
    if st != L.HELP_OK:
        raise HelpError(st, what)


def run(s):
    op, le, d, v = s["op"], s["le"], s["d"], s["v"]
    if op == "predict":
        return s["net"].predict(le, d, v[0])
    if op == "train":
        loss, grad = s["net"].loss_grad(le, d, v[0], v[1], want_grad=True)
        return [loss, grad]
    if s["host"]:                    # the Python interface, host arrays
        if op in ("iteration", "build"):
            le.renew(d)
        if op == "build":
            return [le.pcg_apply(v[0])]
        if op == "pcg":
            return list(le.solve(d, v[0], v[1]))
        (x1a, x2a), (x1b, x2b) = le.solve2(d, v[0], v[1], v[2], v[3])
        return [x1a, x2a, x1b, x2b] + list(le.solve(d, v[4], v[5]))
    lib, h, dp = L.lib(), le.h, _p(d)     # the C interface, device arrays
    vp, x = [_p(t) for t in v], s["x"]
    xp = [_p(t) for t in x]
    if op in ("iteration", "build"):
        _ok(lib.help_gpu_renew(h, dp, None), "renew")
    if op == "build":
        _ok(lib.help_gpu_pcg_apply(h, vp[0], xp[0]), "pcg_apply")
    elif op == "pcg":
        _ok(lib.help_gpu_solve(h, dp, vp[0], vp[1], xp[0], xp[1], None), "solve")
    else:
        _ok(lib.help_gpu_solve2(h, dp, vp[0], vp[1], xp[0], xp[1], vp[2], vp[3], xp[2], xp[3], None, None), "solve2")
        _ok(lib.help_gpu_solve(h, dp, vp[4], vp[5], xp[4], xp[5], None), "solve")
    return x


# ---------------------------------------------------------------------- work
@functools.lru_cache(maxsize=16)
def _fill(family, size, size2, order):
    """(entries of L, factor flops) of the instance under the ordering"""
    m, n, colptr, rowind, val = _pattern(family, size, size2)
    le = LinearEquation(symbolic_only=True, ordering=L.ORDER_AMD if order == "amd" else L.ORDER_ND)
    le.construct(Instance(m, n, colptr, rowind, np.ones(len(rowind)) if val is None else val, np.zeros(m), np.zeros(n)))
    info = le.symbolic_info()
    return info.nnz_l_exact, info.factor_flops


def work(case):
    m, n, colptr, rowind, _ = _pattern(case["family"], case["size"], case["size2"])
    nnz, op = len(rowind), case["op"]
    a = 12 * nnz + 8 * n                       # A once: values, indices, pointers
    if op in ("iteration", "solves"):
        nl, fl = _fill(case["family"], case["size"], case["size2"], case["order"])
        es = 8 if case["mode"] == "fp64" else 4
        # three systems: A read for the right-hand side and for x1, L read in
        # each direction, by two systems at once the first time
        by = 3 * (2 * a + 8 * (3 * n + 2 * m)) + 2 * 2 * es * nl
        fp = 3 * (4 * nnz + 4 * nl)
        if op == "iteration":
            by += a + 8 * n + es * nl
            fp += fl + 2 * nnz
        return {"bytes": by, "flops": fp}
    if op in ("build", "pcg"):
        k, es = case["k"], 4 if case["fp32"] else 8
        if op == "build":                      # the m x k factor written once and read by one apply
            return {"bytes": a + 8 * n + (8 + es) * m * k + 32 * m, "flops": 1.0 * m * k * k + 4 * m * k}
        # an iteration reads A and its transpose and the factor once; about twenty of them
        return {"bytes": 20 * (2 * a + es * m * k + 64 * m) + 2 * a, "flops": 20 * (4 * nnz + 4 * m * k)}
    es = 2 if case["bf16"] else 4
    nodes = (m + n) * HIDDEN * es              # one width of activations of every node
    layers = 2 * 2 * HIDDEN * HIDDEN * 2 * (m + n) + 2 * HIDDEN * HIDDEN * m + 4 * 2 * nnz * HIDDEN
    by = 4 * a + 8 * nodes + 16 * (m + n)
    return {"bytes": by, "flops": layers} if op == "predict" else {"bytes": 3 * by, "flops": 3 * layers}


# --------------------------------------------------------------------- exact
def _sparse(inst, dev):
    """A and A^T as CSR tensors in 64 bits"""
    cp, ri, v = (torch.from_numpy(x).to(dev) for x in (inst.colptr, inst.rowind.astype(np.int64), inst.val))
    At = torch.sparse_csr_tensor(cp, ri, v, size=(inst.n, inst.m))
    col = torch.repeat_interleave(torch.arange(inst.n, device=dev), cp[1:] - cp[:-1])
    order = torch.argsort(ri, stable=True)
    rp = torch.zeros(inst.m + 1, dtype=torch.int64, device=dev)
    rp[1:] = torch.cumsum(torch.bincount(ri, minlength=inst.m), 0)
    return torch.sparse_csr_tensor(rp, col[order], v[order], size=(inst.m, inst.n)), At, ri, col, v


def _normal_solve(A, At, diag, dinv, beta, rhs, most=6000):
    """(A D^-1 A^T + beta I) x = rhs by conjugate gradients with the diagonal
    as preconditioner, restarted from the true residual; None if it does not
    get to the rounding floor."""
    def mul(x):
        return A @ (dinv * (At @ x)) + beta * x
    x, floor = torch.zeros_like(rhs), 3e-15 * torch.linalg.norm(rhs)
    w, used = 1.0 / (diag + beta), 0
    for _ in range(4):
        r = rhs - mul(x)
        goal = max(float(1e-10 * torch.linalg.norm(r)), float(0.2 * floor))
        z = w * r
        p, rz = z.clone(), torch.dot(r, z)
        while float(torch.linalg.norm(r)) > goal:
            for _ in range(10):
                q = mul(p)
                al = rz / torch.dot(p, q)
                x = x + al * p
                r = r - al * q
                z = w * r
                rn = torch.dot(r, z)
                p, rz = z + (rn / rz) * p, rn
            used += 10
            if used > most:
                return None
    return x


def _pivoted(A, At, inst, ri, col, v, diag, dinv, K, r):
    """M^-1 r with the greedy partial Cholesky factor of A D^-1 A^T (K
    pivots): M = [L11 0; L21 I] diag(D, S) [L11 0; L21 I]^T."""
    m, dev = inst.m, r.device
    S, rp, ci, av = diag.clone(), A.crow_indices(), A.col_indices(), A.values()
    Lf, D = torch.zeros((K, m), dtype=torch.float64, device=dev), torch.zeros(K, dtype=torch.float64, device=dev)
    free, piv = torch.ones(m, dtype=torch.bool, device=dev), []
    for k in range(K):
        i = int(torch.argmax(torch.where(free, S, torch.full_like(S, -np.inf))))
        b, e = int(rp[i]), int(rp[i + 1])
        t = torch.zeros(inst.n, dtype=torch.float64, device=dev)
        t[ci[b:e]] = av[b:e] * dinv[ci[b:e]]
        w = D[:k] * Lf[:k, i]
        u = A @ t - w @ Lf[:k]
        D[k] = u[i]
        free[i] = False
        Lf[k] = torch.where(free, u / D[k], torch.zeros_like(u))
        Lf[k, i] = 1.0
        S = torch.where(free, S - D[k] * Lf[k] ** 2, S)
        piv.append(i)
    at = torch.tensor(piv, device=dev)
    L11 = Lf[:, at].T
    y1 = torch.linalg.solve_triangular(L11, r[at, None], upper=False, unitriangular=True)[:, 0]
    z = torch.where(free, (r - y1 @ Lf) / S, torch.zeros_like(r))
    # the pivots' own diagonal is the Schur diagonal at the time they were taken
    w = y1 / S[at] - Lf @ z
    z[at] = torch.linalg.solve_triangular(L11.T, w[:, None], upper=True, unitriangular=True)[:, 0]
    return z


def _network(case, inst, A, At, diag, dinv, r, dy):
    """The network's guess, or its loss and weight gradient, in 64 bits."""
    dev = r.device
    flat = torch.from_numpy(np.load(NET)["params"]).to(dev)
    if case["bf16"]:
        flat = flat.to(torch.bfloat16)
    flat = flat.double().requires_grad_(case["op"] == "train")
    at = [0]

    def take(*shape):
        b = at[0]
        at[0] += int(np.prod(shape))
        return flat[b:at[0]].reshape(shape)
    H = HIDDEN
    Wr, br, Wc, bc = take(4, H), take(H), take(2, H), take(H)
    lay = [(take(2 * H, H), take(H)) for _ in range(4)]
    Wh, bh, wo, bo = take(H, H), take(H), take(H), take(1)
    rs = torch.sqrt(torch.mean(r * r))
    mu, nu = torch.log(diag).mean(), torch.log(dinv).mean()
    jac = torch.clamp(torch.exp(mu) * r / (rs * diag), -10.0, 10.0)
    one = torch.ones_like
    xr = torch.stack([r / rs, (torch.log(diag) - mu) / 10, jac / 10, one(r)], 1)
    xc = torch.stack([(torch.log(dinv) - nu) / 10, one(dinv)], 1)
    degr = torch.clamp((A.crow_indices()[1:] - A.crow_indices()[:-1]).double(), min=1.0)[:, None]
    degc = torch.clamp((At.crow_indices()[1:] - At.crow_indices()[:-1]).double(), min=1.0)[:, None]

    class Mean(torch.autograd.Function):
        @staticmethod
        def forward(ctx, h, B, Bt, deg):
            ctx.Bt, ctx.deg = Bt, deg
            return (B @ h) / deg

        @staticmethod
        def backward(ctx, g):
            return ctx.Bt @ (g / ctx.deg).contiguous(), None, None, None
    relu = torch.relu
    hr, hc = relu(xr @ Wr + br), relu(xc @ Wc + bc)
    for l, (W, b) in enumerate(lay):
        if l % 2 == 0:
            hc = relu(torch.cat([hc, Mean.apply(hr, At, A, degc)], 1) @ W + b)
        else:
            hr = relu(torch.cat([hr, Mean.apply(hc, A, At, degr)], 1) @ W + b)
    y = relu(hr @ Wh + bh) @ wo + bo
    if case["op"] == "predict":
        return y.detach() * rs / diag
    t = dy * diag / rs
    loss = ((y - t) ** 2).sum() / (t * t).sum()
    loss.backward()
    return [float(loss.detach()), flat.grad]


def exact(case, seed):
    op = case["op"]
    inst, d, vec = _inputs(case, seed)
    if op == "build" and inst.m > 40000 or op in ("iteration", "solves") and case["family"] == "mcf" and inst.m > 60000:
        return None                            # minutes in plain torch
    dev = "cuda"
    A, At, ri, col, v = _sparse(inst, dev)
    dt = torch.from_numpy(d).to(dev)
    dinv = 1.0 / dt
    vec = [torch.from_numpy(x).to(dev) for x in vec]
    diag = torch.zeros(inst.m, dtype=torch.float64, device=dev).index_add_(0, ri, v * v * dinv[col])
    if op in ("predict", "train"):
        return _network(case, inst, A, At, diag, dinv, vec[0], vec[1])
    if op == "build":
        return [_pivoted(A, At, inst, ri, col, v, diag, dinv, case["k"], vec[0])]
    beta = BETA if op in ("iteration", "solves") else 0.0
    out = []
    for b1, b2 in zip(vec[0::2], vec[1::2]):
        x2 = _normal_solve(A, At, diag, dinv, beta, A @ (b1 / dt) - b2)
        if x2 is None:
            return None
        out += [(b1 - At @ x2) / dt, x2]
    return out
