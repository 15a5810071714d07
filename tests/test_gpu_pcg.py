"""GPU parity of the matrix-free PCG mode (HELP PCG.cpp / UsePCG_CPU.cpp):
the partial-Cholesky preconditioner against the CPU oracle, the solve against
dense and sparse direct solves, and the HSD driver end to end."""
import ctypes as C
import json
import os

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import oracle_bind as O
from help_amd import Instance, LinearEquation, instances
from help_amd import _lib as L

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


def _flush(msg):
    print(msg, flush=True)


def _csc(inst):
    return sp.csc_matrix((inst.val, inst.rowind, inst.colptr), shape=(inst.m, inst.n))


def _oracle_pchol(inst, d, K):
    rp, ci, pos = O.csr(inst)
    cv = np.ascontiguousarray(inst.val[pos])
    pc = O.PChol()
    O.lib().or_pchol_build(inst.m, inst.n, O.i64(rp), O.i32(ci), O.d(cv), O.d(d), 0.0, 0.0, K, pc)
    m = inst.m
    out = (np.ctypeslib.as_array(pc.perm, shape=(m,)).copy(),
           np.ctypeslib.as_array(pc.D, shape=(K,)).copy(),
           np.ctypeslib.as_array(pc.diag_s, shape=(m,)).copy(),
           np.ctypeslib.as_array(pc.L, shape=(m * K,)).reshape(m, K).copy())
    O.lib().or_pchol_free(pc)
    return out


@pytest.mark.parametrize("name,maker,K", [
    ("random", lambda: instances.random_lp(300, 600, 4, seed=21), 20),
    ("zipf-heavy-rows", lambda: instances.zipf(3000, 9000, 6, 1.1, seed=22), 40)])
def test_partial_cholesky_matches_oracle(name, maker, K):
    inst = maker()
    rp = O.csr(inst)[0]
    _flush(f"pcg factor {name} m={inst.m} n={inst.n} K={K} max row nnz={int(np.diff(rp).max())}")
    rng = np.random.default_rng(1)
    d = np.exp(rng.uniform(-2, 2, inst.n) * np.log(10.0))
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=K)
    be.construct(inst)
    be.renew(d)
    perm, D, S, Lg = be.pcg_factor()
    be.destruct()
    operm, oD, oS, oL = _oracle_pchol(inst, d, K)
    assert np.array_equal(perm, operm)
    assert np.allclose(D, oD, rtol=1e-11, atol=0)
    assert np.allclose(S, oS, rtol=1e-9, atol=1e-12 * np.abs(oS).max())
    assert np.allclose(Lg, oL, rtol=1e-9, atol=1e-11)


def _spread(inst, rng):
    return np.exp(rng.uniform(-2, 2, inst.n) * np.log(10.0))


def _shared_column(inst, rng):
    """d so small on one column that its rows lead the Schur diagonal until the
    first of them is taken: the others were candidates and fall behind"""
    d = np.exp(rng.uniform(-0.5, 0.5, inst.n) * np.log(10.0))
    d[3] = 1e-8
    return d


@pytest.mark.parametrize("name,maker,K,dfun", [
    ("one pivot", lambda: instances.random_lp(300, 600, 4, seed=71), 1, _spread),
    ("one block", lambda: instances.random_lp(300, 600, 4, seed=72), 16, _spread),
    ("a block and one", lambda: instances.random_lp(300, 600, 4, seed=73), 17, _spread),
    ("fewer rows than candidates", lambda: instances.random_lp(5, 9, 3, seed=74), 5, _spread),
    ("ties", lambda: instances.mcf(side=6, commodities=2, pairs=3, seed=75), 40, lambda inst, rng: np.ones(inst.n)),
    ("candidates that fall behind", lambda: instances.random_lp(400, 700, 12, seed=76), 37, _shared_column),
    ("zipf-heavy-rows", lambda: instances.zipf(3000, 9000, 6, 1.1, seed=77), 50, _spread)])
def test_partial_cholesky_blocks_match_oracle(name, maker, K, dfun):
    """The build takes its pivots from blocks of 16 candidates: the greedy order
    of the oracle all the same, and the factor within the bars of
    test_partial_cholesky_matches_oracle."""
    inst = maker()
    d = dfun(inst, np.random.default_rng(5))
    _flush(f"pcg factor blocks, {name}: m={inst.m} n={inst.n} K={K}")
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=K)
    be.construct(inst)
    be.renew(d)
    perm, D, S, Lg = be.pcg_factor()
    be.destruct()
    operm, oD, oS, oL = _oracle_pchol(inst, d, K)
    assert np.array_equal(perm, operm)
    assert np.allclose(D, oD, rtol=1e-11, atol=0)
    assert np.allclose(S, oS, rtol=1e-9, atol=1e-12 * np.abs(oS).max())
    assert np.allclose(Lg, oL, rtol=1e-9, atol=1e-11)


def _parallel_rows(sizes, tail, seed):
    """Rows in groups of the given sizes, a group's rows nearly parallel (three
    columns of entries 1 +- 0.001), each group's diagonals 0.97 times those of the
    one before, `tail` small rows behind, every row with a small column of its
    own and weakly coupled to others; and a d under which the groups' columns
    hardly count and all rows differ."""
    rng = np.random.default_rng(seed)
    G, m = len(sizes), sum(sizes) + tail
    first = np.concatenate(([0], np.cumsum(sizes)))
    grp = [np.arange(first[g], first[g + 1]) for g in range(G)] * 3
    far = np.sort(rng.integers(0, m, (2 * m, 4)), axis=1)
    far = far[(far[:, 1:] != far[:, :-1]).all(axis=1)]
    counts = np.concatenate(([len(r) for r in grp], np.full(len(far), 4), np.ones(m, int)))
    rowind = np.concatenate(grp + [far.ravel(), np.arange(m)]).astype(np.int32)
    val = np.concatenate((1 + 1e-3 * rng.standard_normal(3 * sum(sizes)), 0.01 * rng.standard_normal(far.size), np.ones(m)))
    n = len(counts)
    inst = Instance(m, n, np.concatenate(([0], np.cumsum(counts))).astype(np.int64), rowind, val, np.ones(m), np.ones(n))
    close, apart = np.ones(n), np.ones(n)
    close[:3 * G] = np.tile(1e-4 / 0.97 ** np.arange(G), 3)
    close[-m:] = 1e3
    apart[:3 * G] = 1e6
    apart[-m:] = np.exp(rng.uniform(-1, 1, m) * np.log(10.0))
    return inst, close, apart


@pytest.mark.parametrize("name,sizes,K", [
    ("groups of 20", [20] * 60, 50),
    ("few pivots", [20] * 30, 3),
    ("at most two blocks of pivots", [20] * 30, 27),
    ("groups, then single rows, then groups", [20] * 9 + [1] * 90 + [20] * 40, 120),
    ("single rows, then groups of 5", [1] * 55 + [5] * 60, 99),
    ("single rows", [1] * 150, 130)])
def test_partial_cholesky_parallel_rows_match_oracle(name, sizes, K):
    """Where few of a group's candidates are taken the build goes on pivot by
    pivot, and back to blocks where many are: the oracle's pivots and factor
    within the bars of test_partial_cholesky_matches_oracle.  (The groups' leaders
    stay ahead of what a first pivot leaves of the others, some 1e-6 of it.)"""
    inst, d, _ = _parallel_rows(sizes, 300, seed=81)
    _flush(f"pcg factor, {name}: m={inst.m} n={inst.n} K={K}")
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=K)
    be.construct(inst)
    be.renew(d)
    perm, D, S, Lg = be.pcg_factor()
    be.destruct()
    operm, oD, oS, oL = _oracle_pchol(inst, d, K)
    assert np.array_equal(perm, operm)
    assert np.allclose(D, oD, rtol=1e-11, atol=0)
    assert np.allclose(S, oS, rtol=1e-9, atol=1e-12 * np.abs(oS).max())
    assert np.allclose(Lg, oL, rtol=1e-9, atol=1e-11)


@pytest.mark.parametrize("sizes", [[20] * 30, [1] * 60])
@pytest.mark.parametrize("K", [7, 8, 9])
def test_partial_cholesky_first_blocks_match_oracle(K, sizes):
    """The fewest pivots that a block can follow the first four ones with, and
    one fewer (no memory for blocks then), within the bars of
    test_partial_cholesky_matches_oracle."""
    inst, d, _ = _parallel_rows(sizes, 300, seed=84)
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=K)
    be.construct(inst)
    be.renew(d)
    perm, D, S, Lg = be.pcg_factor()
    be.destruct()
    operm, oD, oS, oL = _oracle_pchol(inst, d, K)
    assert np.array_equal(perm, operm)
    assert np.allclose(D, oD, rtol=1e-11, atol=0)
    assert np.allclose(S, oS, rtol=1e-9, atol=1e-12 * np.abs(oS).max())
    assert np.allclose(Lg, oL, rtol=1e-9, atol=1e-11)


def test_no_block_memory_without_pivots():
    """A handle with pcg_k = 0 (a diagonal preconditioner, or the network's graph
    alone) holds nothing of the build: what one with K = 64 holds beside it is
    at least the build's blocks, 16 n + 80 m doubles, and 63 more factor columns
    in FP64 and FP32 (64 MiB for the allocator's rounding)."""
    from test_zz_no_alloc import _hip
    hip = _hip()
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t)] * 2

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value
    inst = instances.random_lp(400000, 800000, 3, seed=85)
    held = {}
    for K in (0, 64):
        be = LinearEquation(mode=L.MODE_PCG, pcg_k=0)
        be.construct(instances.random_lp(100, 200, 3, seed=86))   # (the runtime's own allocations)
        be.destruct()
        before = free()
        be = LinearEquation(mode=L.MODE_PCG, pcg_k=K)
        be.construct(inst)
        held[K] = before - free()
        be.destruct()
    _flush(f"m={inst.m} n={inst.n}: {held[0] / 2**20:.0f} MiB with K = 0, {held[64] / 2**20:.0f} MiB with K = 64")
    assert held[64] - held[0] >= 8 * (16 * inst.n + 80 * inst.m) + 63 * 12 * inst.m - 2**26


def test_partial_cholesky_cost_on_parallel_rows():
    """A block of 16 candidates that takes one of them costs several single
    pivots.  Rows in groups of 20 near-parallel ones (one candidate per block)
    against the same instance with all rows apart (every candidate taken), 200
    pivots of 200,000 rows: 3.2 times as long pivot by pivot, 10 times in
    blocks; the bar is between the two."""
    inst, close, apart = _parallel_rows([20] * 10000, 0, seed=82)
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=200)
    be.construct(inst)
    ms = {}
    for name, d in (("apart", apart), ("close", close)):
        for _ in range(5):
            be.renew(d)
            ms[name] = min(ms.get(name, np.inf), be.renew_stats.ms_precond)
    be.destruct()
    _flush(f"build of 200 pivots, m={inst.m}: rows apart {ms['apart']:.2f} ms, in groups {ms['close']:.2f} ms")
    assert ms["close"] <= 5.5 * ms["apart"]


def test_partial_cholesky_ends_without_numbers():
    """Where every Schur diagonal left is NaN the pivots are the rows at the next
    positions: the build ends with a permutation."""
    inst = instances.random_lp(300, 600, 4, seed=83)
    for bad in (1, inst.n):
        d = np.ones(inst.n)
        d[:bad] = np.nan
        be = LinearEquation(mode=L.MODE_PCG, pcg_k=60)
        be.construct(inst)
        be.renew(d)
        perm = be.pcg_factor()[0]
        be.destruct()
        assert np.array_equal(np.sort(perm), np.arange(inst.m))


def test_pcg_solve_matches_dense():
    inst = instances.random_lp(400, 800, 4, seed=23)
    rng = np.random.default_rng(2)
    d = np.exp(rng.uniform(-2, 2, inst.n) * np.log(10.0))
    b1 = rng.standard_normal(inst.n)
    b2 = rng.standard_normal(inst.m)
    _flush("pcg solve vs dense, random 400x800")
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=30, pcg_tol=1e-12)
    be.construct(inst)
    be.renew(d)
    x1, x2 = be.solve(d, b1, b2)
    st = be.solve_stats
    be.destruct()
    A = _csc(inst).toarray()
    M = A @ np.diag(1.0 / d) @ A.T          # gamma = delta = 0 (UsePCG_CPU.cpp:154-155)
    x2r = np.linalg.solve(M, A @ (b1 / d) - b2)
    x1r = (b1 - A.T @ x2r) / d
    _flush(f"  iterations {st.pcg_iters} rel residual {st.rel_residual:.2e}")
    assert 0 < st.pcg_iters < 400 and st.rel_residual <= 1e-12
    assert np.linalg.norm(x2 - x2r) <= 1e-8 * np.linalg.norm(x2r)
    assert np.linalg.norm(x1 - x1r) <= 1e-8 * np.linalg.norm(x1r)


def test_pcg_solve_heavy_rows_matches_sparse_direct():
    """Rows with thousands of nonzeros go through the chunked product."""
    inst = instances.zipf(3000, 9000, 6, 1.1, seed=24)
    rng = np.random.default_rng(3)
    d = np.exp(rng.uniform(-1, 1, inst.n) * np.log(10.0))
    b1 = rng.standard_normal(inst.n)
    b2 = rng.standard_normal(inst.m)
    _flush("pcg solve vs sparse direct, zipf 3000x9000")
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=50, pcg_tol=1e-12, pcg_max_iter=3000)
    be.construct(inst)
    be.renew(d)
    x1, x2 = be.solve(d, b1, b2)
    st = be.solve_stats
    be.destruct()
    A = _csc(inst)
    M = (A @ sp.diags(1.0 / d) @ A.T).tocsc()
    x2r = spla.spsolve(M, A @ (b1 / d) - b2)
    _flush(f"  iterations {st.pcg_iters} rel residual {st.rel_residual:.2e}")
    assert st.rel_residual <= 1e-12
    assert np.linalg.norm(x2 - x2r) <= 1e-7 * np.linalg.norm(x2r)


@pytest.mark.parametrize("device", [False, True])
def test_hsd_pcg_mode_reaches_highs_objective(device):
    from help_amd.hsd import GpuBackend, solve_lp
    spec = json.load(open(os.path.join(HERE, "golden", "hsd_objectives.json")))["random_300x600_s1000"]
    inst = getattr(instances, spec["generator"])(**spec["params"])
    _flush(f"hsd pcg mode device_driver={device}")
    gb = GpuBackend(mode=L.MODE_PCG, pcg_k=50)
    res, rows = solve_lp(inst, gb.table, device=device)
    gb.close()
    _flush(f"  status {res.status} iters {res.iterations} pobj {res.primal_obj!r} (HiGHS {spec['objective']!r})")
    assert res.backend_error == 0
    assert L.HSD_STATUS[res.status] == "OK"
    assert abs(res.primal_obj - spec["objective"]) <= 1e-6 * (1 + abs(spec["objective"]))


@pytest.mark.parametrize("fp32", [1, 0])
@pytest.mark.parametrize("name,maker,K", [
    ("random", lambda: instances.random_lp(300, 600, 4, seed=31), 20),
    ("zipf-heavy-rows", lambda: instances.zipf(3000, 9000, 6, 1.1, seed=32), 40)])
def test_preconditioner_apply_matches_oracle(name, maker, K, fp32):
    """The apply z = M^-1 r of PCG.cpp:183-196 (L^-T D_S^-1 L^-1 with
    L = [L11 0; L21 I]) against the oracle's or_pchol_apply, which the CPU
    tests pin to the explicit dense inverse.  FP64 factor: within 1e-12
    relative.  FP32 factor (every L21 entry rounded to FP32, relative 6e-8,
    vectors and sums in FP64): within 1e-5 relative."""
    inst = maker()
    rng = np.random.default_rng(7)
    d = np.exp(rng.uniform(-2, 2, inst.n) * np.log(10.0))
    r = rng.standard_normal(inst.m)
    _flush(f"pcg apply {name} m={inst.m} K={K} fp32={fp32}")
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=K, pcg_fp32_precond=fp32)
    be.construct(inst)
    be.renew(d)
    z = be.pcg_apply(r)
    z2 = be.pcg_apply(r)
    be.destruct()
    rp, ci, pos = O.csr(inst)
    cv = np.ascontiguousarray(inst.val[pos])
    pc = O.PChol()
    O.lib().or_pchol_build(inst.m, inst.n, O.i64(rp), O.i32(ci), O.d(cv), O.d(d), 0.0, 0.0, K, pc)
    perm = np.ctypeslib.as_array(pc.perm, shape=(inst.m,)).copy()
    rperm = np.ascontiguousarray(r[perm])
    zp = np.empty(inst.m)
    work = np.empty(2 * inst.m)
    O.lib().or_pchol_apply(pc, O.d(rperm), O.d(zp), O.d(work))
    O.lib().or_pchol_free(pc)
    zo = np.empty(inst.m)
    zo[perm] = zp
    err = np.linalg.norm(z - zo) / np.linalg.norm(zo)
    _flush(f"  rel err vs oracle {err:.3e}")
    assert np.array_equal(z, z2)
    assert err <= (1e-5 if fp32 else 1e-12)


@pytest.mark.parametrize("K", [1, 2, 127, 129, 256, 257, 512, 513])
@pytest.mark.parametrize("fp32", [0, 1])
def test_preconditioner_apply_column_counts(K, fp32):
    """The apply at the edges of its column groups (four columns per workgroup of
    the transposed product, eight interleaved chains and 64 pivots in the last
    one; an odd K has a zero column after it), m no multiple of its rows'
    blocks, against the oracle within the bars of
    test_preconditioner_apply_matches_oracle."""
    inst = instances.random_lp(1237, 2400, 4, seed=61)
    rng = np.random.default_rng(9)
    d = np.exp(rng.uniform(-1, 1, inst.n) * np.log(10.0))
    r = rng.standard_normal(inst.m)
    _flush(f"pcg apply m={inst.m} K={K} fp32={fp32}")
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=K, pcg_fp32_precond=fp32)
    be.construct(inst)
    be.renew(d)
    z = be.pcg_apply(r)
    be.destruct()
    rp, ci, pos = O.csr(inst)
    cv = np.ascontiguousarray(inst.val[pos])
    pc = O.PChol()
    O.lib().or_pchol_build(inst.m, inst.n, O.i64(rp), O.i32(ci), O.d(cv), O.d(d), 0.0, 0.0, K, pc)
    perm = np.ctypeslib.as_array(pc.perm, shape=(inst.m,)).copy()
    rperm = np.ascontiguousarray(r[perm])
    zp, work, zo = np.empty(inst.m), np.empty(2 * inst.m), np.empty(inst.m)
    O.lib().or_pchol_apply(pc, O.d(rperm), O.d(zp), O.d(work))
    O.lib().or_pchol_free(pc)
    zo[perm] = zp
    err = np.linalg.norm(z - zo) / np.linalg.norm(zo)
    _flush(f"  rel err vs oracle {err:.3e}")
    assert err <= (1e-5 if fp32 else 1e-12)


def test_heavy_rows_in_column_blocks():
    """Rows above 1,024 nonzeros are cut into chunks of 4,096 dealt out to the
    XCDs by their columns: on an instance with rows of more than 64 chunks,
    the Schur diagonal before the first pivot (K = 0) is the diagonal of A D^-1 A^T
    within the rounding of a sum of that many positive terms."""
    inst = instances.zipf(2000, 600000, 6, 1.1, seed=62)
    rng = np.random.default_rng(10)
    d = np.exp(rng.uniform(-1, 1, inst.n) * np.log(10.0))
    most = int(np.bincount(inst.rowind, minlength=inst.m).max())
    _flush(f"heavy rows m={inst.m} n={inst.n} longest {most}")
    assert most > 262144
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=0)
    be.construct(inst)
    be.renew(d)
    _, _, S, _ = be.pcg_factor()
    be.destruct()
    ref = np.bincount(inst.rowind, inst.val ** 2 / np.repeat(d, np.diff(inst.colptr)), inst.m)
    assert np.allclose(S, ref, rtol=most * np.finfo(float).eps, atol=0)


def test_column_products_in_chunks():
    """A^T x adds each column from LDS chunks of 1,024 nonzeros: columns that
    end inside, at and beyond a chunk (one of 2,500), 256 to a workgroup with a
    last partial one; the solution's residual by a CPU product at the stop
    tolerance (1e-10, within ten times it for the recursive residual), and x1
    from x2 within the rounding of sums of at most 2,500 terms."""
    rng = np.random.default_rng(17)
    m = 2500
    lens = np.concatenate(([1024, 1, 1023, 2500, 1, 2, 3, 1025], rng.integers(1, 12, 700), [m - 1, 4]))
    cols = [np.sort(rng.choice(m, k, replace=False)) for k in lens] + [np.array([i]) for i in range(m)]
    vals = [rng.standard_normal(len(c)) / np.sqrt(len(c)) for c in cols[:len(lens)]] + [np.ones(1)] * m
    inst = Instance(m, len(cols), np.concatenate(([0], np.cumsum([len(c) for c in cols]))).astype(np.int64),
                    np.concatenate(cols).astype(np.int32), np.concatenate(vals), np.ones(m), np.ones(len(cols)))
    assert inst.n % 256 != 0
    A = _csc(inst)
    d = np.exp(rng.uniform(-1, 1, inst.n) * np.log(10.0))
    b1, b2 = rng.standard_normal(inst.n), rng.standard_normal(m)
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=20, pcg_tol=1e-10, pcg_max_iter=5000)
    be.construct(inst)
    be.renew(d)
    x1, x2 = be.solve(d, b1, b2)
    be.destruct()
    r = A @ (b1 / d) - b2
    rel = np.linalg.norm(r - A @ ((A.T @ x2) / d)) / np.linalg.norm(r)
    bs = np.linalg.norm(x1 - (b1 - A.T @ x2) / d) / np.linalg.norm(x1)
    _flush(f"column chunks: relative residual {rel:.2e}, back-substitution {bs:.1e}")
    assert rel <= 1e-9 and bs <= 1e-12


def test_pcg_cap_reports_noconv():
    """A PCG solve stopped by pcg_max_iter short of pcg_tol returns
    HELP_ERR_NOCONV (with its last iterate and the residual in the stats),
    and the HSD drivers stop with STALLED / HELP_STALL_BACKEND instead of
    iterating on an unconverged direction."""
    from help_amd.backend import HelpError
    from help_amd.hsd import GpuBackend, solve_lp
    inst = instances.random_lp(300, 600, 4, seed=41)
    rng = np.random.default_rng(3)
    d = np.exp(rng.uniform(-3, 3, inst.n) * np.log(10.0))
    b1, b2 = rng.standard_normal(inst.n), rng.standard_normal(inst.m)
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=10, pcg_max_iter=2)
    be.construct(inst)
    be.renew(d)
    with pytest.raises(HelpError) as ei:
        be.solve(d, b1, b2)
    assert ei.value.code == L.HELP_ERR_NOCONV
    assert be.solve_stats.pcg_iters == 2 and be.solve_stats.rel_residual > 1e-10
    be.destruct()
    for device in (True, False):
        gb = GpuBackend(mode=L.MODE_PCG, pcg_k=10, pcg_max_iter=2)
        try:
            res, _ = solve_lp(inst, gb.table, device=device)
        finally:
            gb.close()
        _flush(f"  hsd device={device}: status {res.status} stall {res.stall_reason} "
               f"backend_error {res.backend_error} iterations {res.iterations}")
        assert res.status == 1 and res.stall_reason == 3 and res.backend_error == L.HELP_ERR_NOCONV


def test_pcg_full_size_zipf_residuals():
    """The Zipf LP at its full size (m=10^6, n=4*10^6, nnz=1.9*10^7) in PCG
    mode with K=500: the backend's solution of A D^-1 A^T x2 = r (the PCG
    mode's operator has no diagonal shift, as PCG.cpp's), r = A D^-1 b1 - b2,
    checked by an independent CPU product (scipy) against the stop tolerance
    (the recursive CG residual and the true one differ by rounding), at d = 1
    and at a log-uniform d over +-1 decade, plus x1 = D^-1 (b1 - A^T x2).  The
    oracle's partial Cholesky takes too long at this size; its parity is
    pinned on the smaller instances above."""
    inst = instances.by_config(3)
    A = inst.to_scipy().tocsr()
    At = A.T.tocsr()
    rng = np.random.default_rng(5)
    be = LinearEquation(mode=L.MODE_PCG, pcg_k=500, pcg_tol=1e-10, pcg_max_iter=5000)
    be.construct(inst)
    for name, d in (("d=1", np.ones(inst.n)), ("d log-uniform +-1", np.exp(rng.uniform(-1, 1, inst.n) * np.log(10.0)))):
        b1, b2 = rng.standard_normal(inst.n), rng.standard_normal(inst.m)
        be.renew(d)
        x1, x2 = be.solve(d, b1, b2)
        r = A @ (b1 / d) - b2
        res = r - A @ ((At @ x2) / d)
        rel = np.linalg.norm(res) / np.linalg.norm(r)
        bs = np.linalg.norm(x1 - (b1 - At @ x2) / d) / np.linalg.norm(x1)
        _flush(f"zipf m={inst.m} {name}: {be.solve_stats.pcg_iters} CG iterations, relative residual {rel:.2e} "
               f"(library {be.solve_stats.rel_residual:.2e}), x1 back-substitution {bs:.1e}")
        assert rel <= 1e-9
        assert bs <= 1e-12
    be.destruct()
