"""GPU parity of the CG solver (src/cgd.c:40-129) through the C ABI.

Bar: the same stopping rule as the reference (sqrt(r.r) <= error), the same
relative residual reached and an iteration count within +-2 of the oracle
at one thread; at full size, size-independent properties (true residual,
determinism).
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def true_rel(oracle, rp, ri, rv, x, b):
    r = b - oracle.spmv(rp, ri, rv, x)
    return np.linalg.norm(r) / np.linalg.norm(b)


def test_stop_by_tolerance_and_by_cap_give_the_same_x(gb):
    # the iteration that meets the tolerance still adds alpha p to x: capping
    # the solve at that iteration count gives the same bits
    rp, ri, rv = gb.laplacian(3, 30)
    b = gb.uniform(8, rp.size - 1)
    err = 1e-9 * np.linalg.norm(b)
    x1, i1 = gb.cgd(rp, ri, rv, b, err)
    assert i1.status == 1
    x2, i2 = gb.cgd(rp, ri, rv, b, 0.0, niter=int(i1.niter))
    assert i2.status == 2 and i2.niter == i1.niter
    assert np.array_equal(x1, x2)
    x3, _ = gb.cgd(rp, ri, rv, b, 0.0, niter=int(i1.niter) - 1)
    assert not np.array_equal(x1, x3)


def test_config1_cg_vs_oracle(gb, oracle):
    rp, ri, rv = gb.laplacian(2, 256)
    b = gb.uniform(0, 65536)
    err = 1e-8 * np.linalg.norm(b)
    x, info = gb.cgd(rp, ri, rv, b, err, niter=2000)
    xr, it, rmse, _ = oracle.cgd(rp, ri, rv, b, err, niter=2000)
    assert info.converged == 1 and info.status == 1
    assert abs(int(info.niter) - it) <= 2, (info.niter, it)
    assert info.rnorm <= err and rmse <= err
    assert true_rel(oracle, rp, ri, rv, x, b) < 2e-8
    assert np.max(np.abs(x - xr)) <= 1e-6 * np.max(np.abs(xr))


def test_3d_laplacian_cg_vs_oracle(gb, oracle):
    rp, ri, rv = gb.laplacian(3, 40)
    n = rp.size - 1
    b = gb.uniform(1, n)
    err = 1e-10 * np.linalg.norm(b)
    x, info = gb.cgd(rp, ri, rv, b, err)
    xr, it, rmse, _ = oracle.cgd(rp, ri, rv, b, err)
    assert info.converged == 1
    assert abs(int(info.niter) - it) <= 2, (info.niter, it)
    assert true_rel(oracle, rp, ri, rv, x, b) < 5e-10


def test_first_iterations_track_oracle(gb, oracle):
    # with the reference's update order and separately rounded products, the
    # residual history differs only through the dot-product summation order
    rp, ri, rv = gb.laplacian(2, 64)
    b = gb.uniform(3, 4096)
    for k in (1, 2, 5, 20):
        x, info = gb.cgd(rp, ri, rv, b, 0.0, niter=k)
        xr, it, rmse, _ = oracle.cgd(rp, ri, rv, b, 0.0, niter=k)
        assert info.niter == k and info.status == 2 and it == k
        assert abs(info.rnorm - rmse) <= 1e-12 * np.linalg.norm(b)
        assert np.max(np.abs(x - xr)) <= 1e-12 * np.max(np.abs(xr))


def band_spd(n, half, seed):
    """A symmetric, strictly dominant band matrix; each row's off-diagonals at
    distances 1 .. half, a third of them missing."""
    rng = np.random.default_rng(seed)
    ii, jj, vv = [], [], []
    for d in range(1, min(half, n - 1) + 1):
        keep = np.nonzero(rng.random(n - d) < 2 / 3)[0]
        v = rng.uniform(-1, 0, keep.size)
        ii += [keep, keep + d]
        jj += [keep + d, keep]
        vv += [v, v]
    ii = np.concatenate(ii + [np.arange(n)]) if ii else np.arange(n)
    off = np.bincount(ii[:ii.size - n], weights=-np.concatenate(vv) if vv else None, minlength=n)
    jj = np.concatenate(jj + [np.arange(n)])
    vv = np.concatenate(vv + [1.05 * off + 0.1])
    order = np.lexsort((jj, ii))
    rp = np.concatenate([[0], np.cumsum(np.bincount(ii, minlength=n))]).astype(np.uint32)
    return rp, jj[order].astype(np.uint32), vv[order]


def solve_both(gb, monkeypatch, rp, ri, rv, b, tol, niter=0):
    """One launch for the run of iterations, and (its waits given up at once)
    one launch per step."""
    N = gb.Matrix(rp, ri, rv)
    x1, i1 = N.cgd(b, tol, gb.TOL_RELATIVE, niter=niter)
    workgroups = N.kernels()["cg_workgroups"]
    monkeypatch.setenv("GOOSEBERRY_CG_SPINS", "0")
    M = gb.Matrix(rp, ri, rv)
    x2, i2 = M.cgd(b, tol, gb.TOL_RELATIVE, niter=niter)
    x3, i3 = M.cgd(b, tol, gb.TOL_RELATIVE, niter=niter)  # stays with that
    monkeypatch.delenv("GOOSEBERRY_CG_SPINS")
    assert i3.niter == i2.niter and np.array_equal(x2, x3)
    # (a workgroup alone waits for nobody)
    assert M.kernels()["cg_workgroups"] == (1 if workgroups == 1 else 0)
    return (x1, i1), (x2, i2)


# rows around the sizes of the one-launch solve: one workgroup (512 rows), 64
# workgroups of 512 to 2048 rows, 128 and 256 workgroups, and past them; and, on
# both sides with several launches, rows of over 64 entries and more entries than
# LDS holds (SHAPES below says which is which)
@pytest.mark.parametrize("n,half", [
    (1, 0), (2, 1), (64, 3), (511, 2), (512, 2), (513, 2), (1025, 40), (5000, 44), (32768, 2),
    (32769, 2), (40000, 20), (65600, 2), (131072, 2), (131073, 2), (262145, 2), (524289, 2)])
def test_small_systems_in_one_launch(gb, oracle, monkeypatch, n, half):
    print("cg one launch", n, half, flush=True)
    rp, ri, rv = band_spd(n, half, n)
    b = gb.uniform(n, n)
    (x1, i1), (x2, i2) = solve_both(gb, monkeypatch, rp, ri, rv, b, 1e-11)
    xr, it, rmse, _ = oracle.cgd(rp, ri, rv, b, 1e-11 * np.linalg.norm(b))
    for x, i in ((x1, i1), (x2, i2)):
        assert i.status == 1 and abs(int(i.niter) - it) <= 2
        # residuals of 1e-11 and a condition number below 43 (the rows'
        # dominance): x within 43 x 2e-11 of the oracle's
        assert np.linalg.norm(x - xr) <= 1e-9 * np.linalg.norm(xr)
        assert true_rel(oracle, rp, ri, rv, x, b) <= 1.05e-11
    # the first iterations differ only by the order of the dot products
    if n > 64:
        (y1, j1), (y2, j2) = solve_both(gb, monkeypatch, rp, ri, rv, b, 0.0, niter=3)
        assert j1.niter == j2.niter == 3 and j1.status == j2.status == 2
        assert np.max(np.abs(y1 - y2)) <= 1e-13 * np.max(np.abs(y2))


def test_one_launch_scattered_columns_and_repeats(gb, oracle):
    # random columns all over the system, rows of very different lengths; a
    # matrix solved twice (and with another x) gives the same bits
    M = gb.generate_sdd(20000, 7, 2, 25)
    rp, ri, rv = M.download()
    b = gb.uniform(2, 20000)
    x, info = M.cgd(b, 1e-10, gb.TOL_RELATIVE)
    x2, info2 = M.cgd(b, 1e-10, gb.TOL_RELATIVE)
    assert info.status == 1 and info2.niter == info.niter and np.array_equal(x, x2)
    _, it, _, _ = oracle.cgd(rp, ri, rv, b, 1e-10 * np.linalg.norm(b))
    assert abs(int(info.niter) - it) <= 2
    assert true_rel(oracle, rp, ri, rv, x, b) <= 1.05e-10


# (workgroups, rows each) of the one-launch solve on 256 CUs; (0, 0): rows over
# 64 entries, entries that fit no choice of workgroups, more than 2048 rows a
# workgroup
SHAPES = [
    (1, 0, 1, 64), (512, 2, 1, 512), (513, 2, 2, 320), (1025, 20, 3, 384), (10000, 15, 20, 512),
    (20000, 22, 53, 384), (32768, 2, 64, 512), (32769, 2, 57, 576), (40000, 18, 90, 448),
    (65600, 2, 61, 1088), (80000, 15, 157, 512), (131072, 2, 64, 2048), (131073, 2, 121, 1088),
    (262145, 2, 241, 1088), (400000, 3, 250, 1600), (524288, 1, 256, 2048),
    (1025, 40, 0, 0), (40000, 20, 0, 0), (524289, 2, 0, 0)]


@pytest.mark.parametrize("n,half,workgroups,rows", SHAPES)
def test_one_launch_shapes(gb, oracle, n, half, workgroups, rows):
    print("cg shape", n, half, flush=True)
    rp, ri, rv = band_spd(n, half, n)
    M = gb.Matrix(rp, ri, rv)
    b = gb.uniform(n, n)
    x, info = M.cgd(b, 1e-10, gb.TOL_RELATIVE)
    want = {"cg_workgroups": workgroups, "cg_rows": rows}
    assert {k: M.kernels()[k] for k in want} == want
    assert info.status == 1 and true_rel(oracle, rp, ri, rv, x, b) <= 1.05e-10
    # the allocation-free entry point takes the same kernels, also first
    N = gb.Matrix(rp, ri, rv)
    db, dx, i2 = gb.DeviceArray.from_host(b), gb.DeviceArray(n), gb.CgdInfo()
    assert gb.lib().gooseberry_matrix_cgd_noalloc(N.h, db.ptr, dx.ptr, 1e-10, gb.TOL_RELATIVE, 0,
                                                 ctypes.byref(i2)) == gb.SUCCESS
    assert {k: N.kernels()[k] for k in want} == want
    assert i2.niter == info.niter and np.array_equal(dx.numpy(), x)


def test_one_launch_choice_follows_the_plan_and_reports_failures(gb):
    rp, ri, rv = gb.laplacian(2, 100)
    M = gb.Matrix(rp, ri, rv)
    b = gb.uniform(1, M.nrows)
    # the first launch of a plan's first solve counts its entries
    gb.inject_fault(gb.FAULT_LAUNCH, 0)
    try:
        with pytest.raises(gb.GooseberryError) as e:
            M.cgd(b, 1e-8, gb.TOL_RELATIVE)
    finally:
        gb.inject_fault(gb.FAULT_LAUNCH, -1)
    assert e.value.name == "DEVICE" and M.kernels()["cg_workgroups"] == 0
    x, _ = M.cgd(b, 1e-8, gb.TOL_RELATIVE)
    assert M.kernels()["cg_workgroups"] == 20
    for plan in ({"csplit": 2}, {"xtile": 1024}, {"short_max": 4}):
        M.replan(plan)
        y, info = M.cgd(b, 1e-8, gb.TOL_RELATIVE)
        assert info.status == 1 and M.kernels()["cg_workgroups"] == 0
        assert np.linalg.norm(x - y) <= 1e-5 * np.linalg.norm(x)
    M.replan(None)
    y, _ = M.cgd(b, 1e-8, gb.TOL_RELATIVE)
    assert M.kernels()["cg_workgroups"] == 20 and np.array_equal(x, y)


# A wait given up in one launch, by exchange: the first one (workgroups may
# still be starting), one amid the run, and the last of the run, after which
# the other workgroups have the solve's end (iteration cap, convergence) and
# only the one that gave up lacks its rows of x
@pytest.mark.parametrize("end", ["cap", "converged"])
@pytest.mark.parametrize("exchange", ["first", "second", "amid", "last"])
@pytest.mark.parametrize("n,half", [(1025, 2), (40000, 2), (262144, 2), (20000, 22)])
def test_wait_given_up_is_never_a_result(gb, oracle, monkeypatch, n, half, exchange, end):
    print("cg wait given up", n, half, exchange, end, flush=True)
    # waits that do run out afterwards end after some ten milliseconds
    monkeypatch.setenv("GOOSEBERRY_CG_SPINS", "20000")
    rp, ri, rv = band_spd(n, half, n)
    b = gb.uniform(n, n)
    niter = 3 if end == "cap" else 0
    tol = 0.0 if end == "cap" else 1e-10
    x1, i1 = gb.Matrix(rp, ri, rv).cgd(b, tol, gb.TOL_RELATIVE, niter=niter)
    M = gb.Matrix(rp, ri, rv)
    last = 2 * int(i1.niter) - 1
    at = {"first": 0, "second": 1, "amid": last // 2, "last": last}[exchange]
    gb.inject_fault(gb.FAULT_CG_WAIT, at)
    try:
        x2, i2 = M.cgd(b, tol, gb.TOL_RELATIVE, niter=niter)
    finally:
        gb.inject_fault(gb.FAULT_CG_WAIT, -1)
    assert i2.status == i1.status == (2 if end == "cap" else 1)
    assert abs(int(i2.niter) - int(i1.niter)) <= 2
    if end == "cap":
        # three iterations differ only by the order of the dot products
        assert np.max(np.abs(x1 - x2)) <= 1e-13 * np.max(np.abs(x1))
    else:
        assert true_rel(oracle, rp, ri, rv, x2, b) <= 1.05e-10
    # the matrix stays with the other kernels, and gives what they gave
    x3, i3 = M.cgd(b, tol, gb.TOL_RELATIVE, niter=niter)
    assert i3.niter == i2.niter and np.array_equal(x2, x3)


@pytest.mark.parametrize("first", ["cgd", "noalloc"])
def test_a_wait_given_up_is_remembered_by_the_matrix(gb, monkeypatch, first):
    # after one entry point gave up a wait, neither runs in one launch again (the
    # armed fault is not taken), and both give the same bits; a new plan may
    monkeypatch.setenv("GOOSEBERRY_CG_SPINS", "20000")
    rp, ri, rv = gb.laplacian(2, 150)
    M = gb.Matrix(rp, ri, rv)
    b = gb.uniform(9, M.nrows)
    db, dx = gb.DeviceArray.from_host(b), gb.DeviceArray(b.size)

    def solve(entry):
        info = gb.CgdInfo()
        f = getattr(gb.lib(), "gooseberry_matrix_cgd" + ("" if entry == "cgd" else "_noalloc"))
        log = (None,) if entry == "cgd" else ()
        assert f(M.h, db.ptr, dx.ptr, 1e-9, gb.TOL_RELATIVE, 0, *log,
                 ctypes.byref(info)) == gb.SUCCESS
        return dx.numpy().tobytes(), int(info.niter), info.rnorm

    other = "noalloc" if first == "cgd" else "cgd"
    one = solve(other)
    assert solve(first) == one and M.kernels()["cg_workgroups"] == 44
    try:
        gb.inject_fault(gb.FAULT_CG_WAIT, 2)
        several = solve(first)
        assert M.kernels()["cg_workgroups"] == 0 and several != one
        gb.inject_fault(gb.FAULT_CG_WAIT, 0)
        assert solve(other) == several and solve(first) == several
        M.replan(None)
        assert M.kernels()["cg_workgroups"] == 0
        assert solve(other) == several and M.kernels()["cg_workgroups"] == 0  # takes the fault
        M.replan(None)
        assert solve(other) == one and solve(first) == one
        assert M.kernels()["cg_workgroups"] == 44
    finally:
        gb.inject_fault(gb.FAULT_CG_WAIT, -1)


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("exchange", [None, 0, 5, "last"])
def test_solve_in_the_place_of_b(gb, monkeypatch, exchange, noalloc):
    # x written over b: the same bits as beside it, also when a wait was given
    # up and the solve started again
    monkeypatch.setenv("GOOSEBERRY_CG_SPINS", "20000")
    rp, ri, rv = gb.laplacian(2, 200)
    b = gb.uniform(5, rp.size - 1)
    db, dx = gb.DeviceArray.from_host(b), gb.DeviceArray(b.size)

    def solve(to):
        M = gb.Matrix(rp, ri, rv)  # a matrix of its own: none that gave up before
        info = gb.CgdInfo()
        f = gb.lib().gooseberry_matrix_cgd_noalloc if noalloc else gb.lib().gooseberry_matrix_cgd
        log = () if noalloc else (None,)
        assert f(M.h, db.ptr, to.ptr, 1e-9, gb.TOL_RELATIVE, 0, *log,
                 ctypes.byref(info)) == gb.SUCCESS
        return info

    at = exchange if exchange != "last" else 2 * int(solve(dx).niter) - 1
    got = []
    for to in (dx, db):
        if at is not None:
            gb.inject_fault(gb.FAULT_CG_WAIT, at)
        try:
            info = solve(to)
        finally:
            gb.inject_fault(gb.FAULT_CG_WAIT, -1)
        got.append((to.numpy().tobytes(), int(info.niter), info.status, info.rnorm))
    assert got[0] == got[1] and got[0][2] == 1


@pytest.mark.parametrize("kind", ["zero_b", "nan_b", "zero_matrix", "indefinite"])
def test_one_launch_stops_as_the_steps_do(gb, monkeypatch, kind):
    rp, ri, rv = gb.laplacian(2, 40)
    b = gb.uniform(4, 1600)
    if kind == "zero_b":
        b = np.zeros(1600)
    elif kind == "nan_b":
        b[700] = np.nan
    elif kind == "zero_matrix":
        rv = np.zeros_like(rv)
    else:
        rv = np.where(np.arange(rv.size) % 2 == 0, rv, -rv)
    got = []
    for spins in (None, "0"):
        if spins:
            monkeypatch.setenv("GOOSEBERRY_CG_SPINS", spins)
        M = gb.Matrix(rp, ri, rv)
        x, info = M.cgd(b, 1e-10, gb.TOL_RELATIVE, niter=12)
        got.append((int(info.status), int(info.niter)))
        if kind in ("zero_b", "zero_matrix"):
            assert np.array_equal(x, np.zeros(1600))
    assert got[0] == got[1], got


def test_config2_full_size_true_residual(gb, oracle):
    rp, ri, rv = gb.laplacian(3, 160)
    n = rp.size - 1
    b = gb.uniform(1, n)
    M = gb.Matrix(rp, ri, rv)
    x, info = M.cgd(b, 1e-10, gb.TOL_RELATIVE)
    assert info.converged == 1
    assert info.rnorm <= 1e-10 * info.bnorm
    assert 200 < info.niter < 2000
    r = b - M.spmv(x)
    assert np.linalg.norm(r) / np.linalg.norm(b) < 1e-9
    # deterministic: fixed reduction order
    x2, info2 = M.cgd(b, 1e-10, gb.TOL_RELATIVE)
    assert info2.niter == info.niter and np.array_equal(x, x2)


def test_config2_cg_vs_oracle(gb, oracle):
    # the headline system at full size: 160^3 Laplacian, b from seed 1,
    # relative residual 1e-10.  The oracle runs the reference's loop on 16
    # threads (one thread would take minutes); its dot products then add in
    # a thread-count dependent order, which the +-2 bar allows.
    rp, ri, rv = gb.laplacian(3, 160)
    n = rp.size - 1
    b = gb.uniform(1, n, stream=1)
    err = 1e-10 * float(np.linalg.norm(b))
    M = gb.Matrix(rp, ri, rv)
    x, info = M.cgd(b, err, gb.TOL_ABSOLUTE)
    oracle.set_threads(16)
    try:
        xr, it, rmse, _ = oracle.cgd(rp, ri, rv, b, err)
    finally:
        oracle.set_threads(1)
    assert info.converged == 1 and info.status == 1
    assert abs(int(info.niter) - it) <= 2, (info.niter, it)
    # the same stopping rule met on both sides, and the same true residual
    assert info.rnorm <= err and rmse <= err
    rel = true_rel(oracle, rp, ri, rv, x, b)
    rel_ref = true_rel(oracle, rp, ri, rv, xr, b)
    assert rel < 1.5e-10 and rel_ref < 1.5e-10
    assert abs(rel - rel_ref) <= 0.5 * max(rel, rel_ref)
    assert np.max(np.abs(x - xr)) <= 1e-6 * np.max(np.abs(xr))


def test_irregular_spd_vs_oracle(gb, oracle):
    # symmetric, diagonally dominant, rows of very different lengths
    rng = np.random.default_rng(4)
    n = 6000
    import scipy.sparse as sp
    L = sp.random(n, n, density=0.0015, random_state=5, format="csr")
    L.data = -rng.uniform(0, 1, L.nnz)
    hub = sp.csr_matrix((-rng.uniform(0, 1, 3000), (np.zeros(3000, int),
                                                    rng.choice(n, 3000, replace=False))),
                        shape=(n, n))
    A = L + L.T + hub + hub.T
    A = sp.csr_matrix(A)
    A.setdiag(0)
    A.eliminate_zeros()
    d = 1.01 * np.asarray(abs(A).sum(axis=1)).ravel() + 1e-3
    A = sp.csr_matrix(A + sp.diags(d))
    A.sort_indices()
    b = rng.uniform(-1, 1, n)
    err = 1e-10 * np.linalg.norm(b)
    x, info = gb.cgd(A.indptr, A.indices, A.data, b, err)
    xr, it, rmse, _ = oracle.cgd(A.indptr, A.indices, A.data, b, err)
    assert info.converged == 1 and abs(int(info.niter) - it) <= 2
    assert np.linalg.norm(b - A @ x) / np.linalg.norm(b) < 1e-9


def test_zero_rhs_and_caps(gb):
    rp, ri, rv = gb.laplacian(2, 32)
    n = rp.size - 1
    x, info = gb.cgd(rp, ri, rv, np.zeros(n), 1e-8)
    assert info.niter == 0 and info.converged == 1 and np.all(x == 0)
    x, info = gb.cgd(rp, ri, rv, gb.uniform(5, n), 0.0, niter=7)
    assert info.niter == 7 and info.status == 2 and info.converged == 0


def test_nonsquare_rejected(gb):
    with pytest.raises(gb.GooseberryError) as e:
        M = gb.Matrix(np.array([0, 1, 2], np.uint32), np.array([0, 2], np.uint32),
                      np.ones(2), ncols=3)
        M.cgd(np.ones(2), 1e-8)
    assert e.value.name == "INVALIDINPUT"


def test_indefinite_breakdown_reported(gb):
    # p.Ap == 0 at the first step: the reference would produce NaNs; the
    # build stops and reports a breakdown
    rp = np.array([0, 1, 2], np.uint32)
    ri = np.array([0, 1], np.uint32)
    rv = np.array([1.0, -1.0])
    x, info = gb.cgd(rp, ri, rv, np.array([1.0, 1.0]), 1e-12)
    assert info.status == 3
