"""Scalar CG solves that run in one launch with the vectors on chip,
against the launch-per-step solver on the same handle (`set_on_chip(False)`) and the
oracle: same status, iteration counts within +-2 % (+-1 below
50), solutions within 1e-6."""
import ctypes

import numpy as np
import pytest

import oracle
from monolis_amd import api, workloads as W
from monolis_amd.matrix import Matrix

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init(hip):
    oracle.set_threads(1)
    yield


def _matrix(n, far, wide, seed):
    """Diagonally dominant rows of uneven length (1 entry in every fifth row, more than 8 with `wide`),
    some coupling `far` rows apart."""
    rng = np.random.default_rng(seed)
    reps = 4 if wide else 1
    i = rng.integers(0, n, reps * n)
    d = np.where(rng.uniform(size=reps * n) < 0.3, far, rng.integers(1, 30, reps * n))
    keep = (i + d < n) & (i % 5 != 0) & ((i + d) % 5 != 0)
    if not wide:   # at most 3 entries on each side of the diagonal
        _, first = np.unique(i, return_index=True)
        one = np.zeros(reps * n, bool)
        one[first] = True
        keep &= one & (rng.uniform(size=reps * n) < 0.9)
    key = np.unique(i[keep] * n + i[keep] + d[keep])
    i, j = key // n, key % n
    v = -rng.uniform(0.1, 1.0, len(i))
    rows, cols = np.concatenate([i, j, np.arange(n)]), np.concatenate([j, i, np.arange(n)])
    off = np.bincount(np.concatenate([i, j]), weights=np.abs(np.concatenate([v, v])), minlength=n)
    vals = np.concatenate([v, v, off + 0.05])
    order = np.lexsort((cols, rows))
    index = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int32)
    return Matrix(n, n, 1, index, (cols[order] + 1).astype(np.int32), vals[order]).ensure_dof_index()


def _prm(precond=1, tol=1e-8, init_x=True, max_iter=3000):
    prm = api.Prm().quiet()
    prm.Iarray[api.MONOLIS_PRM_I_PRECOND] = precond
    prm.Iarray[api.MONOLIS_PRM_I_MAX_ITER] = max_iter
    prm.Iarray[api.MONOLIS_PRM_I_IS_INIT_X] = int(init_x)
    prm.Rarray[api.MONOLIS_PRM_R_TOL] = tol
    return prm


def _near(a, b):
    return abs(a - b) <= max(1, int(0.02 * max(a, b)))


def _both(mat, b, precond=1, x0=None, **kw):
    """(x, iterations, residual history) on chip and step by step."""
    dm = api.DeviceMatrix(mat)
    db, dx = api.DeviceBuffer.from_numpy(b), api.DeviceBuffer(mat.n)
    out = []
    for steps in (False, True):
        if x0 is not None:
            dx.upload(x0)
        dm.set_on_chip(not steps)
        prm = _prm(precond, init_x=x0 is None, **kw)
        h = dm.solve(db, dx, prm, hist_len=3001)
        it = int(prm.Iarray[api.MONOLIS_PRM_I_CUR_ITER])
        out.append((dx.numpy(), it, h, int(prm.Iarray[api.MONOLIS_PRM_I_IERR]), prm.Rarray[api.MONOLIS_PRM_R_CUR_RESID]))
    assert dm.on_chip_solves() == (1, 0)
    (x, it, h, st, res), (xs, its, hs, sts, ress) = out
    assert st == sts and _near(it, its), (it, its)
    assert np.linalg.norm(x - xs) <= 1e-6 * np.linalg.norm(xs)
    assert h[it] == res and np.all(h[1:it + 1] >= 0) and not h[it + 1:].any()
    k = min(5, it, its)
    assert np.allclose(h[1:k], hs[1:k], rtol=1e-6)
    return x, it


# one row, a whole and a partial slice, one member and the first team, four and eight rows per thread, rows
# of more and fewer than eight entries
@pytest.mark.parametrize("precond", [1, 0])
@pytest.mark.parametrize("n, far, wide", [(1, 1, False), (64, 5, False), (1000, 333, True), (2048, 700, False),
                                          (2049, 700, True), (70001, 9000, False), (70001, 2000, True)])
def test_on_chip_matches_steps_and_oracle(n, far, wide, precond):
    mat = _matrix(n, far, wide, seed=n + wide)
    b = oracle.matvec(mat, W.uniform_vector(n, seed=2))
    x, it = _both(mat, b, precond)
    xo, st, I, R = oracle.solve(mat, b, precond=precond, max_iter=3000)
    assert st == 0 and _near(it, int(I[4]))
    assert np.linalg.norm(x - xo) <= 1e-6 * np.linalg.norm(xo)


def test_on_chip_past_the_replacement_and_from_a_start_vector():
    # 64^3 rows take the largest team four rows per thread, 72^3 eight, with x in LDS
    for e in (64, 72):
        mat = W.poisson7(e)
        b = W.uniform_vector(mat.n, seed=3)
        x, it = _both(mat, b, tol=1e-11)
        assert it > 200
        # both end within tol * ||r0|| * cond of the solution: 1.8e-6 apart at 1e-8 from this start, 1e-8 here
        _both(mat, b, x0=W.uniform_vector(mat.n, seed=4), tol=1e-10)


def test_on_chip_zero_rhs_limit_and_repeat():
    mat = _matrix(5000, 600, False, 9)
    dm = api.DeviceMatrix(mat)
    db, dx = api.DeviceBuffer.from_numpy(np.zeros(5000)), api.DeviceBuffer.from_numpy(np.ones(5000))
    dm.solve(db, dx, _prm())
    assert not dx.numpy().any()
    b = W.uniform_vector(5000, seed=1)
    db.upload(b)
    prm = _prm(max_iter=7)
    dm.solve(db, dx, prm)
    assert prm.Iarray[api.MONOLIS_PRM_I_IERR] == 1 and prm.Iarray[api.MONOLIS_PRM_I_CUR_ITER] == 7
    xo, st, I, R = oracle.solve(mat, b, max_iter=7)
    assert np.linalg.norm(dx.numpy() - xo) <= 1e-6 * np.linalg.norm(xo)
    dm.solve(db, dx, _prm())
    x = dx.numpy()
    for _ in range(3):
        dm.solve(db, dx, _prm())
        assert np.array_equal(x, dx.numpy())
    # new values on the same pattern
    dm.set_values(mat.A * 2.0)
    dm.solve(db, dx, _prm())
    mat2 = Matrix(5000, 5000, 1, mat.index, mat.item, mat.A * 2.0).ensure_dof_index()
    xo, st, I, R = oracle.solve(mat2, b)
    assert np.linalg.norm(dx.numpy() - xo) <= 1e-6 * np.linalg.norm(xo)


def test_solver_tuning_times_the_launches_that_the_variant_is_of():
    """The SpMV variants are those of the launch-per-step solver: tuning on a system that also fits on chip
    takes that solver, with the unpreconditioned form as well; later solves run on chip again."""
    mat = _matrix(3000, 500, False, 12)
    dm = api.DeviceMatrix(mat)
    for precond in (1, 0):
        t = dm.autotune_solver(fp32=False, precond=precond, iters=6, reps=1)
        assert dm.on_chip_solves() == (0, 0)
        assert all(v > 0 for v in t["ms_per_iter"]) and t["ms_per_iter"][t["best"]] == min(t["ms_per_iter"])
    db, dx = api.DeviceBuffer.from_numpy(W.uniform_vector(3000, seed=1)), api.DeviceBuffer(3000)
    dm.solve(db, dx, _prm())
    assert dm.on_chip_solves() == (1, 0)


def test_on_chip_handles_of_one_kernel_and_different_lds():
    """Kernels are shared by the handles: an older handle that takes much LDS (members with a long halo) is
    solved again after a younger one with little has been built, singly and as a batch."""
    def handle(mat):
        db, dx = api.DeviceBuffer.from_numpy(W.uniform_vector(mat.n, seed=5)), api.DeviceBuffer(mat.n)
        return api.DeviceMatrix(mat), db, dx

    # four rows per thread with the matrix in registers; eight; 26 rows per thread
    for big, small in ((_matrix(70001, 9000, False, 1), _matrix(64, 5, False, 2)),
                       (W.poisson7(72), W.poisson7(65)),
                       (_matrix(70001, 9000, True, 1), _matrix(2049, 9, True, 2))):
        a, b = handle(big), handle(small)
        a[0].solve(a[1], a[2], _prm())
        x = a[2].numpy()
        b[0].solve(b[1], b[2], _prm())
        a[2].upload(np.zeros(big.n))
        a[0].solve(a[1], a[2], _prm())
        assert a[0].on_chip_solves() == (2, 0) and b[0].on_chip_solves() == (1, 0)
        assert np.array_equal(x, a[2].numpy())
    out = []
    for edges in ([40, 40, 38], [8, 9]):
        mat, sys_row = W.poisson_batch(edges=edges)
        B = api.DeviceBatch(mat, sys_row)
        assert B.schedule(15)["split"] == 1
        db, dx = api.DeviceBuffer.from_numpy(W.uniform_vector(mat.n, seed=6)), api.DeviceBuffer(mat.n)
        B.solve(db, dx, _prm())
        out.append((B, db, dx, dx.numpy()))
    B, db, dx, x = out[0]
    dx.upload(np.zeros(len(x)))
    B.solve(db, dx, _prm())
    assert np.array_equal(x, dx.numpy())


@pytest.mark.parametrize("init_x", [True, False])
def test_on_chip_wait_that_gives_up_is_redone_by_steps(init_x):
    """With wait limit 0 a team gives up at its start: the solve is redone launch by launch from the same start
    vector, the next ones take that solver at once, and setting the limit again brings the team back."""
    mat = W.poisson7(32)
    b, x0 = W.uniform_vector(mat.n, seed=3), W.uniform_vector(mat.n, seed=4)
    I, R = oracle.default_arrays(max_iter=12)
    I[10] = int(init_x)
    xo, st, I, R = oracle.solve(mat, b, x0=x0, Iarray=I, Rarray=R)
    dm = api.DeviceMatrix(mat)
    db, dx = api.DeviceBuffer.from_numpy(b), api.DeviceBuffer(mat.n)

    def check(solves, gave_up):
        dx.upload(x0)
        prm = _prm(max_iter=12, init_x=init_x)
        h = dm.solve(db, dx, prm, hist_len=20)
        assert dm.on_chip_solves() == (solves, gave_up)
        assert int(prm.Iarray[api.MONOLIS_PRM_I_IERR]) == st and int(prm.Iarray[api.MONOLIS_PRM_I_CUR_ITER]) == 12
        assert h[12] == prm.Rarray[api.MONOLIS_PRM_R_CUR_RESID] and np.linalg.norm(dx.numpy() - xo) <= 1e-9 * np.linalg.norm(xo)

    check(1, 0)
    dm.set_on_chip(True, 0.0)
    check(1, 1)
    check(1, 1)
    dm.set_on_chip(True, 5.0)
    check(2, 1)
    dm.set_on_chip(False)
    check(2, 1)
    with pytest.raises(RuntimeError):
        dm.set_on_chip(True, -1.0)


def test_on_chip_settings_reach_the_transpose():
    mat = _matrix(3000, 500, False, 12)      # symmetric: the solution of A^T x = b is that of A x = b
    dm = api.DeviceMatrix(mat)
    db, dx = api.DeviceBuffer.from_numpy(W.uniform_vector(3000, seed=1)), api.DeviceBuffer(3000)
    dm.set_on_chip(False)
    dm.solve_transpose(db, dx, _prm())
    assert dm.on_chip_solves() == (0, 0)
    xs = dx.numpy()
    dm.set_on_chip(True, 0.0)
    dm.solve_transpose(db, dx, _prm())
    assert dm.on_chip_solves() == (0, 1) and np.array_equal(xs, dx.numpy())
    dm.set_on_chip(True)
    dm.solve_transpose(db, dx, _prm())
    assert dm.on_chip_solves() == (1, 1) and np.linalg.norm(dx.numpy() - xs) <= 1e-6 * np.linalg.norm(xs)


def _matchings(n, count, seed):
    """Rows of a diagonal and `count` random partners (symmetric): a member's rows couple to the whole system."""
    rng = np.random.default_rng(seed)
    i, j = [], []
    for _ in range(count):
        p = rng.permutation(n)[:n // 2 * 2].reshape(-1, 2)
        i.append(p[:, 0])
        j.append(p[:, 1])
    i, j = np.concatenate(i), np.concatenate(j)
    key = np.unique(np.concatenate([i * n + j, j * n + i, np.arange(n) * (n + 1)]))
    rows, cols = key // n, key % n
    index = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int32)
    return Matrix(n, n, 1, index, (cols + 1).astype(np.int32), np.where(rows == cols, count + 0.5, -1.0)).ensure_dof_index()


# rows whose matrix is streamed and is too much for that (no plan is built); a halo that exceeds LDS (known
# only once the plan is built)
@pytest.mark.parametrize("make, built", [(lambda: _box27(56), False), (lambda: _matchings(400000, 7, 3), True)])
def test_a_system_that_stays_off_the_chip_keeps_no_plan(hip, make, built):
    def left():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    mat = make()
    b = W.uniform_vector(mat.n, seed=1)
    dm = api.DeviceMatrix(mat)
    db, dx = api.DeviceBuffer.from_numpy(b), api.DeviceBuffer(mat.n)
    dm.set_on_chip(False)
    dm.solve(db, dx, _prm())
    x = dx.numpy()
    api.trim()
    before = left()
    dm.set_on_chip(True)
    for first in (True, False):
        dm.solve(db, dx, _prm())
        assert dm.on_chip_solves() == (0, 0) and np.array_equal(x, dx.numpy())
        assert (api.trim() > 0) == (built and first) and left() == before


def _box27(e):
    n = e ** 3
    ids = np.arange(n)
    z, y, x = ids // (e * e), ids // e % e, ids % e
    rows, cols = [], []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                ok = (z + dz >= 0) & (z + dz < e) & (y + dy >= 0) & (y + dy < e) & (x + dx >= 0) & (x + dx < e)
                rows.append(ids[ok])
                cols.append((ids + (dz * e + dy) * e + dx)[ok])
    key = np.sort(np.concatenate(rows) * n + np.concatenate(cols))
    rows, cols = key // n, key % n
    index = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int32)
    return Matrix(n, n, 1, index, (cols + 1).astype(np.int32), np.where(rows == cols, 27.0, -1.0)).ensure_dof_index()


# one workgroup; teams with four and eight rows per thread and the matrix in registers; a streamed matrix;
# 26 rows per thread
@pytest.mark.parametrize("make", [lambda: _matrix(1000, 333, True, 1), lambda: W.poisson7(32), lambda: W.poisson7(72),
                                  lambda: _box27(32), lambda: W.poisson7(78)])
@pytest.mark.parametrize("precond", [1, 0])
def test_time_output_does_not_change_the_solve(make, precond):
    """The flags that ask for the time split (on by default) measure the same solve on chip: same bits of x and
    of the history; the split's parts are positive and within the solution time, and 0 without the flags."""
    mat = make()
    b = W.uniform_vector(mat.n, seed=2)
    dm = api.DeviceMatrix(mat)
    db, dx = api.DeviceBuffer.from_numpy(b), api.DeviceBuffer(mat.n)
    out = []
    for k, flag in enumerate([None, api.MONOLIS_PRM_I_SHOW_TIME, api.MONOLIS_PRM_I_IS_MEASUREMENT,
                              api.MONOLIS_PRM_I_SHOW_TIME_STATISTICS, None]):
        prm = _prm(precond, max_iter=260)
        if flag is not None:
            prm.Iarray[flag] = 1
        h = dm.solve(db, dx, prm, hist_len=261)
        assert dm.on_chip_solves() == (k + 1, 0)
        out.append((dx.numpy(), h, int(prm.Iarray[api.MONOLIS_PRM_I_CUR_ITER])))
        total, spmv, dotp, prec, c0, c1 = prm.Rarray[[3, 5, 6, 7, 8, 9]]
        assert c0 == c1 == 0
        if flag is None:
            assert spmv == dotp == prec == 0
        else:
            assert spmv > 0 and dotp > 0 and (prec > 0) == bool(precond) and spmv + dotp + prec <= total
    for x, h, it in out[1:]:
        assert np.array_equal(x, out[0][0]) and np.array_equal(h, out[0][1]) and it == out[0][2]
