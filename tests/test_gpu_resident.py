"""The resident BiCGSTAB kernel (resident.hip) against the three-kernel iteration and against
exact solutions: with one row per thread both form every sum in the same order, so the
solutions are the same bits; with more, each solution satisfies the system."""
import threading
import time

import numpy as np
import pytest
import scipy.sparse as sp

import prism_amd as P
from devmem import full_device

pytestmark = pytest.mark.gpu


def scattered(n, row, seed=3):
    """Strictly diagonally dominant, nonsymmetric, `row` scattered off-diagonals a row at most."""
    rng = np.random.default_rng(seed)
    A = sp.coo_matrix((rng.uniform(-1.0, 0.3, n * row), (np.repeat(np.arange(n), row), rng.integers(0, n, n * row))),
                      shape=(n, n)).tocsr()
    A.setdiag(0.0)
    A.setdiag(1.1 * np.asarray(abs(A).sum(axis=1)).ravel() + 0.1)
    A.sort_indices()
    return A


def diagonals(n, offsets, seed=4):
    """The same on the given diagonals."""
    rng = np.random.default_rng(seed)
    A = sp.diags([rng.uniform(-1.0, 0.3, n - abs(o)) for o in offsets], offsets, shape=(n, n), format="csr")
    A = (A + sp.diags(1.1 * np.asarray(abs(A).sum(axis=1)).ravel() + 0.1)).tocsr()
    A.sort_indices()
    return A


def matrix(hip, A):
    return P.Matrix(hip, A.indptr, A.indices, A.data)


def solve(hip, A, monkeypatch, resident, **kw):
    monkeypatch.setenv("PRISM_KRYLOV_RESIDENT", "1" if resident else "0")
    b = np.random.default_rng(9).standard_normal(A.shape[0])
    hip.set_timing(True)
    hip.reset_timing()
    out = []
    x = P.solver.BiCGSTAB(tol=1e-12, max_iters=2000, **kw).step(matrix(hip, A), np.zeros(A.shape[0]), b, out)
    names = set(hip.kernel_stats())
    hip.set_timing(False)
    return x, b, out[0], any(k.startswith(("bicgstab_resident", "sgs_resident")) for k in names)


SYSTEMS = {
    "sell5_1": scattered(1, 1), "sell5_63": scattered(63, 3), "sell5_512": scattered(512, 4),
    "sell5_513": scattered(513, 4), "sell8_640": scattered(640, 7), "sell8_9001": scattered(9001, 7),
    "sell16_700": scattered(700, 14), "sell16_6400": scattered(6400, 12),
    "dia3_513": diagonals(513, (-1, 1)), "dia5_1600": diagonals(1600, (-40, -1, 1, 40)),
    "dia7_4095": diagonals(4095, (-195, -13, -1, 1, 13, 195)),
    "dia8_2049": diagonals(2049, (-500, -20, -3, -1, 1, 20, 500)),
}


@pytest.mark.parametrize("precision,precond", [("fp64", None), ("fp64", "jacobi"), ("fp32", None), ("fp32", "jacobi")])
@pytest.mark.parametrize("name", list(SYSTEMS))
def test_same_bits_as_three_kernels(hip, monkeypatch, name, precision, precond):
    print(f"case resident {name} {precision} {precond}", flush=True)
    A = SYSTEMS[name]
    x1, b, r1, used1 = solve(hip, A, monkeypatch, True, precision=precision, precond=precond)
    x0, _, r0, used0 = solve(hip, A, monkeypatch, False, precision=precision, precond=precond)
    assert not used0 and (used1 or r1.krylov_iters == 0)
    np.testing.assert_array_equal(x1, x0)
    assert (r1.krylov_iters, r1.refinements, r1.restarts) == (r0.krylov_iters, r0.refinements, r0.restarts)
    # ||b - A x|| <= 1e-12 ||b|| recomputed by the library, to twice that here (other rounding)
    assert np.linalg.norm(b - A @ x1) <= 2e-12 * np.linalg.norm(b)


@pytest.mark.parametrize("n", [6400, 100000])
def test_ends_of_launches(hip, monkeypatch, n):
    """Short solves end while blocks may still wait for the last p of others: every one of many
    has the same bits."""
    print(f"case resident ends {n}", flush=True)
    A = scattered(n, 12)
    x0 = solve(hip, A, monkeypatch, False)[0]
    for _ in range(20):
        np.testing.assert_array_equal(solve(hip, A, monkeypatch, True)[0], x0)


@pytest.mark.parametrize("n,precision", [(255 * 512 + 1, "fp64"), (262144, "fp64"), (255 * 1536, "fp64"),
                                         (255 * 512 + 1, "fp32"), (400001, "fp32"), (255 * 2048, "fp32")])
def test_several_rows_per_thread(hip, monkeypatch, n, precision):
    print(f"case resident rows {n} {precision}", flush=True)
    A = diagonals(n, (-4096, -64, -1, 1, 64, 4096))
    x, b, r, used = solve(hip, A, monkeypatch, True, precision=precision)
    assert used
    assert r.krylov_rel_residual <= 1e-12
    assert np.linalg.norm(b - A @ x) <= 2e-12 * np.linalg.norm(b)


def near(n, row, seed=3):
    """`row` off-diagonals a row within 100 columns (16-bit sliced ELL), other ones in each row."""
    rng = np.random.default_rng(seed)
    rows = np.repeat(np.arange(n), row)
    cols = np.clip(rows + rng.integers(-100, 100, n * row), 0, n - 1)
    A = sp.coo_matrix((rng.uniform(-1.0, 0.3, n * row), (rows, cols)), shape=(n, n)).tocsr()
    A.setdiag(0.0)
    A.setdiag(1.1 * np.asarray(abs(A).sum(axis=1)).ravel() + 0.1)
    A.sort_indices()
    return A


EIGHT = (-500, -20, -3, -1, 1, 20, 500)
SEVEN = (-4096, -64, -1, 1, 64, 4096)


@pytest.mark.parametrize("build,n,arg,precision,precond", [
    # sliced ELL, five and eight entries, two rows per thread up to the most
    (scattered, 255 * 512 + 1, 4, "fp64", None), (scattered, 255 * 512 + 1, 7, "fp64", None),
    (near, 255 * 1024 + 1, 4, "fp64", None), (near, 255 * 1024, 7, "fp64", None),
    (scattered, 255 * 1536, 4, "fp64", None), (near, 255 * 1536, 7, "fp64", None),
    (scattered, 255 * 512 + 1, 4, "fp32", None), (near, 255 * 512 + 1, 7, "fp32", None),
    (near, 255 * 1536 + 1, 4, "fp32", None), (scattered, 255 * 1536 + 1, 7, "fp32", None),
    (near, 255 * 2048, 4, "fp32", None), (near, 255 * 2048, 7, "fp32", None),
    # eight diagonals
    (diagonals, 255 * 512 + 1, EIGHT, "fp64", None), (diagonals, 255 * 1536, EIGHT, "fp64", None),
    (diagonals, 255 * 1024 + 1, EIGHT, "fp32", None), (diagonals, 255 * 2048, EIGHT, "fp32", None),
    # Jacobi, with coefficients kept and read again for each product
    (diagonals, 262144, SEVEN, "fp64", "jacobi"), (near, 200001, 4, "fp64", "jacobi"),
    (scattered, 200001, 7, "fp32", "jacobi"), (diagonals, 255 * 2048, SEVEN, "fp32", "jacobi"),
    (diagonals, 255 * 2048 + 1, SEVEN, "fp64", "jacobi"), (diagonals, 255 * 3072, SEVEN, "fp32", "jacobi")])
def test_every_plan_of_several_rows(hip, monkeypatch, build, n, arg, precision, precond):
    print(f"case resident plan {build.__name__} {n} {arg} {precision} {precond}", flush=True)
    A = build(n, arg)
    x, b, r, used = solve(hip, A, monkeypatch, True, precision=precision, precond=precond)
    assert used
    assert r.krylov_rel_residual <= 1e-12
    assert np.linalg.norm(b - A @ x) <= 2e-12 * np.linalg.norm(b)


@pytest.mark.parametrize("nx,precond", [(128, None), (300, "sgs")])
def test_more_iterations_than_two_launches(hip, monkeypatch, nx, precond):
    """A weakly dominant system, one row per thread: the state goes from full launch to full launch."""
    print(f"case resident launches {nx} {precond}", flush=True)
    line = sp.diags([-1.0, 2.0, -1.0], [-1, 0, 1], shape=(nx, nx))
    A = (sp.kron(sp.identity(nx), line) + sp.kron(line, sp.identity(nx))).tocsr()
    A.sort_indices()
    A.data *= np.where(A.data < 0, np.random.default_rng(12).uniform(0.98, 1.02, A.nnz), 1.0)
    b = np.random.default_rng(9).standard_normal(nx * nx)
    xs, rs = [], []
    for resident in "10":
        monkeypatch.setenv("PRISM_KRYLOV_RESIDENT", resident)
        out = []
        xs.append(P.solver.BiCGSTAB(tol=1e-10, precond=precond).step(matrix(hip, A), 0.0 * b, b, out))
        rs.append(out[0])
    assert rs[0].krylov_iters > 256
    assert (rs[0].krylov_iters, rs[0].restarts) == (rs[1].krylov_iters, rs[1].restarts)
    np.testing.assert_array_equal(xs[0], xs[1])


@pytest.mark.parametrize("n,offsets,precision", [
    (255 * 1536 + 1, (-4096, -64, -1, 1, 64, 4096), "fp64"), (255 * 2048, (-511, -1, 1, 511), "fp64"),
    (255 * 2048 + 1, (-4096, -64, -1, 1, 64, 4096), "fp64"), (255 * 2560, (-4097, -63, -1, 1, 63, 4097), "fp64"),
    (255 * 2560, (-300001, -5, 5, 300001), "fp64"),
    (255 * 2048 + 1, (-4096, -64, -1, 1, 64, 4096), "fp32"), (255 * 2560 + 1, (-511, -1, 1, 511), "fp32"),
    (255 * 3072, (-4097, -63, -1, 1, 63, 4097), "fp32")])
def test_streamed_coefficients(hip, monkeypatch, n, offsets, precision):
    """Rows per thread at which the coefficients are read again for each product."""
    print(f"case resident streamed {n} {len(offsets) + 1} {precision}", flush=True)
    A = diagonals(n, offsets)
    x, b, r, used = solve(hip, A, monkeypatch, True, precision=precision)
    assert used
    assert r.krylov_rel_residual <= 1e-12
    assert np.linalg.norm(b - A @ x) <= 2e-12 * np.linalg.norm(b)


@pytest.mark.parametrize("n", [255 * 2048 + 1, 255 * 2560 + 1])
def test_streamed_zero_row_sums(hip, monkeypatch, n):
    """FP32 without a diagonal term in the difference form (symmetric, singular, consistent)."""
    print(f"case resident zero row sums {n}", flush=True)
    rng = np.random.default_rng(6)
    U = sp.diags([-rng.integers(32, 64, n - o) / 64.0 for o in (1, 64, 4096)], (1, 64, 4096), shape=(n, n))
    A = (U + U.T).tocsr()
    A = (A - sp.diags(np.asarray(A.sum(axis=1)).ravel())).tocsr()
    A.sort_indices()
    monkeypatch.setenv("PRISM_KRYLOV_RESIDENT", "1")
    b = A @ rng.standard_normal(n)
    out = []
    x = P.solver.BiCGSTAB(tol=1e-10, max_iters=4000, precision="fp32").step(matrix(hip, A), np.zeros(n), b, out)
    assert out[0].krylov_rel_residual <= 1e-10
    assert np.linalg.norm(b - A @ x) <= 2e-10 * np.linalg.norm(b)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_wait_that_runs_out_falls_back(hip, monkeypatch, precision):
    """One poll per wait: the blocks give up at their first wait, and the solve goes on with the
    three-kernel iteration."""
    print(f"case resident spin {precision}", flush=True)
    hip = P.Backend.hip(0)  # it rests from resident kernels afterwards: not the other tests' context
    monkeypatch.setenv("PRISM_KRYLOV_SPIN", "1")
    A = scattered(9001, 7)
    x, b, r, used = solve(hip, A, monkeypatch, True, precision=precision)
    assert used and r.krylov_rel_residual <= 1e-12
    assert np.linalg.norm(b - A @ x) <= 2e-12 * np.linalg.norm(b)


@pytest.mark.parametrize("precond,kernel", [(None, "bicgstab_resident_f64"), ("sgs", "sgs_resident")])
def test_waits_that_run_out_are_remembered(hip, monkeypatch, precond, kernel):
    """A context whose resident kernels gave up keeps off them for a multiple of the time lost,
    longer each time, and takes them again afterwards."""
    print(f"case resident rest {precond}", flush=True)
    monkeypatch.delenv("PRISM_KRYLOV_RESIDENT", raising=False)
    monkeypatch.setenv("PRISM_KRYLOV_SPIN", "1")
    be = P.Backend.hip(0)
    A = diagonals(5000, (-22, -1, 1, 22))
    M, b = matrix(be, A), np.random.default_rng(9).standard_normal(5000)
    s = P.solver.BiCGSTAB(tol=1e-12, precond=precond)

    def launches(times):
        be.set_timing(True)
        be.reset_timing()
        for _ in range(times):
            x = s.step(M, np.zeros(5000), b)
            assert np.linalg.norm(b - A @ x) <= 2e-12 * np.linalg.norm(b)
        n = be.kernel_stats().get(kernel, (0,))[0]
        be.set_timing(False)
        return n

    # a context that forgets would launch one in each solve
    assert 1 <= launches(200) < 200
    monkeypatch.delenv("PRISM_KRYLOV_SPIN")
    for _ in range(300):  # a rest is 1024 times the last wait's 0.1 ms or less, as a rule
        if launches(1):
            break
        time.sleep(0.1)
    assert launches(5) >= 5
    be.close()


def test_without_room_for_the_exchange(hip, monkeypatch):
    """A solve whose other buffers are there, on a device with at most 24 of the 24.9 MiB left that
    the exchanged words take: the single kernels."""
    print("case resident without room", flush=True)
    n = 255 * 2560
    A = diagonals(n, (-4096, -1, 1, 4096))
    M, b = matrix(hip, A), np.random.default_rng(9).standard_normal(n)
    s = P.solver.BiCGSTAB(tol=1e-12)
    monkeypatch.setenv("PRISM_KRYLOV_RESIDENT", "0")
    expected = s.step(M, np.zeros(n), b)
    monkeypatch.setenv("PRISM_KRYLOV_RESIDENT", "1")
    with full_device(8 << 20) as left:
        assert left < 5 * 8 * n
        x = s.step(M, np.zeros(n), b)
    np.testing.assert_array_equal(x, expected)  # the resident sums run in another order here
    hip.set_timing(True)
    hip.reset_timing()
    s.step(M, np.zeros(n), b)
    assert "bicgstab_resident_f64" in hip.kernel_stats()
    hip.set_timing(False)


def test_two_threads_share_the_device(hip, monkeypatch):
    """Two contexts solve at once; together their blocks exceed the device, so one of them takes
    the three-kernel iteration now and then: the same bits either way."""
    print("case resident two threads", flush=True)
    monkeypatch.delenv("PRISM_KRYLOV_RESIDENT", raising=False)
    A = diagonals(100000, (-2000, -50, -1, 1, 50, 2000))
    b = np.random.default_rng(1).standard_normal(A.shape[0])
    alone = P.solver.BiCGSTAB(tol=1e-12).step(matrix(hip, A), np.zeros(A.shape[0]), b)
    out = {}

    def work(k):
        be = P.Backend.hip(0)
        M = matrix(be, A)
        out[k] = [P.solver.BiCGSTAB(tol=1e-12).step(M, np.zeros(A.shape[0]), b) for _ in range(3)]

    ts = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for k in range(2):
        for x in out[k]:
            np.testing.assert_array_equal(x, alone)


@pytest.mark.parametrize("n,offsets,precision,precond", [
    (50000, (-2000, -50, -1, 1, 50, 2000), "fp64", None),      # 98 blocks each: both run
    (100000, (-2000, -50, -1, 1, 50, 2000), "fp32", None),     # one at a time; the single kernels beside it
    (150000, (-2000, -50, -1, 1, 50, 2000), "fp64", None),     # two rows per thread: they take turns
    (64 * 64 * 40, (-4096, -64, -1, 1, 64, 4096), "fp32", None),
    (100000, (-50, -1, 1, 50), "fp64", "sgs")])
def test_threads_do_not_change_the_bits(hip, monkeypatch, n, offsets, precision, precond):
    """Three contexts solve at once, beside each other, in turns, or with the single kernels where
    these give the same bits: the bits of a solve alone."""
    print(f"case resident threads {n} {precision} {precond}", flush=True)
    monkeypatch.delenv("PRISM_KRYLOV_RESIDENT", raising=False)
    A = diagonals(n, offsets)
    b = np.random.default_rng(2).standard_normal(n)
    s = P.solver.BiCGSTAB(tol=1e-12, precision=precision, precond=precond)
    alone = s.step(matrix(hip, A), np.zeros(n), b)
    out = [[] for _ in range(3)]

    def work(xs):
        M = matrix(P.Backend.hip(0), A)
        xs.extend(s.step(M, np.zeros(n), b) for _ in range(4))

    ts = [threading.Thread(target=work, args=(xs,)) for xs in out]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for xs in out:
        assert len(xs) == 4
        for x in xs:
            np.testing.assert_array_equal(x, alone)


@pytest.mark.parametrize("n,row", [(1, 1), (64, 3), (257, 4), (513, 5), (5000, 5), (40000, 3)])
def test_sgs_same_bits_as_its_launches(hip, monkeypatch, n, row):
    """The resident SGS iteration (sgs_resident.hip), on patterns of two to eight colours."""
    print(f"case resident sgs {n} {row}", flush=True)
    offsets = [o for k in range(1, (row + 1) // 2 + 1) for o in (-(7 * k * k - 6), 7 * k * k - 6) if 7 * k * k - 6 < n]
    A = diagonals(n, tuple(offsets)) if offsets else scattered(1, 1)
    x1, b, r1, used1 = solve(hip, A, monkeypatch, True, precond="sgs")
    x0, _, r0, used0 = solve(hip, A, monkeypatch, False, precond="sgs")
    assert used1 and not used0
    np.testing.assert_array_equal(x1, x0)
    assert (r1.krylov_iters, r1.restarts, r1.converged) == (r0.krylov_iters, r0.restarts, r0.converged)
    assert np.linalg.norm(b - A @ x1) <= 2e-12 * np.linalg.norm(b)


def broken_down(n, sgs):
    """2 x 2 blocks on which rho is exactly zero after the first iteration (from b, which has no
    second components, s and t have none of the first): A M^-1 has the blocks
    [[1, 0], [k, h]] with (k, h) = (1/8, 3/4) and (-1/8, 5/4) in turn, so the first iteration
    leaves a residual.  sgs: A has those blocks after preconditioning ([[1, a], [1/2, 1]], a = +-1/2)."""
    odd = np.arange(n // 2) % 2 == 1
    d, low, up = np.ones(n), np.zeros(n - 1), np.zeros(n - 1)
    if sgs:
        low[::2], up[::2] = 0.5, np.where(odd, -0.5, 0.5)
    else:
        d[1::2], low[::2] = np.where(odd, 1.25, 0.75), np.where(odd, -0.125, 0.125)
    A = sp.diags([low, d, up], [-1, 0, 1], format="csr")
    A.eliminate_zeros()
    b = np.zeros(n)
    b[::2] = 1.0
    return A, b


@pytest.mark.parametrize("quota", [1, 2, 128])
@pytest.mark.parametrize("n", [4, 1026, 40000, 130560])
@pytest.mark.parametrize("precond", [None, "sgs"])
def test_breakdown_at_a_launch_boundary(hip, monkeypatch, precond, n, quota):
    """The restart after a rho breakdown that a launch finds in its first test (quota 1: that
    launch ends before its blocks have exchanged anything), and in a later one."""
    print(f"case resident breakdown {precond} {n} {quota}", flush=True)
    A, b = broken_down(n, precond == "sgs")
    monkeypatch.setenv("PRISM_KRYLOV_QUOTA", str(quota))
    xs, rs = [], []
    for resident in "10":
        monkeypatch.setenv("PRISM_KRYLOV_RESIDENT", resident)
        out = []
        xs.append(P.solver.BiCGSTAB(tol=1e-12, precond=precond).step(matrix(hip, A), np.zeros(n), b, out))
        rs.append(out[0])
    np.testing.assert_array_equal(xs[0], xs[1])
    assert [(r.krylov_iters, r.restarts, r.converged) for r in rs] == [(rs[0].krylov_iters, 1, 1)] * 2
    assert np.linalg.norm(b - A @ xs[0]) <= 2e-12 * np.linalg.norm(b)


@pytest.mark.parametrize("quota", [1, 2, 3])
@pytest.mark.parametrize("precision,precond", [("fp64", None), ("fp32", "jacobi"), ("fp64", "sgs")])
@pytest.mark.parametrize("name", ["dia7_4095", "sell8_640", "sell5_513"])
def test_state_handed_from_launch_to_launch(hip, monkeypatch, name, precision, precond, quota):
    print(f"case resident hand-over {name} {precision} {precond} {quota}", flush=True)
    A = SYSTEMS[name]
    monkeypatch.setenv("PRISM_KRYLOV_QUOTA", str(quota))
    x1, b, r1, used = solve(hip, A, monkeypatch, True, precision=precision, precond=precond)
    x0, _, r0, _ = solve(hip, A, monkeypatch, False, precision=precision, precond=precond)
    assert used
    np.testing.assert_array_equal(x1, x0)
    assert (r1.krylov_iters, r1.refinements, r1.restarts) == (r0.krylov_iters, r0.refinements, r0.restarts)


def test_sgs_wait_that_runs_out_falls_back(hip, monkeypatch):
    print("case resident sgs spin", flush=True)
    hip = P.Backend.hip(0)
    monkeypatch.setenv("PRISM_KRYLOV_SPIN", "1")
    A = diagonals(5000, (-22, -1, 1, 22))
    x, b, r, _ = solve(hip, A, monkeypatch, True, precond="sgs")
    assert r.converged
    assert np.linalg.norm(b - A @ x) <= 2e-12 * np.linalg.norm(b)
