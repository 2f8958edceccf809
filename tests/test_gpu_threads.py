"""Calls from two threads at once on handles of one context: each gives what it gives alone."""
import threading

import numpy as np
import pytest
import scipy.sparse as sp

import prism_amd as P

pytestmark = pytest.mark.gpu


def together(*work):
    """Runs the functions at once, each in a thread; raises what one of them raised."""
    start, errors = threading.Barrier(len(work)), []

    def run(f):
        try:
            start.wait()
            f()
        except BaseException as e:
            errors.append(e)

    ts = [threading.Thread(target=run, args=(f,)) for f in work]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    if errors:
        raise errors[0]


@pytest.mark.parametrize("n", [7, 3000])
def test_products_of_one_matrix(hip, n):
    print(f"case threads products {n}", flush=True)
    rng = np.random.default_rng(n)
    D = sp.random(n, n, 5.0 / n, random_state=1, format="csr") + sp.diags(rng.uniform(4.0, 5.0, n))
    D.sort_indices()
    A = P.Matrix(hip, D.indptr, D.indices, D.data)
    xs = rng.standard_normal((3, n))
    bound = 1e-13 * np.abs(D).sum(axis=1).max() * np.abs(xs).max()

    def products(x):
        for _ in range(200):
            assert np.abs(A.spmv(x) - D @ x).max() <= bound

    def steps():
        exact = xs[2] + (xs[1] - D @ xs[2]) / D.diagonal()
        for _ in range(200):
            assert np.abs(P.solver.Jacobi().step(A, xs[2], xs[1]) - exact).max() <= bound

    together(lambda: products(xs[0]), lambda: products(xs[1]), steps)


def test_green_gauss_fields_of_one_mesh(hip):
    """The sweep in one workgroup shares its scratch among the mesh's fields."""
    print("case threads gradients", flush=True)
    data = P.box(60, 50, 1, jitter=0.0)
    bcs = {s: {"T": ("fixed", 0.5), "f": ("fixed", 0.25)} for s in data.patch_names}
    rng = np.random.default_rng(8)
    values = {name: rng.standard_normal((20, data.n_cells)) for name in ("T", "f")}

    def sweeps(m, name, out):
        field = m.scalar(name, values=values[name][0])
        for v in values[name]:
            field.values = v
            out.append(field.grad())

    def mesh():
        return P.Mesh(hip, data, bcs, [("T", "scalar", "greenGauss"), ("f", "scalar", "greenGauss")])

    alone, shared = {"T": [], "f": []}, {"T": [], "f": []}
    one, two = mesh(), mesh()
    for name in alone:
        sweeps(one, name, alone[name])
    together(*[lambda name=name: sweeps(two, name, shared[name]) for name in shared])
    for name in alone:
        np.testing.assert_array_equal(shared[name], alone[name])


@pytest.mark.parametrize("precond", [None, "sgs"])
def test_solves_on_one_context(hip, precond):
    """Each solve polls its own scalars, through the context's one pinned buffer."""
    print(f"case threads solves {precond}", flush=True)
    systems, alone = [], []
    for n in (900, 5000):
        rng = np.random.default_rng(n)
        A = sp.diags([rng.uniform(-1.0, 0.3, n - o) for o in (1, 22)] * 2, (1, 22, -1, -22), format="csr")
        A = (A + sp.diags(1.02 * np.asarray(abs(A).sum(axis=1)).ravel() + 0.01)).tocsr()
        A.sort_indices()
        b = rng.standard_normal(n)

        def solves(times, M=P.Matrix(hip, A.indptr, A.indices, A.data), b=b):
            s = P.solver.BiCGSTAB(tol=1e-12, precond=precond)
            return [s.step(M, np.zeros(len(b)), b) for _ in range(times)]

        systems.append(solves)
        alone.append(solves(1)[0])
        assert np.linalg.norm(b - A @ alone[-1]) <= 2e-12 * np.linalg.norm(b)
    got = [None, None]

    def run(k):
        got[k] = systems[k](10)

    together(lambda: run(0), lambda: run(1))
    for xs, x in zip(got, alone):
        for y in xs:
            np.testing.assert_array_equal(y, x)
