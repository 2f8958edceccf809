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
