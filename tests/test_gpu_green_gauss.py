"""The Green-Gauss sweep in one workgroup (narrow levels, among them levels wider than the
workgroup) and as a launch for each level (wide ones), against the oracle's sequential sweep,
twice: the second sweep starts from the first one's gradients."""
import numpy as np
import pytest

import prism_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,kw", [((1, 1, 1), {}), ((5, 1, 1), {}), ((9, 7, 5), dict(jitter=0.2, tets=True)),
                                     ((700, 700, 1), dict(jitter=0.0)), ((40, 38, 36), dict(jitter=0.2)),
                                     ((44, 44, 44), dict(jitter=0.2))],
                         ids=["one_cell", "line", "tets", "wider_than_workgroup", "narrow", "wide"])
def test_sweep_matches_oracle(hip, ref, dims, kw):
    print(f"case green-gauss {dims}", flush=True)
    data = P.box(*dims, **kw)
    out = []
    for be in (hip, ref):
        bcs = {s: {"T": ("fixed", 0.5)} for s in data.patch_names}
        bcs["front"]["T"] = ("zero-gradient", None)
        m = P.Mesh(be, data, bcs, [("T", "scalar", "greenGauss")])
        rng = np.random.default_rng(5)
        T = m.scalar("T", values=rng.standard_normal(m.n_cells))
        g1 = T.grad()
        T.values = rng.standard_normal(m.n_cells)
        out.append((g1, T.grad()))
    for a, b in zip(*out):
        # the same expressions in the same order: at most the last bits of compiled divisions part
        assert np.abs(a - b).max() <= 1e-13 * np.abs(b).max()
