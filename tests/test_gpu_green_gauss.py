"""The Green-Gauss sweep in one workgroup (narrow levels, among them levels wider than the
workgroup) and as a launch for each level (wide ones), against the oracle's sequential sweep,
twice: the second sweep starts from the first one's gradients."""
import numpy as np
import pytest

import prism_amd as P
from devmem import full_device

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


def test_sweep_without_room_for_its_scratch(hip):
    """A device without the memory for the sweep's scratch (176 MB here, 96 MB are left): the level
    launches take over, in the failing call and in later ones."""
    print("case green-gauss without scratch", flush=True)
    data = P.box(700, 700, 1, jitter=0.0)
    bcs = {s: {"T": ("fixed", 0.5)} for s in data.patch_names}
    rng = np.random.default_rng(6)
    values = [rng.standard_normal(data.n_cells) for _ in range(2)]
    meshes = [P.Mesh(hip, data, bcs, [("T", "scalar", "greenGauss")]) for _ in range(2)]
    fields = [m.scalar("T", values=values[0]) for m in meshes]
    expected = fields[0].grad()
    with full_device(96 << 20) as left:
        assert left < 360 * data.n_cells
        got = fields[1].grad()
    assert np.abs(got - expected).max() <= 1e-13 * np.abs(expected).max()
    for f in fields:
        f.values = values[1]
    expected, got = fields[0].grad(), fields[1].grad()
    assert np.abs(got - expected).max() <= 1e-13 * np.abs(expected).max()
