"""GPU solver paths beyond the FP64 default: FP32 + FP64 refinement against the FP64 oracle,
the reference-cell system (deflated on the device) against the oracle's exact solve of the
reference's fixed system, and a Jacobi-preconditioned solve."""
import numpy as np
import pytest

import prism_amd as P
from prism_amd import cases

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def advection(be):
    c = cases.advection_diffusion(be, P.box(14, 12, 10, jitter=0.2, seed=2), scheme="Upwind")
    return c


@pytest.mark.usefixtures("iteration")
@pytest.mark.parametrize("precision,tol,bound", [("fp64", 1e-12, 1e-10), ("fp32", 1e-10, 1e-8)])
def test_precisions_against_oracle(hip, ref, precision, tol, bound):
    out = {}
    for name, be in (("hip", hip), ("ref", ref)):
        c = advection(be)
        slv = P.solver.BiCGSTAB(tol=tol, precision=precision)
        r = slv.solve(c["eqn"], 2, 1e-20)
        out[name] = (c["T"].values, r)
    assert rel(out["hip"][0], out["ref"][0]) <= bound
    if precision == "fp32":
        assert out["hip"][1].refinements >= 2  # the FP64 residual was recomputed


@pytest.mark.usefixtures("iteration")
@pytest.mark.parametrize("precision,bound", [("fp64", 1e-10), ("fp32", 1e-7)])
def test_reference_cell_system(hip, ref, precision, bound):
    """All-Neumann pressure correction with reference cell 3 and value 0.25: the device solves
    the deflated system; the oracle solves the reference's fixed system exactly."""
    out = {}
    for name, be in (("hip", hip), ("ref", ref)):
        c = cases.pressure_correction(be, n=14)
        slv = P.solver.BiCGSTAB(tol=1e-12 if precision == "fp64" else 1e-9, precision=precision)
        r = slv.solve(c["eqn"], 2, 1e-30, ref_cell=3, ref_value=0.25)
        out[name] = (c["p"].values, r)
    ph, pr = out["hip"][0], out["ref"][0]
    assert rel(ph, pr) <= bound
    assert abs(ph[3] - 0.25) <= 1e-8
    assert out["hip"][1].final_residual < 1e-8


@pytest.mark.usefixtures("iteration")
def test_jacobi_preconditioned(hip, ref):
    out = {}
    for name, be in (("hip", hip), ("ref", ref)):
        c = advection(be)
        slv = P.solver.BiCGSTAB(tol=1e-12, precond="jacobi")
        slv.solve(c["eqn"], 2, 1e-20)
        out[name] = c["T"].values
    assert rel(out["hip"], out["ref"]) <= 1e-10


@pytest.mark.parametrize("n", [64, 128])
def test_solve_scaled_residual_partials(hip, n):
    """ISolver::solve on the n^3 pressure-correction system (reference cell, FP32 + refinement):
    the scaled residual's reduction runs on up to 1024 blocks of 512-row chunks, more than the
    Krylov kernels' grid (256 or 512 blocks), and its two partial maxima per block must fit the
    workspace buffer (the launcher checks the capacity and raises otherwise)."""
    print(f"case solve scaled residual {n}^3", flush=True)
    c = cases.pressure_correction(hip, n=n)
    r = P.solver.BiCGSTAB(tol=1e-8, precision="fp32").solve(c["eqn"], 1, 1e-30, ref_cell=0)
    assert r.krylov_rel_residual <= 1e-8
    assert np.isfinite(r.final_residual) and r.final_residual < 1e-6


def test_fp32_stall_finishes_in_fp64(hip):
    """128^3 MUSCL advection-diffusion with reliable updates only every 10x of residual drop:
    the three-kernel FP32 iteration stalls near a relative residual of 1 there (two forced
    updates without progress).  The step then restarts from the best reliable update in FP64
    and converges, instead of returning that stalled x."""
    print("case fp32 stall 128^3 inner_tol 0.1", flush=True)
    c = cases.advection_diffusion(hip, P.box(128, 128, 128, jitter=0.2, seed=1), scheme="MUSCL", kappa=1e-3)
    c["eqn"].update_coeffs()
    out = {}
    for prec, inner in (("fp64", 0.0), ("fp32", 0.1)):
        c["T"].fill(0.0)
        r = P.solver.BiCGSTAB(tol=1e-8, precision=prec, inner_tol=inner).step_eqn(c["eqn"])
        assert r.krylov_rel_residual <= 1e-8
        out[prec] = c["T"].values
    assert rel(out["fp32"], out["fp64"]) <= 1e-6


def test_fp32_large_row_pairs(hip):
    """96^3 (several rows per thread, DIA storage, 512 blocks): the FP32 + refinement solution
    against the FP64 GPU solution of the same system."""
    c = cases.advection_diffusion(hip, P.box(96, 96, 96, jitter=0.2, seed=1), scheme="MUSCL", kappa=1e-3)
    c["eqn"].update_coeffs()
    out = {}
    for prec in ("fp64", "fp32"):
        c["T"].fill(0.0)
        r = P.solver.BiCGSTAB(tol=1e-10, precision=prec, max_iters=20000).step_eqn(c["eqn"])
        assert r.krylov_rel_residual <= 1e-9
        out[prec] = c["T"].values
    assert rel(out["fp32"], out["fp64"]) <= 1e-7


def test_wide_offsets_int32_columns(hip, ref):
    """A 75 x 75 x 2 hex box split into tetrahedra (67,500 cells): neighbours across a hex
    layer are 6 x 75 x 75 = 33,750 rows apart, beyond 16-bit offsets from the row, so the
    sliced ELL stores 16-bit offsets from a base per slice and slot.
    Pressure-correction system with the reference cell: FP64 against the oracle, FP32 +
    refinement against FP64."""
    out = {}
    for name, be, prec in (("ref", ref, "fp64"), ("hip64", hip, "fp64"), ("hip32", hip, "fp32")):
        c = cases.pressure_correction(be, n=75, data=P.box(75, 75, 2, tets=True))
        slv = P.solver.BiCGSTAB(tol=1e-14 if prec == "fp64" else 1e-10, precision=prec, max_iters=20000)
        r = slv.solve(c["eqn"], 3, 1e-30, ref_cell=0, ref_value=0.0)
        out[name] = (c["p"].values, r)
        print(name, r, flush=True)
    e64 = rel(out["hip64"][0], out["ref"][0])
    e32 = rel(out["hip32"][0], out["hip64"][0])
    print(f"fp64 vs oracle {e64:.3e}, fp32 vs fp64 {e32:.3e}", flush=True)
    assert e64 <= 1e-9  # this system's conditioning: the FP64 solve to 1e-14 leaves 1.1e-10
    assert out["hip32"][1].krylov_rel_residual <= 1e-9
    assert e32 <= 1e-6
