"""The linear assembly kernels (residual and CG matvec of linear materials) at the
sizes where its tiling can go wrong, against the oracle: grids below, at and one
past the 15-node tile in y and z and odd in x, tensors beside isotropic phases
(staged table, and more phases than it holds), 16-bit ids, per-voxel moduli,
B-bar and one-point elements, and every depth of the x march.

Tolerances: FP64 1e-12 of the field's maximum (about 200 operations per value:
rounding order only), FP32 1e-5 (the same at 6e-8)."""
import numpy as np
import pytest

import oracle
from fans_amd import gpu
from fans_amd.problem import MaterialGroup, Problem

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return float(np.max(np.abs(np.asarray(a) - np.asarray(b))) / np.max(np.abs(b)))


def _spd(n, rng):
    a = rng.standard_normal((n, n))
    return a @ a.T + n * np.eye(n)


def _groups(model, nph, rng):
    if model == "thermal":
        return 1, [MaterialGroup("LinearThermalIsotropic", list(range(nph)), {"conductivity": list(rng.uniform(1, 9, nph))})]
    if model == "elastic":
        return 3, [MaterialGroup("LinearElasticIsotropic", list(range(nph)),
                                 {"bulk_modulus": list(rng.uniform(2, 60, nph)),
                                  "shear_modulus": list(rng.uniform(1, 30, nph))})]
    h, n, iso, tri, s = ((1, 3, "LinearThermalIsotropic", "LinearThermalTriclinic", "K") if model == "thermal_tensor"
                         else (3, 6, "LinearElasticIsotropic", "LinearElasticTriclinic", "C"))
    Cs = [_spd(n, rng) for _ in range(nph - 1)]
    props = {f"{s}_{i + 1}{j + 1}": [float(C[i, j]) for C in Cs] for i in range(n) for j in range(i, n)}
    one = {"conductivity": [3.0]} if h == 1 else {"bulk_modulus": [20.0], "shear_modulus": [7.0]}
    return h, [MaterialGroup(tri, list(range(1, nph)), props), MaterialGroup(iso, [0], one)]


@pytest.mark.parametrize("model,nph,dims,fe,L", [
    ("elastic", 3, (4, 6, 8), "HEX8", (1.0, 1.0, 1.0)),        # tiles wrap the grid more than once, unequal edges
    ("elastic", 2, (9, 15, 16), "HEX8", (9.0, 15.0, 16.0)),    # whole tile in y, one node past it in z; cubic voxels
    ("elastic", 2, (15, 32, 30), "BBAR", (15.0, 32.0, 30.0)),
    ("elastic", 2, (5, 18, 48), "HEX8R", (1.0, 2.0, 1.0)),
    ("elastic", 300, (10, 16, 18), "HEX8", (10.0, 16.0, 18.0)),  # 16-bit ids: table in memory
    ("thermal", 3, (3, 5, 2), "HEX8", (1.0, 1.0, 1.0)),
    ("thermal", 2, (9, 30, 32), "HEX8", (9.0, 30.0, 32.0)),
    ("thermal_tensor", 4, (6, 16, 12), "HEX8", (1.0, 1.5, 0.5)),
    ("thermal_tensor", 300, (12, 10, 16), "HEX8R", (1.0, 1.0, 1.0)),
    ("elastic_tensor", 4, (6, 16, 12), "HEX8", (1.0, 1.5, 0.5)),
    ("elastic_tensor", 5, (9, 15, 32), "BBAR", (1.0, 1.0, 1.0)),
    ("elastic_tensor", 200, (8, 18, 16), "HEX8", (1.0, 1.0, 1.0)),  # byte ids, more tensors than LDS takes
    ("elastic_tensor", 300, (8, 18, 16), "HEX8R", (1.0, 1.0, 1.0)),
])
def test_linear_assembly_against_oracle(model, nph, dims, fe, L):
    print(f"[gpu-case] assembly {model} {nph} phases {dims} {fe}", flush=True)
    rng = np.random.default_rng(11)
    h, groups = _groups(model, nph, rng)
    ms = rng.integers(0, nph, size=dims).astype(np.uint16)
    p = Problem(dims=dims, howmany=h, ms=ms, groups=groups, fe_type=fe, method="cg", L=L, tol=1e-10, n_it=10)
    u = rng.standard_normal(dims + (h,)) * 0.01
    g0 = rng.uniform(-0.01, 0.01, 3 if h == 1 else 6)
    o = oracle.Oracle(p)
    o.set_gradient(g0)
    r_o, k_o = o.residual(u), o.residual(u, linear_kd=True)
    for precision in ("fp64", "mixed"):  # each form has its own kernel
        g = gpu.GpuSolver(p, precision=precision)
        try:
            g.set_gradient(g0)
            for planes in (None, 1, 2, 3, dims[0]):
                if planes:
                    g.set_asm_planes(planes)
                assert relerr(g.residual(u), r_o) < 1e-12, (precision, planes)
                assert relerr(g.residual(u, linear_kd=True), k_o) < 1e-12, (precision, planes)
            if precision == "mixed":
                g.set_operator_fp32(True)
                assert relerr(g.residual(u, linear_kd=True), k_o) < 1e-5
        finally:
            g.close()


@pytest.mark.parametrize("h,dims,L", [(3, (6, 16, 12), (6.0, 16.0, 12.0)), (3, (5, 9, 18), (1.0, 1.0, 2.0)),
                                      (1, (9, 18, 16), (9.0, 18.0, 16.0))])
def test_voxel_moduli_match_phases(h, dims, L):
    """Per-voxel moduli equal to the phases' give the phases' matvec (and so the
    oracle's)."""
    print(f"[gpu-case] voxel moduli matvec h={h} {dims}", flush=True)
    rng = np.random.default_rng(3)
    model = "thermal" if h == 1 else "elastic"
    _, groups = _groups(model, 3, rng)
    ms = rng.integers(0, 3, size=dims).astype(np.uint16)
    p = Problem(dims=dims, howmany=h, ms=ms, groups=groups, fe_type="HEX8", method="cg", L=L, tol=1e-10, n_it=10)
    u = rng.standard_normal(dims + (h,)) * 0.01
    k_o = oracle.Oracle(p).residual(u, linear_kd=True)
    for precision in ("fp64", "mixed"):
        g = gpu.GpuSolver(p, precision=precision)
        try:
            pr = groups[0].param_matrix()
            g.set_voxel_moduli(pr[ms, 0], None if h == 1 else pr[ms, 1])
            assert relerr(g.residual(u, linear_kd=True), k_o) < 1e-12
            if precision == "mixed":
                g.set_operator_fp32(True)
                assert relerr(g.residual(u, linear_kd=True), k_o) < 1e-5
        finally:
            g.close()
