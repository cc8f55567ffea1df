"""Error norm and scalar products of the z passes whose workgroups end in a
partial wavefront (144 threads at n_z = 48 and 96, 240 and 160 at 80): the error
history of the first CG iterations in every measure against the oracle, with the
only inclusion, and so the residual's peak, in the nodes those last lanes hold; the
linear CG with folded scalars and with reduction launches, and the nonlinear CG.

Tolerance: sums of n = 4e3 .. 2e4 terms differ by 1e-16 sqrt(n) < 1e-13 relative,
and k <= 6 steps amplify that by no more than about the condition number (1e2 at a
contrast of ten): 1e-10 of each error.  Nonlinear CG: a secant quotient a step,
1e-8, the bound of the load-step tests."""
import numpy as np
import pytest

import oracle
from fans_amd import gpu
from fans_amd.problem import MaterialGroup, Problem
from tests import cases

pytestmark = pytest.mark.gpu

#: the inclusion's z range, among the nodes of the workgroups' last wavefronts
_LAYERS = {(48, 3): (43, 47), (96, 3): (44, 47), (80, 3): (66, 72), (80, 1): (60, 66), (48, 1): (20, 24)}


def _microstructure(dims, h):
    ms = np.zeros(dims, dtype=np.uint16)
    z0, z1 = _LAYERS[dims[2], h]
    ms[2:5, 3:6, z0:z1] = 1
    return ms


@pytest.mark.parametrize("chunks", [1, 2])  # folded scalars, reduction launches
@pytest.mark.parametrize("measure", ["Linfinity", "L1", "L2"])
@pytest.mark.parametrize("dims,h", [((8, 8, 48), 3), ((8, 16, 96), 3), ((8, 8, 80), 3), ((8, 8, 80), 1), ((8, 8, 48), 1)])
def test_error_history_matches_oracle(dims, h, measure, chunks):
    print(f"[gpu-case] error history {dims} h={h} {measure} chunks={chunks}", flush=True)
    groups = [MaterialGroup("LinearThermalIsotropic", [0, 1], {"conductivity": [1.0, 10.0]}) if h == 1 else
              MaterialGroup("LinearElasticIsotropic", [0, 1], {"bulk_modulus": [3.0, 30.0], "shear_modulus": [1.0, 10.0]})]
    p = Problem(dims=dims, howmany=h, ms=_microstructure(dims, h), groups=groups, fe_type="HEX8", method="cg",
                L=tuple(float(n) for n in dims), tol=1e-300, n_it=6, measure=measure, err_type="absolute")
    g0 = [0.01] + [0.0] * (p.n_str - 2) + [0.02]
    o, g = oracle.Oracle(p), gpu.GpuSolver(p)
    try:
        g.set_fft_chunks(chunks)
        o.set_gradient(g0)
        g.set_gradient(g0)
        assert g.solve() == o.solve() == 6
        ho, hg = np.asarray(o.error_history()), g.error_history()
        assert hg.shape == ho.shape
        assert np.max(np.abs(hg - ho) / ho) < 1e-10
    finally:
        g.close()


@pytest.mark.parametrize("nz", [48, 80])
def test_nonlinear_error_history_matches_oracle(nz):
    print(f"[gpu-case] nonlinear error history nz={nz}", flush=True)
    p = cases.j2(dims=(8, 8, nz), seed=1, count=1, rmin=2.0, rmax=3.0)
    p.ms = _microstructure(p.dims, 3)
    p.n_it, p.tol = 4, 1e-300
    g0 = [0.004, 0.0, -0.001, 0.0, 0.002, 0.0]
    o, g = oracle.Oracle(p), gpu.GpuSolver(p)
    try:
        o.set_gradient(g0)
        g.set_gradient(g0)
        assert g.solve() == o.solve() == 4
        ho, hg = np.asarray(o.error_history()), g.error_history()
        assert hg.shape == ho.shape
        assert np.max(np.abs(hg - ho) / ho) < 1e-8
    finally:
        g.close()
