"""Nonlinear CG whose stop test, controller and line-search scalars stay on the
device: runs cut after a few iterations (the launches queued behind a stop test
must do nothing: displacement, gradient and the per-call visco-plastic update), a
strain-controlled run, and one that has converged before its first iteration,
against the oracle.

Tolerance: 1e-8 of each quantity's maximum, the bound of the other load-step tests
(rounding 1e-16 through at most 8 secant searches, each dividing by a difference
of two products that agree to 1e-3 or so)."""
import numpy as np
import pytest

import oracle
from fans_amd import gpu
from tests import cases
from tests.test_gpu_visco import visco_problem

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return float(np.max(np.abs(np.asarray(a) - np.asarray(b))) / max(np.max(np.abs(b)), 1e-300))


def _problem(kind, ms):
    if kind == "visco":
        return visco_problem(ms, True, Kh=0.3, Hk=0.2)
    return cases.j2(dims=(10, 18, 16), seed=2, count=5, rmin=2.0, rmax=4.0)


@pytest.mark.parametrize("kind,n_it", [("j2", 1), ("j2", 2), ("j2", 8), ("visco", 1), ("visco", 3)])
def test_cut_runs_match_oracle(kind, n_it, sphere32_ms):
    print(f"[gpu-case] nonlinear cut run {kind} n_it={n_it}", flush=True)
    p = _problem(kind, sphere32_ms)
    p.n_it, p.tol = n_it, 1e-300
    mbc = cases.uniaxial_mixed(2, 0.02 if kind == "j2" else 0.006)
    o, g = oracle.Oracle(p), gpu.GpuSolver(p)
    try:
        for t in range(2):
            o.enable_mixed_bc(mbc, t)
            g.enable_mixed_bc(mbc, t)
            assert g.solve() == o.solve() == n_it
            assert relerr(g.macro_gradient(), o.macro_gradient()) < 1e-8, t
            assert relerr(g.get_u(), o.get_u()) < 1e-8, t
            assert relerr(g.homogenized_stress(), o.homogenized_stress()) < 1e-8, t
    finally:
        g.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_strain_control_and_converged_start(precision):
    print(f"[gpu-case] nonlinear strain control {precision}", flush=True)
    p = cases.j2(dims=(9, 16, 12), seed=3, count=4, rmin=2.0, rmax=3.0)
    g0 = [0.004, 0.0, -0.001, 0.0, 0.002, 0.0]
    o, g = oracle.Oracle(p), gpu.GpuSolver(p, precision=precision)
    try:
        o.set_gradient(g0)
        g.set_gradient(g0)
        o.solve()
        g.solve()
        assert relerr(g.homogenized_stress(), o.homogenized_stress()) < 1e-8
        u = g.get_u().copy()
        assert g.solve() == 0  # the residual at the solution is below the tolerance already
        assert np.array_equal(g.get_u(), u)
        assert relerr(g.macro_gradient(), g0) < 1e-15
    finally:
        g.close()


@pytest.mark.parametrize("timing", [False, True])
@pytest.mark.parametrize("mixed_bc", [False, True])
def test_iterations_and_history_of_the_stopping_iteration(mixed_bc, timing):
    """The host takes the stop flag and the iteration from memory that the device
    writes: read before the stream is waited for, a run could report the iteration
    before its last.  Runs cut at n_it and one to convergence, many of each, on a grid
    whose kernels end before the host looks; exact comparisons only."""
    print(f"[gpu-case] nonlinear stop, mixed_bc={mixed_bc} timing={timing}", flush=True)
    p = cases.j2(dims=(4, 6, 8), seed=3, count=1, rmin=1.0, rmax=1.5)
    for n_it in (1, 2, 3, 300):
        p.n_it, p.tol = n_it, (1e-300 if n_it < 300 else 1e-9)
        g = gpu.GpuSolver(p, timing=timing)
        try:
            first = None
            for _ in range(25):
                g.reset_state()
                if mixed_bc:
                    g.enable_mixed_bc(cases.uniaxial_mixed(2, 0.02), 0)
                else:
                    g.set_gradient([0.004, 0.0, -0.001, 0.0, 0.002, 0.0])
                n, h = g.solve(), g.error_history().copy()
                assert h.shape == (n + 1,) and (h > 0.0).all()
                assert h[-1] == g.stats.final_error
                assert bool(g.stats.converged) == (h[-1] <= p.tol)
                if n_it < 300:
                    assert n == n_it
                else:
                    assert g.stats.converged and (h[:-1] > p.tol).all()
                if first is None:
                    first = h
                assert np.array_equal(h, first)
        finally:
            g.close()
