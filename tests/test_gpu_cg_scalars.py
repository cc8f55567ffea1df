"""Linear CG whose z passes fold the reduction scalars against the same CG with
reduction launches (a grid with its FFT in two kz chunks takes those): every
error measure, workgroups of whole and of partial wavefronts, runs stopped before,
at and after a turn of the direction ring, a mixed solve that continues its
inner loop, and a grid past the partials limit.

Tolerance: the two differ in the order of sums alone, 1e-16 sqrt(n) < 1e-13 per
scalar; within k <= 40 steps CG amplifies a relative change by no more than about
the condition number (1e3 here), so 1e-9 of each quantity's maximum; after a mixed
solve, 1e-7 (FP32 steps at 6e-8 between FP64 residuals)."""
import numpy as np
import pytest

from fans_amd import gpu
from fans_amd.problem import MaterialGroup, Problem

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return float(np.max(np.abs(np.asarray(a) - np.asarray(b))) / np.max(np.abs(b)))


def _problem(kind, dims, measure, err_type, tol, n_it):
    thermal = kind == "thermal"
    ms = np.random.default_rng(3).integers(0, 2, size=dims).astype(np.uint16)
    groups = [MaterialGroup("LinearThermalIsotropic", [0, 1], {"conductivity": [1.0, 10.0]}) if thermal else
              MaterialGroup("LinearElasticIsotropic", [0, 1], {"bulk_modulus": [3.0, 40.0], "shear_modulus": [1.0, 28.0]})]
    return Problem(dims=dims, howmany=1 if thermal else 3, ms=ms, groups=groups, fe_type="HEX8", method="cg",
                   L=tuple(float(n) for n in dims), tol=tol, n_it=n_it, measure=measure, err_type=err_type)


def _run(p, precision, chunks):
    g = gpu.GpuSolver(p, precision=precision)
    try:
        if chunks > 1:
            g.set_fft_chunks(chunks)
        out = []
        for s in (0.01, -0.02):  # twice on one context: captured iterations are replayed
            g.reset_state()
            g.set_gradient([s] + [0.0] * (p.n_str - 1))
            g.solve()
            out.append((int(g.stats.inner_iterations), g.error_history().copy(), g.get_u().copy()))
        return out
    finally:
        g.close()


@pytest.mark.parametrize("kind,dims,measure,n_it", [
    ("elastic", (8, 6, 10), "Linfinity", 1), ("elastic", (12, 10, 16), "L2", 7), ("elastic", (12, 10, 32), "L1", 8),
    ("elastic", (9, 8, 48), "Linfinity", 9), ("elastic", (16, 8, 80), "L2", 16), ("elastic", (16, 16, 96), "L1", 17),
    ("thermal", (6, 5, 4), "L1", 8), ("thermal", (16, 16, 80), "Linfinity", 23), ("thermal", (32, 32, 32), "L2", 24),
    ("thermal", (25, 24, 18), "Linfinity", 25), ("thermal", (160, 160, 10), "L2", 9),
])
def test_folded_scalars_match_reductions(kind, dims, measure, n_it):
    print(f"[gpu-case] folded CG scalars {kind} {dims} {measure} {n_it}", flush=True)
    p = _problem(kind, dims, measure, "absolute", 1e-300, n_it)
    for (ka, ha, ua), (kb, hb, ub) in zip(_run(p, "fp64", 1), _run(p, "fp64", 2)):
        assert ka == kb == n_it
        assert relerr(ha, hb) < 1e-9
        assert relerr(ua, ub) < 1e-9


@pytest.mark.parametrize("kind,dims", [("elastic", (16, 16, 48)), ("thermal", (20, 18, 24)), ("elastic", (12, 10, 6))])
def test_folded_scalars_in_mixed_solves(kind, dims):
    print(f"[gpu-case] folded CG scalars, mixed {kind} {dims}", flush=True)
    p = _problem(kind, dims, "Linfinity", "relative", 1e-9, 200)
    for (ka, ha, ua), (kb, hb, ub) in zip(_run(p, "mixed", 1), _run(p, "mixed", 2)):
        assert abs(ka - kb) <= 2
        assert relerr(ua, ub) < 1e-7


@pytest.mark.parametrize("kind,precision", [("elastic", "fp64"), ("elastic", "mixed"), ("thermal", "fp64")])
def test_batch_past_the_fold_limit_matches_single_solves(kind, precision):
    """A batch whose workgroups would read more partials than folding pays for
    launches reductions in the folded order: bit for bit the single solves, which
    fold (144-, 192-thread and generic z passes)."""
    dims, n = {"elastic": ((96, 96, 48), 4), "thermal": ((160, 160, 10), 3)}[kind]
    print(f"[gpu-case] batch past the fold limit {kind} {precision} {dims} x {n}", flush=True)
    ps = []
    for s in range(n):
        p = _problem(kind, dims, "Linfinity", "absolute", 1e-300, 9)
        p.ms = np.random.default_rng(s).integers(0, 2, size=dims).astype(np.uint16)
        ps.append(p)
    g0 = [0.01] + [0.0] * (ps[0].n_str - 1)
    single = []
    for p in ps:
        g = gpu.GpuSolver(p, precision=precision)
        try:
            g.set_gradient(g0)
            g.solve()
            single.append((int(g.stats.inner_iterations), g.homogenized_stress().copy(), g.get_u().copy()))
        finally:
            g.close()
    b = gpu.GpuBatch(ps, precision=precision)
    try:
        for k, p in enumerate(ps):
            b.load_slot(k, p, g0)
        b.solve()
        its = b.results()[0]
        st = b.stresses()
        for k in range(n):
            assert its[k] == single[k][0]
            assert np.array_equal(st[k], single[k][1])
            b.select(k)
            assert np.array_equal(b.get_u(), single[k][2])
    finally:
        b.close()
