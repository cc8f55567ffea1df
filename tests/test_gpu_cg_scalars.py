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


def test_mixed_batch_that_falls_below_the_fold_limit_matches_single_solves():
    """Five slots of 128 x 128 x 10 elasticity launch reductions, three or fewer of
    them alone would fold (their workgroups read 2.5 million partials per slot and
    iteration).  Slots of small load end after the first FP32 phase, slots of low
    contrast leave the map early within a phase, and later solves on the same context
    run two slots, one, and all of them again (captured iterations of every depth are
    replayed).  Each slot is bit for bit its single solve, and meets the tolerance."""
    dims, big, small = (128, 128, 10), 1e-2, 1e-8
    contrast = [1.2, 1.2, 8.0, 60.0, 60.0]
    ps = []
    for s, f in enumerate(contrast):
        p = _problem("elastic", dims, "Linfinity", "absolute", 1e-10, 400)
        p.ms = np.random.default_rng(s).integers(0, 2, size=dims).astype(np.uint16)
        p.groups = [MaterialGroup("LinearElasticIsotropic", [0, 1], {"bulk_modulus": [1.0, f], "shear_modulus": [0.6, 0.6 * f]})]
        ps.append(p)
    load = lambda a: [a] + [0.0] * 5
    runs = [[small, small, big, big, big], [0.0, 0.0, 0.0, big, big], [0.0, 0.0, 0.0, 0.0, big],
            [big, small, big, small, big]]
    single = {}
    for k, a in sorted({(k, a) for r in runs for k, a in enumerate(r) if a}):
        print(f"[gpu-case] single mixed solve, slot {k} load {a}", flush=True)
        g = gpu.GpuSolver(ps[k], precision="mixed")
        try:
            g.set_gradient(load(a))
            g.solve()
            assert g.stats.converged
            single[k, a] = (int(g.stats.inner_iterations), g.homogenized_stress().copy(), g.get_u().copy())
        finally:
            g.close()
    b = gpu.GpuBatch(ps, precision="mixed")
    try:
        for r in runs:
            print(f"[gpu-case] mixed batch below the fold limit, loads {r}", flush=True)
            for k, p in enumerate(ps):
                b.load_slot(k, p, load(r[k]))
            b.solve()
            its, conv, _ = b.results()
            its, conv, st = list(its), list(conv), b.stresses()
            assert all(conv)
            for k, a in enumerate(r):
                b.select(k)
                u = b.get_u()
                if not a:
                    assert its[k] == 0 and not u.any()
                    continue
                assert its[k] == single[k, a][0]
                assert np.array_equal(st[k], single[k, a][1])
                assert np.array_equal(u, single[k, a][2])
    finally:
        b.close()
