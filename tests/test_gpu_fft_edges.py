"""The staged FFT passes and the x+Green pass at the lengths where their stage
plans and tiles can go wrong: one stage (2, 3, 5), two, three and four stages,
lengths above 256, odd lengths (the Green operator stored in full), columns and
frequencies that do not fill the last tile, both component counts and
precisions, and LDS budgets that force the narrowest tiles.

Tolerances, relative to the field's maximum: a transform rounds a value in about
log2(N) < 20 butterfly levels at 1.1e-16 each, with growth sqrt(log2 N), so 1e-13
for FP64 transforms.  The convolution adds the operator's entries, whose smallest
frequency cancels 1 - cos(2 pi / n) on both sides: 1e-12 + 2e-16 n^2.  FP32 1e-5
(20 levels and the 3x3 product at 6e-8, the operator itself rounded once)."""
import numpy as np
import pytest

import oracle
from fans_amd import gpu
from fans_amd.problem import MaterialGroup, Problem

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return float(np.max(np.abs(np.asarray(a) - np.asarray(b))) / np.max(np.abs(b)))


@pytest.mark.parametrize("shape", [(2, 3, 4, 3), (3, 5, 2, 1), (5, 2, 6, 3), (4, 125, 10, 3),
                                   (9, 250, 30, 3), (15, 375, 18, 1), (2, 1000, 8, 1), (2, 1280, 4, 3),
                                   (27, 12, 1000, 1), (60, 45, 400, 3), (375, 4, 12, 1), (540, 2, 6, 3)])
def test_transform_edge_lengths(shape):
    print(f"[gpu-case] fft {shape}", flush=True)
    x = np.random.default_rng(5).standard_normal(shape)
    ref = np.fft.rfftn(x, axes=(0, 1, 2))
    assert relerr(gpu.fft_r2c(x), ref) < 1e-13
    back = np.fft.irfftn(ref, s=shape[:3], axes=(0, 1, 2)) * np.prod(shape[:3])
    assert relerr(gpu.fft_c2r(ref, shape[2]), back) < 1e-13


@pytest.mark.parametrize("kind,dims", [
    ("elastic", (2, 3, 4)), ("elastic", (3, 2, 6)), ("elastic", (5, 5, 10)), ("elastic", (6, 10, 30)),
    ("elastic", (12, 15, 8)), ("elastic", (20, 9, 48)), ("elastic", (45, 6, 20)), ("elastic", (125, 4, 6)),
    ("elastic", (144, 3, 10)), ("elastic", (250, 2, 12)), ("elastic", (320, 2, 4)), ("elastic", (64, 48, 20)),
    ("thermal", (2, 2, 2)), ("thermal", (5, 3, 4)), ("thermal", (27, 10, 18)), ("thermal", (80, 96, 12)),
    ("thermal", (375, 3, 8)), ("thermal", (16, 25, 32)),
])
def test_convolution_edge_lengths(kind, dims):
    print(f"[gpu-case] convolve {kind} {dims}", flush=True)
    thermal = kind == "thermal"
    ms = np.random.default_rng(3).integers(0, 2, size=dims).astype(np.uint16)
    groups = [MaterialGroup("LinearThermalIsotropic", [0, 1], {"conductivity": [1.0, 10.0]}) if thermal else
              MaterialGroup("LinearElasticIsotropic", [0, 1], {"bulk_modulus": [3.0, 40.0], "shear_modulus": [1.0, 28.0]})]
    p = Problem(dims=dims, howmany=1 if thermal else 3, ms=ms, groups=groups, fe_type="HEX8", method="cg",
                L=tuple(float(n) for n in dims), tol=1e-10, n_it=10)
    r = np.random.default_rng(7).standard_normal(dims + (p.howmany,))
    o, g = oracle.Oracle(p), gpu.GpuSolver(p, precision="mixed")
    try:
        ref, tol = o.convolve(r), 1e-12 + 2e-16 * max(dims) ** 2
        for kib in (None, 8, 64):
            if kib:
                g.set_fft_lds_kib(kib)
            g.set_operator_fp32(False)
            assert relerr(g.convolve(r), ref) < tol, kib
            g.set_operator_fp32(True)
            assert relerr(g.convolve(r), ref) < 1e-5, kib
    finally:
        g.close()
