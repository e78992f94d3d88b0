"""GPU test of the z pass with fcomb as its epilogue (psx_fft_periodic) against
the separate stages (psx_assign_quad, psx_fft3d, psx_fcomb_periodic), on every
element: the planes 0 and N/2, where indices alias and one store survives, odd
numbers of line pairs in the last tile, and tiles of 6 to 16 lines.

Tolerance: the same sums through other kernels; float32 FFT rounding 2e-6,
float64 1e-12 of the largest element."""
import numpy as np
import pytest
import torch

from pyspectrum_amd import _lib as L

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N", [4, 6, 18, 54, 96, 150, 128, 640])
def test_fused_z_pass_matches_stages(N, prec):
    print("[case] zcomb", N, prec, flush=True)
    Lbox, n = 100.0, 20000
    gen = torch.Generator(device=DEV)
    gen.manual_seed(N)
    xyz = torch.rand((3, n), generator=gen, device=DEV) * Lbox
    cd = torch.complex128 if prec == "fp64" else torch.complex64
    p = L.PREC[prec]
    ctx = L.Context(0)
    got = torch.empty((N, N, N // 2 + 1), dtype=cd, device=DEV)
    ctx.call("psx_fft_periodic", L.ptr(xyz), None, n, N, Lbox, float(n), float(n), L.ptr(got), p)
    grid = torch.empty((N, N, N), dtype=cd, device=DEV)
    ref = torch.empty_like(got)
    ctx.call("psx_assign_quad", L.ptr(xyz), None, n, N, float(np.float32(N / Lbox)), 0.0, 0.0,
             float(np.float32(Lbox * (1 - 1e-6))), float(n), L.ptr(grid), p)
    ctx.call("psx_fft3d", L.ptr(grid), N, 1, p)
    ctx.call("psx_fcomb_periodic", L.ptr(grid), L.ptr(ref), N, float(n), p)
    tol = (1e-12 if prec == "fp64" else 2e-6) * float(ref.abs().max())
    assert float((got - ref).abs().max()) <= tol
    ctx.close()
