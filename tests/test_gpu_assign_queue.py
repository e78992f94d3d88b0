"""GPU test of the assignment's list of (particle, grid, z row) entries against
the oracle: counts around the 256 particles and entries of one pass over the
list, points of one tile (entries carried from pass to pass), grids whose
stencils wrap onto most tiles, and weights of both signs.

Tolerance: float64 stencils and the 2^-40 fixed point 1e-11; float32 stencil
products (four roundings each) 5e-7 of the field's norm."""
import numpy as np
import pytest
import torch

from oracle import spectrum as S
from pyspectrum_amd import _lib as L

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N,n,tile", [(4, 1, False), (4, 257, False), (6, 255, False),
                                      (6, 256, True), (20, 1023, True), (20, 3000, False),
                                      (48, 64, False), (48, 1500, True)])
def test_assignment_list_edges(N, n, tile, prec):
    print("[case] assignment list", N, n, tile, prec, flush=True)
    Lbox = 200.0
    rng = np.random.default_rng(N + n)
    xyz = rng.uniform(0, Lbox, size=(3, n))
    if tile:
        xyz[1:] *= 2.0 / N   # y and z in the first two cells
    w = rng.uniform(0.5, 1.5, size=n) * rng.choice([-1.0, 1.0], size=n, p=[0.2, 0.8])
    kf_ks = np.float32(N / Lbox)
    A, B = S.assign_quad(S.clip_positions(xyz, Lbox), w.astype(np.float32).astype(np.float64), N,
                         kf_ks)
    x = torch.from_numpy(np.ascontiguousarray(xyz.astype(np.float32))).to(DEV)
    wd = torch.from_numpy(w.astype(np.float32)).to(DEV)
    g = torch.empty((N, N, N), dtype=torch.complex128 if prec == "fp64" else torch.complex64,
                    device=DEV)
    ctx = L.Context(0)
    ctx.call("psx_assign_quad", L.ptr(x), L.ptr(wd), n, N, float(kf_ks), 0.0, 0.0,
             float(np.float32(Lbox * (1 - 1e-6))), float(np.abs(w).sum()), L.ptr(g), L.PREC[prec])
    out = g.cpu().numpy().transpose(2, 1, 0)
    ctx.close()
    tol = 1e-11 if prec == "fp64" else 5e-7
    for got, ref in ((out.real, A), (out.imag, B)):
        assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N,n,tile", [(4, 1025, False), (32, 1, False), (40, 1023, True),
                                      (40, 30000, True), (64, 5000, False), (72, 5000, False)])
def test_small_grids_match_stages(N, n, tile, prec):
    """The assignment with the x pass, in wide workgroups up to N = 64, against
    psx_assign_quad and psx_fft3d on every element (float32 FFT rounding 2e-6,
    float64 1e-12 of the largest)."""
    print("[case] small grid", N, n, tile, prec, flush=True)
    Lbox = 100.0
    rng = np.random.default_rng(N + n)
    xyz = rng.uniform(0, Lbox, size=(3, n))
    if tile:
        xyz[1:] *= 2.0 / N
    x = torch.from_numpy(xyz.astype(np.float32)).to(DEV)
    cd = torch.complex128 if prec == "fp64" else torch.complex64
    p = L.PREC[prec]
    ctx = L.Context(0)
    got = torch.empty((N, N, N // 2 + 1), dtype=cd, device=DEV)
    ctx.call("psx_fft_periodic", L.ptr(x), None, n, N, Lbox, float(n), float(n), L.ptr(got), p)
    grid = torch.empty((N, N, N), dtype=cd, device=DEV)
    ref = torch.empty_like(got)
    ctx.call("psx_assign_quad", L.ptr(x), None, n, N, float(np.float32(N / Lbox)), 0.0, 0.0,
             float(np.float32(Lbox * (1 - 1e-6))), float(n), L.ptr(grid), p)
    ctx.call("psx_fft3d", L.ptr(grid), N, 1, p)
    ctx.call("psx_fcomb_periodic", L.ptr(grid), L.ptr(ref), N, float(n), p)
    tol = (1e-12 if prec == "fp64" else 2e-6) * float(ref.abs().max())
    assert float((got - ref).abs().max()) <= tol
    ctx.close()
