"""GPU test of the FP64 triangle sums on their point sets (cubic grids below
N^3, half-cell copies, the direct sums of a few aliased triangles): the sums
of psx_bk_raw against the general path, the shell fields on the N^3 grid and
their contraction, on the same half field.

Tolerance: both sides are float64 FFTs (relative rounding of a field value
below 1e-14) and sums; a sum of three-field products is compared with the sum
of their absolute values, 1e-13."""
import numpy as np
import pytest
import torch

from pyspectrum_amd import _lib as L

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
F64 = L.PREC["fp64"]


@pytest.mark.parametrize("N,step,ncut,nmax", [
    (48, 1, 1, 7), (128, 6, 6, 5), (144, 4, 8, 8), (180, 4, 4, 11), (192, 2, 2, 19),
    (240, 3, 0, 20), (300, 3, 3, 30), (30, 1, 1, 4), (64, 1, 1, 31),
])
def test_layer_sums_match_grid_sums(N, step, ncut, nmax):
    print("[case] layers", N, step, ncut, nmax, flush=True)
    ctx = L.Context(0)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(N + nmax)
    half = torch.randn((N, N, N // 2 + 1), generator=gen, device=DEV, dtype=torch.complex128)
    ijl = L.triangles(step, ncut, nmax)
    ntri, ns = len(ijl), nmax - ncut // step + 1
    got = torch.empty(ntri, dtype=torch.float64, device=DEV)
    p0k = torch.empty(nmax, dtype=torch.float64, device=DEV)
    ctx.call("psx_bk_raw", L.ptr(half), N, step, ncut, nmax, L.ptr(got), L.ptr(p0k), F64)
    D = torch.empty((ns, N ** 3), dtype=torch.float64, device=DEV)
    ctx.call("psx_bk_shell_fields", L.ptr(half), N, step, ncut, nmax, L.ptr(D), F64)
    ref = torch.empty(ntri, dtype=torch.float64, device=DEV)
    ctx.call("psx_bk_contract", L.ptr(D), N, step, ncut, nmax, L.ptr(ref), F64)
    scale = torch.empty_like(ref)
    A = D.abs()
    ctx.call("psx_bk_contract", L.ptr(A), N, step, ncut, nmax, L.ptr(scale), F64)
    got, ref, scale = (t.cpu().numpy() for t in (got, ref, scale))
    assert np.all(np.isfinite(got))
    assert np.all(np.abs(got - ref) <= 1e-13 * scale), np.max(np.abs(got - ref) / scale)
    again = torch.empty(ntri, dtype=torch.float64, device=DEV)
    ctx.call("psx_bk_raw", L.ptr(half), N, step, ncut, nmax, L.ptr(again), L.ptr(p0k), F64)
    assert np.array_equal(again.cpu().numpy(), got)
    ctx.close()
