"""GPU test of the two workgroup widths of the double assignment at run-time
lengths of 257 to 512 tiles, either side of one particle a cell and at the
lengths whose tile counts surround 256: the field of psx_fft_periodic against
the stages (psx_assign_quad, psx_fft3d, psx_fcomb_periodic), every element.

Tolerance: both sides add the same integers; the float64 FFTs' rounding, 1e-12
of the largest element."""
import numpy as np
import pytest
import torch

from pyspectrum_amd import _lib as L

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("N,n", [(40, 3000), (50, 0), (50, 1), (50, 50 ** 3 - 1), (50, 50 ** 3),
                                 (60, 5000), (60, 60 ** 3), (60, 60 ** 3 + 257)])
def test_double_runtime_lengths_match_stages(N, n):
    print("[case] double assignment width", N, n, flush=True)
    Lbox, p = 100.0, L.PREC["fp64"]
    rng = np.random.default_rng(N + n)
    x = torch.from_numpy(rng.uniform(0, Lbox, size=(3, n)).astype(np.float32)).to(DEV)
    ctx = L.Context(0)
    got = torch.empty((N, N, N // 2 + 1), dtype=torch.complex128, device=DEV)
    sumw = float(max(n, 1))
    ctx.call("psx_fft_periodic", L.ptr(x), None, n, N, Lbox, sumw, sumw, L.ptr(got), p)
    grid = torch.empty((N, N, N), dtype=torch.complex128, device=DEV)
    ref = torch.empty_like(got)
    ctx.call("psx_assign_quad", L.ptr(x), None, n, N, float(np.float32(N / Lbox)), 0.0, 0.0,
             float(np.float32(Lbox * (1 - 1e-6))), sumw, L.ptr(grid), p)
    ctx.call("psx_fft3d", L.ptr(grid), N, 1, p)
    ctx.call("psx_fcomb_periodic", L.ptr(grid), L.ptr(ref), N, sumw, p)
    assert float((got - ref).abs().max()) <= 1e-12 * float(ref.abs().max())
    ctx.close()
