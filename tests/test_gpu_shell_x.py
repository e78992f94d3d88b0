"""GPU test of the shell fields' x pass, whose last FFT stage stores to the fields,
on every value: first shells, last shells, tiles with fewer row pairs (N = 48, 360),
an LDS path for the sizes that have no compile-time length (N = 90).

Tolerance: float32 FFT rounding 2e-6, float64 1e-12 of the largest value."""
import pytest
import torch

from pyspectrum_amd import _lib as L

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N,step,ncut,nmax", [(32, 1, 1, 2), (48, 2, 4, 12), (64, 1, 30, 32),
                                              (90, 3, 3, 6), (128, 3, 3, 5), (360, 4, 40, 11),
                                              (512, 3, 3, 3)])
def test_shell_fields_by_value(N, step, ncut, nmax, prec):
    print("[case] shell x", N, step, ncut, nmax, prec, flush=True)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(N)
    real = torch.randn((N, N, N), generator=gen, device=DEV, dtype=torch.float64)
    half = torch.fft.rfftn(real) / N ** 1.5
    cd, rd = ((torch.complex128, torch.float64) if prec == "fp64"
              else (torch.complex64, torch.float32))
    half = half.to(cd).contiguous()
    j0 = ncut // step
    D = torch.empty((nmax - j0 + 1, N, N, N), dtype=rd, device=DEV)
    ctx = L.Context(0)
    ctx.call("psx_bk_shell_fields", L.ptr(half), N, step, ncut, nmax, L.ptr(D), L.PREC[prec])
    f = torch.fft.fftfreq(N, d=1.0 / N, device=DEV, dtype=torch.float64)
    m = f[:, None, None] ** 2 + f[None, :, None] ** 2 + f[None, None, :N // 2 + 1] ** 2
    tol = 1e-12 if prec == "fp64" else 2e-6
    for j in range(j0, nmax + 1):
        # shell j: (2 j - 1) step <= 2 |k| < (2 j + 1) step
        lo, hi = ((2 * j - 1) * step) ** 2, ((2 * j + 1) * step) ** 2
        mask = (4 * m < hi) & ((4 * m >= lo) if j else (m >= 0))
        ref = torch.fft.irfftn(torch.where(mask, half.to(torch.complex128).conj(), 0),
                               s=(N,) * 3) * N ** 3
        assert float((D[j - j0].double() - ref).abs().max()) <= tol * float(ref.abs().max())
    ctx.close()
