"""GPU test of the FFT engine at lengths without a compile-time instantiation
(one wave per line): every radix as the first, a middle and the last stage,
fewer butterflies than lanes, exact and ragged passes of 64, the longest
lengths.

Tolerance: float32 FFT rounding, about 2^-24 sqrt(log2 N^3) relative to the rms
of the result and five to six times that for the largest element: 5e-6 of the
rms scale N^1.5; float64 the same with 2^-53: 1e-14."""
import pytest
import torch

from pyspectrum_amd import _lib as L

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
TOL = {"fp32": 5e-6, "fp64": 1e-14}


def _grid(N, prec, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    cd = torch.complex128 if prec == "fp64" else torch.complex64
    return torch.randn((N, N, N), generator=gen, device=DEV, dtype=cd)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N", [4, 6, 10, 18, 50, 54, 100, 150, 162, 250, 320])
def test_fft3d_runtime_length(N, prec):
    print("[case] fft runtime", N, prec, flush=True)
    x = _grid(N, prec, N)
    for sign, fn in ((1, torch.fft.ifftn), (-1, torch.fft.fftn)):
        g = x.clone()
        L.context(0).call("psx_fft3d", L.ptr(g), N, sign, L.PREC[prec])
        ref = fn(x.to(torch.complex128), norm="forward" if sign > 0 else "backward")
        err = float((g.to(torch.complex128) - ref).abs().max())
        assert err <= TOL[prec] * N ** 1.5, (sign, err / N ** 1.5)


@pytest.mark.parametrize("N,prec", [(1000, "fp32"), (640, "fp64"), (972, "fp32")])
def test_fft3d_long_lengths_round_trip(N, prec):
    print("[case] fft round trip", N, prec, flush=True)
    x = _grid(N, prec, N)
    g = x.clone()
    for sign in (1, -1):
        L.context(0).call("psx_fft3d", L.ptr(g), N, sign, L.PREC[prec])
    g /= N ** 3
    assert float((g - x).abs().max()) <= 2 * TOL[prec]
