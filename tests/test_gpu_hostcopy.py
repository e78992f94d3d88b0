"""GPU test of the host side of the entry points: the copy of device tensors to
host memory (exact at the edges of the chunks that go through the pinned buffers,
on a stream that is not the default one, with the strides the half field has),
the weight sums of several boxes, and the check of the redshifts."""
import numpy as np
import pytest
import torch

from pyspectrum_amd import _lib as L
from pyspectrum_amd import pyspectrum as P

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
PER = L.COPY_CHUNK // 8


@pytest.mark.parametrize("n", [0, 1, PER // 2 - 1, PER // 2, PER - 1, PER, PER + 1, 2 * PER,
                               3 * PER + 5])
def test_copy_to_host_is_exact(n):
    print("[case] host copy", n, flush=True)
    stream = torch.cuda.Stream(device=DEV)
    with torch.cuda.stream(stream):
        t = torch.view_as_complex(torch.randn((n, 2), device=DEV))
        got = L.to_numpy(t)
        t.add_(1.0)  # after the copy
    stream.synchronize()
    assert got.dtype == np.complex64 and got.shape == (n,) and got.flags.writeable
    assert np.array_equal(got + np.complex64(1.0), t.cpu().numpy())


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_half_field_layout(prec):
    print("[case] half field layout", prec, flush=True)
    xyz = np.random.default_rng(1).uniform(0, 100.0, size=(3, 5000))
    N = 128
    got = P.FFT_periodic(xyz, Lbox=100.0, Ngrid=N, precision=prec)
    half = P._half_on_device(xyz, None, 100.0, N, L.PREC[prec], 0)[0]
    ref = half.permute(2, 1, 0).cpu().numpy()
    assert got.strides == ref.strides and np.array_equal(got, ref)
    full = P.reflect_delta(got, Ngrid=N)
    assert full.flags.c_contiguous and np.array_equal(full[1:N // 2], got[1:N // 2])


def test_weight_sums_of_a_list():
    print("[case] weight sums", flush=True)
    rng = np.random.default_rng(2)
    w = [rng.normal(size=n) for n in (1000, 7, 333, 50)]
    ws = [torch.from_numpy(w[0]).to(DEV), w[1], None, torch.from_numpy(w[2]),
          torch.from_numpy(w[3].astype(np.float32)).to(DEV)]
    got = P._weights_list(ws, [1000, 7, 12, 333, 50], 0)
    for (wd, s, a), ref in zip(got, [w[0], w[1], np.ones(12), w[2], w[3].astype(np.float32)]):
        ref = ref.astype(np.float64)
        assert abs(s - ref.sum()) <= 1e-13 * np.abs(ref).sum()
        assert abs(a - np.abs(ref).sum()) <= 1e-13 * np.abs(ref).sum()
        assert wd is None or np.array_equal(wd.cpu().numpy(), ref.astype(np.float32))


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, -1e-9])
def test_redshifts_are_checked(bad):
    print("[case] redshifts", bad, flush=True)
    rng = np.random.default_rng(3)
    cat = np.array([rng.uniform(0, 90, 5000), rng.uniform(-30, 30, 5000),
                    rng.uniform(0.2, 0.4, 5000)])
    cat[2, 4321] = bad
    with pytest.raises(ValueError, match="redshifts"):
        P.FFT_survey_mono(cat, np.full(5000, 1e-4), Lbox=3600.0, Ngrid=32)
