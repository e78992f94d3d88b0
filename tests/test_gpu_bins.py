"""GPU tests of the k-space binning kernels, which add the rows (+-y, +-z)
that share their bins before binning them: P_l along each line of sight and
the shell sums against the oracle, at sizes where a wave's 64 lanes end inside
a row, hold a whole row or span two, and where mirror rows coincide (0, N/2).

Tolerance: float64 sums of at most N^3 terms in another order, compared with
the largest sum of their kind: N^3 * 2^-53 < 2e-9 at N = 256 as a bound, about
its square root in practice; 1e-11 here (N <= 150).  Counts are exact."""
import numpy as np
import pytest
import torch

from oracle import spectrum as S
from pyspectrum_amd import _lib as L
from pyspectrum_amd import pyspectrum as P

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
TOL = 1e-11


def _half(N, seed):
    """Random half field [ix, iy, iz] and its device form [z][y][x]."""
    rng = np.random.default_rng(seed)
    h = rng.standard_normal((N // 2 + 1, N, N)) + 1j * rng.standard_normal((N // 2 + 1, N, N))
    return h, torch.from_numpy(np.ascontiguousarray(h.transpose(2, 1, 0))).to(DEV)


@pytest.mark.parametrize("irsd", [0, 1, 2])
@pytest.mark.parametrize("N,nmu", [(4, 1), (10, 7), (30, 10), (128, 3), (150, 10)])
def test_pk_rsd_row_groups(N, nmu, irsd):
    print("[case] pk_rsd groups", N, nmu, irsd, flush=True)
    h, d = _half(N, 7 * N + irsd)
    got = P._pk_pbox_rsd(d, irsd, 1000, N // 2, nmu, N, L.PREC["fp64"], 0)
    ref = S.pk_pbox_rsd(h, irsd, 1000, N // 2, nmu, N)
    for k in (4, 8):  # mode counts per k bin and per (k, mu) bin
        assert np.array_equal(got[k], ref[k]), k
    for k in (0, 1, 2, 3, 5, 6, 7):
        scale = np.max(np.abs(ref[1])) if k in (2, 3) else np.max(np.abs(ref[k]))
        assert np.max(np.abs(got[k] - ref[k])) <= TOL * scale, k


@pytest.mark.parametrize("N,step,nbins", [(4, 1, 3), (6, 2, 1), (30, 1, 26), (128, 3, 20),
                                          (128, 1, 64), (64, 4096, 2)])
def test_bin_power_row_groups(N, step, nbins):
    print("[case] bin_power groups", N, step, nbins, flush=True)
    h, d = _half(N, 11 * N + step)
    out = torch.empty(3 * nbins, dtype=torch.float64, device=DEV)
    L.context(0).call("psx_bin_power", L.ptr(d), N, step, nbins, 0.25, L.ptr(out), L.PREC["fp64"])
    got = out.cpu().numpy().reshape(3, nbins)
    m = S.kmag2(N)
    b = S.shell_of_m(m, step).ravel()
    full = S.reflect_delta(h, N)
    rows = (0.25 * np.sqrt(m), np.abs(full) ** 2, np.ones(m.shape))
    for r, v in enumerate(rows):
        ref = np.bincount(b, weights=v.ravel(), minlength=nbins + 1)[1:nbins + 1]
        if r == 2:
            assert np.array_equal(got[r], ref)
        else:
            assert np.max(np.abs(got[r] - ref)) <= TOL * max(1e-300, np.max(ref))
