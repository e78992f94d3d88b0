"""GPU test of B(k) from shell 0 on (Ncut < step) against the oracle: its power is
read as the reference's p0k[-1], the last shell's.

Tolerance: float32 fields and sums 1e-5 of max(|B|, shot noise) and of the
largest power; float64 with the 2^-40 fixed point of the assignment 1e-8."""
import numpy as np
import pytest

from oracle import spectrum as S
from pyspectrum_amd import batch as B
from pyspectrum_amd import pyspectrum as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [("fp32", 1e-5), ("fp64", 1e-8)])
@pytest.mark.parametrize("step,ncut,nmax", [(2, 0, 5), (3, 1, 4)])
def test_first_shell_holds_the_zero_mode(step, ncut, nmax, prec, tol):
    print("[case] shell 0", step, ncut, nmax, prec, flush=True)
    N, Lbox = 32, 400.0
    xyz = np.random.default_rng(nmax).uniform(0, Lbox, size=(3, 20000)).astype(np.float32)
    counts = S.counts_Bk123(N, nmax, ncut, step)
    counts[np.rint(counts / N ** 3) == 0] = 0.0
    ref = S.Bk_periodic(xyz, None, Lbox, N, step, ncut, nmax, counts=counts)
    kw = dict(Lbox=Lbox, Ngrid=N, step=step, Ncut=ncut, Nmax=nmax, precision=prec)
    one = P.Bk_periodic(xyz, **kw)
    two = B.Bk_periodic_batch([xyz, xyz], **dict(kw, Lbox=[Lbox, Lbox]))
    assert np.any(ref["i_k3"] == 0)
    for got in (one, two[0], two[1]):
        for k in ("i_k1", "i_k2", "i_k3"):
            assert np.array_equal(got[k], ref[k])
        for k in ("p0k1", "p0k2", "p0k3"):
            big = np.abs(ref[k] + ref["p0k_sn"]).max()
            assert np.abs(got[k] - ref[k]).max() <= tol * big, k
        den = np.maximum(np.abs(ref["b123"]), np.abs(ref["b123_sn"]))
        assert np.all(np.abs(got["b123"] - ref["b123"]) <= tol * den)
