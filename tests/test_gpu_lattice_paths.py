"""GPU test of the FP64 point sets on the other paths that reach them: a captured
graph, a batch, and two slots of the request loop at once.  At Ngrid 128, step 6,
5 shells the sums run on 80^3 points and their half-cell copy (the copy's seven
triangles by direct sums); at 240, step 3, 20 shells also on the grid itself.

Every result equals the eager single box bit for bit: the same kernels on the
same points, sums in a fixed order."""
import numpy as np
import pytest
import torch

from pyspectrum_amd import _lib as L
from pyspectrum_amd import batch as B
from pyspectrum_amd import graphs
from pyspectrum_amd import pyspectrum as P
from pyspectrum_amd import serve

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
SHAPES = [(128, 6, 6, 5), (240, 3, 3, 20)]


def _points(n, Lbox, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.rand((3, n), generator=g, device=DEV) * Lbox


def _has_copy(shape):
    return any(r[1] for r in L.layers(*shape))


@pytest.mark.parametrize("shape", SHAPES)
def test_captured_graph(shape):
    print("[case] layers in a graph", shape, flush=True)
    assert _has_copy(shape)
    N, step, ncut, nmax = shape
    g = graphs.BkGraph(N, step, ncut, nmax, "fp64")
    ctx = L.Context(0)
    refs = []
    for seed in (1, 2):
        gen = torch.Generator(device=DEV)
        gen.manual_seed(seed)
        h = torch.randn(g.half.shape, generator=gen, device=DEV, dtype=torch.complex128)
        b, p = torch.empty_like(g.braw), torch.empty_like(g.p0k)
        ctx.call("psx_bk_raw", L.ptr(h), N, step, ncut, nmax, L.ptr(b), L.ptr(p), L.PREC["fp64"])
        refs.append((h, b, p))
    assert not torch.equal(refs[0][1], refs[1][1])
    for rep in range(3):
        for h, b, p in refs:
            g.half.copy_(h)
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(g.braw, b) and torch.equal(g.p0k, p), rep
            # eager work of the same shape between replays
            other = torch.empty_like(b)
            ctx.call("psx_bk_raw", L.ptr(refs[0][0]), N, step, ncut, nmax, L.ptr(other), None,
                     L.PREC["fp64"])
            assert torch.equal(other, refs[0][1])
    g.close()
    ctx.close()


@pytest.mark.parametrize("shape", SHAPES)
def test_batch(shape):
    print("[case] layers in a batch", shape, flush=True)
    N, step, ncut, nmax = shape
    boxes = [500.0, 800.0, 500.0]
    xyzs = [_points(n, b, n) for n, b in zip((3000, 50000, 200), boxes)]
    kw = dict(Ngrid=N, step=step, Ncut=ncut, Nmax=nmax, precision="fp64")
    got = B.Bk_periodic_batch(xyzs, Lbox=boxes, **kw)
    for x, b, g in zip(xyzs, boxes, got):
        ref = P.Bk_periodic(x, Lbox=b, **kw)
        for k in ("i_k1", "i_k2", "i_k3", "p0k1", "b123", "q123", "counts", "b123_sn"):
            assert np.array_equal(g[k], ref[k], equal_nan=True), k


def test_two_slots():
    """Eight requests of both shapes and of a split-BF16 one on two slots, each as
    run alone, within the bound of the memory they are admitted by."""
    print("[case] layers in two slots", flush=True)

    def requests():
        out = []
        for i in range(8):
            N, step, ncut, nmax = SHAPES[i % 2]
            prec = "bf16x3" if i == 5 else "fp64"
            out.append(serve.Request(i, _points(2000 + 7000 * i, 700.0, i), 700.0, N, step=step,
                                     Ncut=ncut, Nmax=nmax, precision=prec))
        return out
    two = serve.Server(nslots=2)
    mix, _ = two.serve(requests())
    two.close()
    one = serve.Server(nslots=1)
    for r, q in zip(sorted(mix, key=lambda r: r.rid), requests()):
        assert r.error is None, r.error
        alone = one.serve([q])[0][0]
        assert alone.error is None, alone.error
        for k in ("k", "p0k", "p2k", "p4k", "b123", "q123", "p0k1", "b_counts"):
            assert np.array_equal(r.result[k], alone.result[k], equal_nan=True), (r.rid, k)
    one.close()


@pytest.mark.parametrize("shape", SHAPES + [(300, 3, 3, 30), (48, 1, 1, 7)])
def test_workspace_stays_below_its_bound(shape):
    print("[case] layers' workspace", shape, flush=True)
    N, step, ncut, nmax = shape
    n = 20000
    x = _points(n, 500.0, N)
    bound = L.context(0).bk_workspace_bytes(N, step, ncut, nmax, n, "fp64")
    ctx = L.Context(0)
    ijl = L.triangles(step, ncut, nmax)
    cnt = torch.ones(len(ijl), dtype=torch.float64, device=DEV)
    tri = torch.from_numpy(np.ascontiguousarray(ijl)).to(DEV)
    out = torch.empty((7, len(ijl)), dtype=torch.float64, device=DEV)
    p0k = torch.empty(nmax, dtype=torch.float64, device=DEV)
    ctx.call("psx_bk_periodic", L.ptr(x), None, n, N, 500.0, float(n), float(n), step, ncut, nmax,
             L.ptr(cnt), L.ptr(tri), 1.0, 1.0, 1.0, 1.0, 1.0, L.ptr(out), L.ptr(p0k), L.PREC["fp64"])
    torch.cuda.synchronize()
    assert 0 < ctx.workspace_bytes() <= bound
    ctx.close()
