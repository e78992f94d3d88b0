"""CPU test of bench.py's roofline: the operations it counts are those of the
launches that were timed, in FP64 the triangle sums on each point set, so that
the rate of a recorded run stays below the peak."""
import numpy as np
import pytest

import bench
from pyspectrum_amd import _lib as L


class _Box:
    L = L

    def __init__(self, N, step, Ncut, Nmax):
        self.N, self.step, self.Ncut, self.Nmax = N, step, Ncut, Nmax
        self.ijl = L.triangles(step, Ncut, Nmax)
        self.ntri = len(self.ijl)


def _kern(name, launches, ms):
    return {name: {"launches_per_box": launches, "ms_per_launch": ms / launches, "ms_per_box": ms}}


def test_fp64_counts_the_point_sets():
    """Ngrid 360, 40 shells: 9.16 ms a box in two launches on 256^3 points, one
    of 6348 triangles and one of 1706."""
    box = _Box(360, 3, 3, 40)
    rows = L.layers(360, 3, 3, 40)
    assert [tuple(r[:3]) for r in rows] == [(360, 0, 2), (256, 0, 6348), (256, 1, 1706)]
    assert list(rows[:, 4]) == [0, 1, 1]
    r = bench.roofline(box, "fp64", _kern("k_contract", 2, 9.16))
    pairs = rows[1:, 3]
    assert np.all((pairs > 0) & (pairs <= 440))
    flops = 256.0 ** 3 * (float(pairs.sum()) + 2 * (6348 + 1706))
    assert r["flops_per_box"] == pytest.approx(flops, rel=1e-12)
    assert r["flops_per_launch"] == pytest.approx(flops / 2, rel=1e-12)
    assert r["achieved"] == pytest.approx(flops / 9.16e-3 / 1e12, abs=0.01)
    assert 0 < r["frac"] < 1
    assert r["traffic_per_box"] == pytest.approx(2 * r["traffic"])


@pytest.mark.parametrize("name,prec", [("k_contract", "fp64"), ("k_contract", "fp32"),
                                       ("k_xcontract", "bf16x3")])
def test_grid_sums(name, prec):
    """Shapes without point sets, and the single precisions: all N^3 points."""
    box = _Box(96, 3, 3, 15)
    assert len(L.layers(96, 3, 3, 15)) == 0
    r = bench.roofline(box, prec, _kern(name, 1, 5.0))
    npairs = len({tuple(t[:2]) for t in box.ijl.tolist()})
    flops = 96.0 ** 3 * (npairs + 2 * box.ntri)
    if name == "k_xcontract":
        flops += 5.0 * 96.0 ** 3 * np.log2(96) * 8
    assert r["flops_per_box"] == pytest.approx(flops, rel=1e-12)
    assert r["flops_per_launch"] == r["flops_per_box"]


def test_other_kernels_have_no_peak():
    r = bench.roofline(_Box(96, 3, 3, 15), "fp32", _kern("k_shell_x", 1, 5.0))
    assert r["bound"] is None and r["kernel"] == "k_shell_x"
