"""CPU tests of which point sets the FP64 triangle sums of a shape take
(psx_bk_layers, choose_layers of pyspectrum_amd/csrc/psx_lattice.h): the expected
sets by name, also where there are none, and for each of them that every triangle
is summed once, on points that carry its modes.  The grid lengths are those of
the library (PSX_LAT_SIZES), read from its header."""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

from pyspectrum_amd import _lib as L

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pyspectrum_amd", "csrc")

# shape -> (M, shifted, triangles) of each set; none: all triangles on the N^3 grid
SHAPES = {
    (360, 3, 3, 40): [(360, 0, 2), (256, 0, 6348), (256, 1, 1706)],
    (512, 2, 2, 60): [(512, 0, 1), (256, 0, 20274), (256, 1, 5003)],
    (192, 2, 2, 19): [(96, 0, 805), (96, 1, 67)],
    (240, 3, 0, 20): [(240, 0, 2), (128, 0, 944), (128, 1, 272)],
    (300, 3, 3, 30): [(300, 0, 1), (192, 0, 2824), (192, 1, 784)],
    (256, 2, 2, 40): [(192, 0, 6350), (192, 1, 640)],
    (180, 4, 4, 11): [(128, 0, 191), (128, 1, 4)],
    (128, 6, 6, 5): [(80, 0, 28), (80, 1, 7)],
    (144, 4, 8, 8): [(80, 0, 71), (80, 1, 16)],
    (48, 1, 1, 7): [(32, 0, 62)],
    (128, 3, 3, 9): [(96, 0, 115)],
    # too near to aliasing, or too small to gain
    (384, 3, 6, 48): [], (128, 3, 3, 20): [], (64, 1, 1, 31): [], (96, 3, 3, 30): [],
    (1024, 5, 5, 64): [], (30, 1, 1, 3): [], (64, 3, 3, 12): [],
}

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include "psx_lattice.h"
#include "psx_plan.h"
int main(int argc, char** argv) {
  const int N = atoi(argv[1]), step = atoi(argv[2]), ncut = atoi(argv[3]), nmax = atoi(argv[4]);
  std::vector<int> ijl, sizes;
  for (int a = 6; a < argc; ++a) sizes.push_back(atoi(argv[a]));
  psx::triangle_list(step, ncut, nmax, &ijl);
  auto mm = [&](int j) { const long long a = (2LL * j + 1) * step; return (a * a - 1) / 4; };
  for (const auto& l : psx::choose_layers(ijl, N, mm, sizes, atoi(argv[5]) != 0)) {
    printf("%d %d %d", l.M, (int)l.shifted, (int)l.add);
    for (size_t t = 0; t < l.tri.size(); ++t) printf(" %d %.17g", l.tri[t], l.weight[t]);
    printf("\n");
  }
  return 0;
}
"""


def _sizes():
    text = open(os.path.join(CSRC, "psx_fft.h")).read()
    fft, lat = (re.search(r"#define %s\(X\) (.*)" % n, text).group(1)
                for n in ("PSX_FFT_SIZES", "PSX_LAT_SIZES"))
    assert lat.startswith("PSX_FFT_SIZES(X)")
    num = [[int(v) for v in re.findall(r"X\((\d+)\)", t)] for t in (fft, lat)]
    return num[0], sorted(num[0] + num[1])


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("choice")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + CSRC, str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True)
    fast, sizes = _sizes()

    def run(*shape):
        args = list(shape) + [int(shape[0] in fast)] + sizes
        out = subprocess.run([str(d / "driver")] + [str(v) for v in args], check=True,
                             capture_output=True, text=True).stdout
        rows = [line.split() for line in out.splitlines()]
        return [(int(f[0]), int(f[1]), int(f[2]), np.array(f[3::2], dtype=int),
                 np.array(f[4::2], dtype=float)) for f in rows]
    return run


@pytest.mark.parametrize("shape", list(SHAPES), ids=str)
def test_expected_point_sets(shape):
    rows = L.layers(*shape)
    assert [tuple(r[:3].tolist()) for r in rows] == SHAPES[shape]
    tri = L.triangles(*shape[1:])
    for M, shifted, ntri, npairs, mfma in rows:
        assert 0 < npairs <= len({tuple(t[:2]) for t in tri.tolist()})
        assert mfma == 1 or ntri <= 16


@pytest.mark.parametrize("shape", [s for s in SHAPES if SHAPES[s]], ids=str)
def test_every_triangle_is_summed_once(driver, shape):
    N, step, ncut, nmax = shape
    layers = driver(*shape)
    assert [(l[0], l[1], len(l[3])) for l in layers] == SHAPES[shape]
    tri = L.triangles(step, ncut, nmax)
    r = np.sqrt([((2 * j + 1) * step) ** 2 // 4 for j in range(nmax + 1)])
    reach = r[tri].sum(1)
    seen, share = np.zeros(len(tri), dtype=int), np.zeros(len(tri))
    copies = np.concatenate([l[3] for l in layers if l[1]] or [np.zeros(0, dtype=int)])
    for M, shifted, add, t, w in layers:
        assert np.all((seen[t] > 0) == bool(add))
        seen[t] += 1
        share[t] += w * (M / N) ** 3
        if M != N:
            assert np.all(reach[t] < N) and np.all(r[tri[t]] < M / 2)
            assert np.all(reach[t] < np.where(np.isin(t, copies), np.sqrt(2), 1.0) * M)
    assert np.all(seen >= 1) and np.all(np.abs(share - 1) <= 1e-14)
