"""CPU tests of the contraction's wave layout (contract_layout of
pyspectrum_amd/csrc/psx_plan.h) for the layouts of the kernels, on whole triangle
lists and on the subsets that the FP64 point sets give it.

A small C++ driver is compiled against the header with g++ and prints the layout.
Checked:
  * every pair tile has one place, at most maxpt to a wave, without gaps;
  * every block that holds a triangle has its own output slot in its group;
  * no two triangles share an entry, and the entry of a triangle is the row of
    one of its pairs and the column of its remaining shell;
  * the 46 blocks of 40 shells leave at most 12 to a SIMD."""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pyspectrum_amd", "csrc")

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include "psx_plan.h"
static void line(const std::vector<int>& v) {
  for (int x : v) printf("%d ", x);
  printf("\n");
}
int main(int argc, char** argv) {
  const int step = atoi(argv[1]), ncut = atoi(argv[2]), nmax = atoi(argv[3]), most = atoi(argv[4]);
  psx::LayoutShape ls;
  ls.f64 = atoi(argv[5]); ls.simd_balance = atoi(argv[6]); ls.mfma_bound = atoi(argv[7]);
  ls.maxpt = atoi(argv[8]); ls.wpg = atoi(argv[9]);
  std::vector<int> all, ijl;
  psx::triangle_list(step, ncut, nmax, &all);
  int j0 = nmax, top = 0;
  for (size_t t = 0; t < all.size(); t += 3) {
    if (all[t] + all[t + 1] + all[t + 2] > most) continue;
    ijl.insert(ijl.end(), all.begin() + t, all.begin() + t + 3);
    j0 = std::min(j0, all[t + 2]);
    top = std::max(top, all[t]);
  }
  psx::ContractLayout cl;
  if (!psx::contract_layout(ijl, j0, top, ls, &cl)) return 1;
  line({cl.npairs, cl.npt, cl.nblk, cl.waves, cl.nslot, j0, top});
  line(ijl); line(cl.wave_pt); line(cl.wave_mask); line(cl.wave_slot); line(cl.pair_s);
  line(cl.tri_loc); line(cl.tri_grp);
  return 0;
}
"""

# f64, simd_balance, mfma_bound, maxpt, waves per workgroup
KERNELS = {"f64": (1, 0, 1, 4, 8), "f32": (0, 0, 1, 2, 12), "bf16": (0, 0, 0, 2, 12),
           "bf16 4 tiles": (0, 0, 0, 3, 8), "fused": (0, 1, 0, 2, 12)}
ALL = 10 ** 6


@pytest.fixture(scope="module")
def layout(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("layout")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + CSRC, str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True)

    def run(kernel, step, ncut, nmax, most):
        args = [str(v) for v in (step, ncut, nmax, most) + KERNELS[kernel]]
        out = subprocess.run([str(d / "driver")] + args, check=True, capture_output=True,
                             text=True).stdout
        rows = [np.array([int(v) for v in r.split()]) for r in out.splitlines()]
        names = ("ijl", "wave_pt", "wave_mask", "wave_slot", "pair_s", "tri_loc", "tri_grp")
        lay = dict(zip(names, rows[1:]))
        lay.update(zip(("npairs", "npt", "nblk", "waves", "nslot", "j0", "nmax"), rows[0].tolist()))
        return lay
    return run


@pytest.mark.parametrize("step,ncut,nmax,most", [
    (3, 3, 40, ALL), (2, 2, 60, ALL), (3, 3, 12, ALL), (1, 0, 5, ALL), (3, 3, 1, ALL),
    (3, 3, 40, 84), (2, 2, 60, 130), (3, 30, 40, 100), (4, 8, 48, 60),
])
@pytest.mark.parametrize("kernel", list(KERNELS))
def test_every_triangle_has_its_own_entry(layout, kernel, step, ncut, nmax, most):
    f64, _, _, maxpt, wpg = KERNELS[kernel]
    lay = layout(kernel, step, ncut, nmax, most)
    waves, npt = lay["waves"], lay["npt"]
    assert waves % wpg == 0 and npt == -(-lay["npairs"] // 16)
    pt = lay["wave_pt"].reshape(waves, maxpt)
    mask = lay["wave_mask"].reshape(waves, maxpt)
    slot = lay["wave_slot"].reshape(waves, maxpt, 4)
    assert sorted(pt[pt >= 0]) == list(range(npt))
    assert np.all((pt >= 0)[:, :-1] >= (pt >= 0)[:, 1:])  # tiles in use first
    assert np.all(mask[pt < 0] == 0)
    # slots: one for each block of a group, 0, 1, ... below nslot
    used = (mask[:, :, None] >> np.arange(4)) & 1
    assert np.array_equal(slot >= 0, used == 1) and used.sum() == lay["nblk"]
    where = {}
    for w, q, t in zip(*np.nonzero(used)):
        where[(w // wpg, slot[w, q, t])] = (w, q, t)
    assert len(where) == lay["nblk"]
    sizes = [np.sum(slot[g:g + wpg] >= 0) for g in range(0, waves, wpg)]
    assert max(sizes) == lay["nslot"] and slot.max() == lay["nslot"] - 1
    # triangles
    ijl, pair_s = lay["ijl"].reshape(-1, 3), lay["pair_s"].reshape(-1, 2)
    assert len(ijl) > 0
    assert len(set(zip(lay["tri_grp"], lay["tri_loc"]))) == len(ijl)
    blocks = set()
    for tri, loc, grp in zip(ijl, lay["tri_loc"], lay["tri_grp"]):
        s, lane, reg = loc // 256, loc % 256 // 4, loc % 4
        w, q, t = where[(grp, s)]
        row = 4 * reg + lane // 16 if f64 else 4 * (lane // 16) + reg
        a, b = pair_s[pt[w, q] * 16 + row]
        assert a >= 0 and b >= 0
        got = sorted((a + lay["j0"], b + lay["j0"], 16 * t + lane % 16 + lay["j0"]))
        assert got == sorted(tri.tolist())
        blocks.add((w, q, t))
    assert len(blocks) == lay["nblk"]  # no block without a triangle


@pytest.mark.parametrize("kernel", ["f64", "f32"])
def test_blocks_are_shared_by_the_simds(layout, kernel):
    _, _, _, maxpt, wpg = KERNELS[kernel]
    lay = layout(kernel, 3, 3, 40, ALL)
    assert lay["nblk"] == 46 and lay["waves"] == wpg
    per_wave = np.array([bin(m).count("1") for m in lay["wave_mask"]]).reshape(wpg, maxpt).sum(1)
    assert max(per_wave[s::4].sum() for s in range(4)) <= 12
