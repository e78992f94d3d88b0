// Host-side choice of the point sets of the FP64 triangle sums (no device code).
//
// B_t = sum_x d_i d_j d_l over the N^3 grid is a quadrature of a band-limited
// function: its modes k1 + k2 + k3 lie within R_t = r_i + r_j + r_l (r_s the
// largest |k| of shell s).  On any point lattice the mean of such a function
// is exact when no nonzero vector of the reciprocal lattice is that short, so
// the same sum follows from fewer points:
//   * the cubic grid of M^3 points: R_t < M;
//   * that grid and a copy shifted by half a cell along all axes (a body-
//     centred lattice, 2 M^3 points): its reciprocal vectors are M times
//     integer triples of even sum, the shortest M sqrt(2), so R_t < 1.414 M --
//     the 2 M^3 points do the work of 2.83 M^3 of a cubic grid.
// Both are M^3 FFTs (the shift is a phase per mode), and the first is part of
// the second, so triangles with R_t < M need only the unshifted half.
// Triangles with R_t >= N alias on the N^3 grid, which the estimator's
// definition includes: they stay there, and so does every triangle with a
// shell that holds modes of the Nyquist planes.
//
// At N = 360, step 3, 40 shells: M = 256, 6348 triangles on the cubic grid,
// 1706 of them also on the shifted one, 2 on the N^3 grid.  (FP32 and
// split-BF16 sums keep the N^3 grid: their rounding, 1e-7 of a sum, would
// change with the points.)
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace psx {

struct LayerChoice {
  int M = 0;
  bool shifted = false;   // the half-cell copy
  bool add = false;
  std::vector<int> tri;   // indices into the triangle list
  std::vector<double> weight;
};

// Relative cost of a layer of G points: its matrix-core time (the 16x16
// blocks that ntri triangles pack into) and the passes that form its shell
// fields, in picoseconds (measured at N = 360: 18.5 ms for 46 blocks, 7.5 ms
// for 40 shells; lengths without a compile-time FFT take about twice the
// latter), plus its launches.  At most DIRECT_TRI triangles on DIRECT_SHELLS
// shells are summed directly, in one read of the fields.
// Measured against the N^3 grid (psx_bk_raw and the shell fields with their
// contraction, N = 48 to 512): every one of 18 shapes that take layers is faster,
// by 1.3 (256 / step 2 / 44 shells, 8.35 against 10.9 ms) to 4.9 (512 / 2 / 60).
// The rule errs towards the grid: with layers forced, 14 of 28 shapes that it
// leaves there were slower (96 / 3 / 12 0.81, 256 / 3 / 30 0.81, 200 / 3 / 24 0.79),
// but 216 / 3 / 24, 192 / 6 / 9, 128 / 3 / 12 and 240 / 2 / 40 were 1.4 to 1.5 times
// as fast.
constexpr int DIRECT_TRI = 16, DIRECT_SHELLS = 8;
inline double layer_cost(double G, int ntri, int nshells, bool fast_fft) {
  const double blocks = std::max(4.0, 1.65 * ntri / 256.0 + 4.0);
  const double contract = ntri <= DIRECT_TRI && nshells <= DIRECT_SHELLS ? 2.0 * nshells
                                                                         : 8.6 * blocks;
  return G * (contract + (fast_fft ? 4.0 : 8.0) * nshells) * 1e-6 + 35.0;  // microseconds
}

// The layers for the triangles ijl (i >= j >= l) of an N^3 grid, or none when
// the N^3 grid alone is (within 5 %) as cheap.  mmax(j): largest |k|^2 of
// shell j; sizes: the FFT lengths of the layers, ascending; fast: whether N
// itself has a compile-time FFT.
template <typename MMax>
inline std::vector<LayerChoice> choose_layers(const std::vector<int>& ijl, int N, MMax mmax,
                                              const std::vector<int>& sizes, bool fast) {
  const int ntri = (int)(ijl.size() / 3);
  std::vector<LayerChoice> best;
  if (ntri == 0) return best;
  int jmax = 0, jmin = ijl[0];
  for (int v : ijl) { jmax = std::max(jmax, v); jmin = std::min(jmin, v); }
  std::vector<double> r(jmax + 1, 0.0);
  for (int j = jmin; j <= jmax; ++j) r[j] = std::sqrt((double)mmax(j));
  std::vector<double> R(ntri);
  for (int t = 0; t < ntri; ++t) R[t] = r[ijl[3 * t]] + r[ijl[3 * t + 1]] + r[ijl[3 * t + 2]];
  const double eps = 1e-6;  // r is rounded: never take a lattice that just fits
  auto cost = [&](const LayerChoice& l) {
    if (l.tri.empty()) return 0.0;
    int lo = jmax, hi = 0;
    for (int t : l.tri) { lo = std::min(lo, ijl[3 * t + 2]); hi = std::max(hi, ijl[3 * t]); }
    return layer_cost((double)l.M * l.M * l.M, (int)l.tri.size(), hi - lo + 1,
                      l.M != N || fast);
  };
  LayerChoice all;
  all.M = N;
  all.tri.resize(ntri);
  double best_cost = 0.95 * cost(all);
  for (int M : sizes) {
    if (M >= N) break;
    for (int bcc = 0; bcc < 2; ++bcc) {
      const double reach = (bcc ? std::sqrt(2.0) * M : (double)M) - eps;
      LayerChoice a, b, f;
      a.M = b.M = M;
      f.M = N;
      b.shifted = b.add = true;
      const double w = std::pow((double)N / M, 3);
      for (int t = 0; t < ntri; ++t) {
        // modes of the largest side inside both grids' Nyquist planes
        const bool inside = r[ijl[3 * t]] < std::min(N, M) / 2 - eps;
        if (!inside || R[t] >= reach || R[t] >= N - eps) {
          f.tri.push_back(t);
          f.weight.push_back(1.0);
          continue;
        }
        const bool both = R[t] >= M - eps;
        a.tri.push_back(t);
        a.weight.push_back(both ? 0.5 * w : w);
        if (both) {
          b.tri.push_back(t);
          b.weight.push_back(0.5 * w);
        }
      }
      if (a.tri.empty() || (bcc && b.tri.empty())) continue;
      const double c = cost(a) + cost(b) + cost(f);
      if (c >= best_cost) continue;
      best_cost = c;
      best.clear();
      for (LayerChoice* l : {&f, &a, &b})
        if (!l->tri.empty()) best.push_back(std::move(*l));
    }
  }
  return best;
}

}  // namespace psx
