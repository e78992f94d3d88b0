// Host-side triangle planning of the contraction (no device code): the
// reference's triangle order and the shell-pair cover that decides which
// pair's products read each triangle.
#pragma once
#include <algorithm>
#include <cstdint>
#include <map>
#include <numeric>
#include <utility>
#include <vector>

namespace psx {

// -------------------------------------------------------- triangle list ----
// The triangles (i >= j >= l, l >= i - j, shells Ncut//step .. Nmax) in the
// reference's loop order (pyspectrum.py:415-417), as flat (i, j, l) triples.
inline void triangle_list(int step, int ncut, int nmax, std::vector<int>* ijl) {
  const int j0 = ncut / step;
  ijl->clear();
  for (int i = j0; i <= nmax; ++i)
    for (int j = j0; j <= i; ++j)
      for (int l = std::max(i - j, j0); l <= j; ++l) ijl->insert(ijl->end(), {i, j, l});
}

// ------------------------------------------------------- contract plan ----
// Which shell pair reads each triangle.  B is symmetric in its three shells,
// so a triangle (i >= j >= l) is Sum_x P D with P = d_a d_b for any of its
// pairs (i, j), (i, l), (j, l) and D the remaining shell.  Forming a pair's
// products is the costly part of the contraction, so the pairs are a greedy
// set cover (repeatedly the pair that reads most uncovered triangles, ties to
// the smallest key); each triangle then moves to the chosen pair whose
// (pair, 16-column tile) cell reads most triangles, which keeps the number
// of 16x16 output blocks down.  At Nmax = 40, step 3 this is 335 pairs for
// the 440 pairs (i, j) of the reference loop (the greedy cover alone: 339).
// Pair key = a * (nmax + 1) + b, a >= b.  Deterministic.
inline void triangle_cover(const std::vector<int>& ijl, int nmax, int j0, std::vector<int>* tpair,
                           std::vector<int>* tshell) {
  const int ntri = (int)(ijl.size() / 3), nsh = nmax + 1, nkeys = nsh * nsh;
  // the distinct (pair, remaining shell) readings of triangle t
  auto readings = [&](int t, int (&key)[3], int (&rem)[3]) {
    const int i = ijl[3 * t], j = ijl[3 * t + 1], l = ijl[3 * t + 2];
    int n = 0;
    auto add = [&](int a, int b, int c) {
      const int k = a * nsh + b;
      for (int m = 0; m < n; ++m)
        if (key[m] == k) return;
      key[n] = k; rem[n] = c; ++n;
    };
    add(i, j, l); add(i, l, j); add(j, l, i);
    return n;
  };
  int key[3], rem[3];
  std::vector<int> cnt(nkeys, 0);
  std::vector<std::vector<int>> tris_of(nkeys);
  for (int t = 0; t < ntri; ++t) {
    const int n = readings(t, key, rem);
    for (int m = 0; m < n; ++m) { cnt[key[m]]++; tris_of[key[m]].push_back(t); }
  }
  std::vector<char> covered(ntri, 0), chosen(nkeys, 0);
  tpair->assign(ntri, -1);
  tshell->assign(ntri, -1);
  for (;;) {
    int best = -1;
    for (int k = 0; k < nkeys; ++k)
      if (cnt[k] > 0 && (best < 0 || cnt[k] > cnt[best])) best = k;
    if (best < 0) break;
    chosen[best] = 1;
    for (int t : tris_of[best]) {
      if (covered[t]) continue;
      covered[t] = 1;
      const int n = readings(t, key, rem);
      for (int m = 0; m < n; ++m) cnt[key[m]]--;
    }
  }
  // Improve the greedy cover by a fixed number of local-search steps: drop 3
  // to 25 chosen pairs at random, cover the triangles left uncovered again
  // greedily (ties broken at random), prune every pair whose triangles are
  // all read by other chosen pairs (fewest triangles first), and keep the
  // result when it has no more pairs than before.  The generator has a fixed
  // seed, so the plan is the same on every run.  (Nmax 40, step 3: 339 ->
  // 335 pairs, 22 -> 21 row tiles.)
  if (ntri > 0) {
    std::vector<int> cc(ntri, 0);  // chosen readings of each triangle
    for (int k = 0; k < nkeys; ++k)
      if (chosen[k])
        for (int t : tris_of[k]) cc[t]++;
    uint64_t rs = 0x9E3779B97F4A7C15ull;
    auto rnd = [&]() {  // xorshift64*
      rs ^= rs >> 12; rs ^= rs << 25; rs ^= rs >> 27;
      return (rs * 0x2545F4914F6CDD1Dull) >> 33;
    };
    std::vector<char> ch;
    std::vector<int> c2, gain(nkeys), keys, order;
    std::vector<uint32_t> tie(nkeys);
    int nbest = 0;
    for (int k = 0; k < nkeys; ++k) nbest += chosen[k];
    for (int it = 0; it < 400; ++it) {
      ch = chosen; c2 = cc;
      keys.clear();
      for (int k = 0; k < nkeys; ++k)
        if (ch[k]) keys.push_back(k);
      const int kdrop = std::min((int)keys.size(), 3 + (int)(rnd() % 23));
      for (int d = 0; d < kdrop; ++d) {  // partial Fisher-Yates
        const int r = d + (int)(rnd() % (keys.size() - d));
        std::swap(keys[d], keys[r]);
        ch[keys[d]] = 0;
        for (int t : tris_of[keys[d]]) c2[t]--;
      }
      std::fill(gain.begin(), gain.end(), 0);
      int nunc = 0;
      for (int t = 0; t < ntri; ++t)
        if (c2[t] == 0) {
          ++nunc;
          const int n = readings(t, key, rem);
          for (int m = 0; m < n; ++m) gain[key[m]]++;
        }
      while (nunc > 0) {
        int best = -1, nties = 0;
        for (int k = 0; k < nkeys; ++k) {
          if (ch[k] || gain[k] == 0) continue;
          if (best < 0 || gain[k] > gain[best]) { best = k; nties = 1; }
          else if (gain[k] == gain[best] && rnd() % (uint64_t)(++nties) == 0) best = k;
        }
        ch[best] = 1;
        for (int t : tris_of[best]) {
          if (c2[t]++ == 0) {
            --nunc;
            const int n = readings(t, key, rem);
            for (int m = 0; m < n; ++m) gain[key[m]]--;
          }
        }
      }
      order.clear();
      for (int k = 0; k < nkeys; ++k)
        if (ch[k]) { order.push_back(k); tie[k] = (uint32_t)rnd(); }
      std::sort(order.begin(), order.end(), [&](int a, int b) {
        const size_t na = tris_of[a].size(), nb = tris_of[b].size();
        return na != nb ? na < nb : (tie[a] != tie[b] ? tie[a] < tie[b] : a < b);
      });
      int nch = (int)order.size();
      for (int k : order) {
        bool spare = true;
        for (int t : tris_of[k]) spare = spare && c2[t] >= 2;
        if (!spare) continue;
        ch[k] = 0; --nch;
        for (int t : tris_of[k]) c2[t]--;
      }
      if (nch <= nbest) { chosen.swap(ch); cc.swap(c2); nbest = nch; }
    }
  }
  // each triangle read by its first chosen pair
  for (int t = 0; t < ntri; ++t) {
    const int n = readings(t, key, rem);
    for (int m = 0; m < n; ++m)
      if (chosen[key[m]]) { (*tpair)[t] = key[m]; (*tshell)[t] = rem[m]; break; }
  }
  // move triangles to the fullest (pair, column tile) cell among the chosen pairs
  auto cell = [&](int k, int s) { return k * 4 + (s - j0) / 16; };
  std::vector<int> fill(nkeys * 4, 0);
  for (int t = 0; t < ntri; ++t) fill[cell((*tpair)[t], (*tshell)[t])]++;
  for (int pass = 0; pass < 5; ++pass) {
    for (int t = 0; t < ntri; ++t) {
      const int cur = cell((*tpair)[t], (*tshell)[t]);
      const int n = readings(t, key, rem);
      int bk = (*tpair)[t], bs = (*tshell)[t], bscore = fill[cur] - 1;
      for (int m = 0; m < n; ++m) {
        if (!chosen[key[m]] || key[m] == (*tpair)[t]) continue;
        const int score = fill[cell(key[m], rem[m])];
        if (score > bscore) { bk = key[m]; bs = rem[m]; bscore = score; }
      }
      if (bk != (*tpair)[t]) {
        fill[cur]--;
        fill[cell(bk, bs)]++;
        (*tpair)[t] = bk; (*tshell)[t] = bs;
      }
    }
  }
}

// ---------------------------------------------------- contract layout ----
// What the contraction kernel needs to know of the plan: its wave layout.
struct LayoutShape {
  bool f64 = false;           // float64 MFMA output layout
  bool simd_balance = false;  // one workgroup per CU: balance the four SIMDs
  bool mfma_bound = false;    // the blocks' MFMAs, not the products, take the time
  int maxpt = 0, wpg = 0;     // pair tiles per wave, waves per workgroup
};

struct ContractLayout {
  int npairs = 0, npt = 0, nblk = 0, waves = 0, nslot = 0;
  std::vector<int> wave_pt, wave_mask, wave_slot, pair_s, tri_loc, tri_grp;
};

// Split-BF16 contraction: the LDS serves the 16-byte A reads of 8 rows of a
// pair tile per cycle, conflict-free when their distinct shells differ
// modulo 8 (float rows 8 words apart modulo 64 banks).  Swap rows between
// the two 8-row halves of each tile while that lowers the number of shells
// that share a bank group with another shell of their half (i and j
// columns).  Row order inside a tile does not change any result.
inline void arrange_half_tiles(std::vector<int>* prow, int nsh, int j0) {
  auto half_cost = [&](const int* r) {
    int c = 0;
    for (int col = 0; col < 2; ++col) {
      int seen[64], nseen = 0, grp[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      for (int k = 0; k < 8; ++k) {
        if (r[k] < 0) continue;
        const int sh = (col == 0 ? r[k] / nsh : r[k] % nsh) - j0;
        bool dup = false;
        for (int m = 0; m < nseen; ++m) dup |= seen[m] == sh;
        if (dup) continue;
        seen[nseen++] = sh;
        c += grp[sh & 7]++ > 0 ? 1 : 0;
      }
    }
    return c;
  };
  for (size_t t = 0; t + 16 <= prow->size(); t += 16) {
    int* r = prow->data() + t;
    int cur = half_cost(r) + half_cost(r + 8);
    for (bool improved = true; improved;) {
      improved = false;
      for (int a = 0; a < 8; ++a)
        for (int b = 8; b < 16; ++b) {
          std::swap(r[a], r[b]);
          const int c2 = half_cost(r) + half_cost(r + 8);
          if (c2 < cur) { cur = c2; improved = true; }
          else std::swap(r[a], r[b]);
        }
    }
  }
}

// Pair tiles, their assignment to waves and the place of every triangle's sum
// for the triangles ijl on the shells j0..nmax.  False if a triangle has no
// chosen pair.
inline bool contract_layout(const std::vector<int>& ijl, int j0, int nmax, const LayoutShape& ls,
                            ContractLayout* cl) {
  const int ntri = (int)(ijl.size() / 3);
  std::vector<int> tpair, tshell;
  triangle_cover(ijl, nmax, j0, &tpair, &tshell);
  for (int t = 0; t < ntri; ++t)
    if (tpair[t] < 0) return false;
  // pair tiles: pairs grouped by their set of column tiles, whole tiles of one
  // set first, the remainders sorted by (tiles used, set) and cut into tiles
  std::map<int, int> pmask;  // pair key -> column tiles it reads
  for (int t = 0; t < ntri; ++t) pmask[tpair[t]] |= 1 << ((tshell[t] - j0) / 16);
  std::map<int, std::vector<int>> by_mask;
  for (const auto& pm : pmask) by_mask[pm.second].push_back(pm.first);
  std::vector<int> prow;  // pair key of each row, -1 = padding
  std::vector<std::pair<int, int>> rest;
  for (const auto& bm : by_mask) {
    const size_t whole = bm.second.size() / 16 * 16;
    prow.insert(prow.end(), bm.second.begin(), bm.second.begin() + whole);
    for (size_t k = whole; k < bm.second.size(); ++k) rest.push_back({bm.first, bm.second[k]});
  }
  std::stable_sort(rest.begin(), rest.end(), [](const std::pair<int, int>& a, const std::pair<int, int>& b) {
    const int pa = __builtin_popcount(a.first), pb = __builtin_popcount(b.first);
    return pa != pb ? pa < pb : a.first < b.first;
  });
  for (const auto& r : rest) prow.push_back(r.second);
  cl->npairs = (int)prow.size();
  cl->npt = (cl->npairs + 15) / 16;
  prow.resize((size_t)cl->npt * 16, -1);
  const int nsh = nmax + 1;
  arrange_half_tiles(&prow, nsh, j0);
  std::vector<int>& pair_s = cl->pair_s;
  pair_s.assign(2 * prow.size(), -1);
  std::map<int, int> prow_of;
  for (size_t r = 0; r < prow.size(); ++r) {
    if (prow[r] < 0) continue;
    pair_s[2 * r] = prow[r] / nsh - j0;
    pair_s[2 * r + 1] = prow[r] % nsh - j0;
    prow_of[prow[r]] = (int)r;
  }
  std::vector<int> ptmask(cl->npt, 0);
  std::vector<int> tpt(ntri), trow(ntri), tlt(ntri), tcol(ntri);
  for (int t = 0; t < ntri; ++t) {
    const int p = prow_of.at(tpair[t]);
    tpt[t] = p / 16; trow[t] = p % 16;
    tlt[t] = (tshell[t] - j0) / 16; tcol[t] = (tshell[t] - j0) % 16;
    ptmask[tpt[t]] |= 1 << tlt[t];
  }
  cl->nblk = 0;
  for (int m : ptmask) cl->nblk += __builtin_popcount(m);
  // assign pair tiles to waves: groups of WPG waves x maxpt slots, greedy by load
  const int maxpt = ls.maxpt, WPG = ls.wpg;
  const int ngroups = (cl->npt + WPG * maxpt - 1) / (WPG * maxpt);
  const int nw = ngroups * WPG;
  std::vector<int> order(cl->npt);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    return __builtin_popcount(ptmask[a]) > __builtin_popcount(ptmask[b]);
  });
  std::vector<int> load(nw, 0), cnt(nw, 0);
  std::vector<int>&wave_pt = cl->wave_pt, &wave_mask = cl->wave_mask;
  wave_pt.assign(nw * maxpt, -1);
  wave_mask.assign(nw * maxpt, 0);
  std::vector<int> pt_wave(cl->npt), pt_q(cl->npt);
  for (int pt : order) {
    int best = -1;
    if (ls.mfma_bound) {
      // F32/F64: a block's MFMAs take 8 to 16 times as long as a tile's
      // products, so the four SIMDs (wave w on SIMD w % 4) share the blocks:
      // the least loaded SIMD of a group that has room, then its least
      // loaded wave (46 blocks: at most 12 on a SIMD instead of 13; 40 shells
      // at N = 360: FP32 10.15 -> 9.67 ms, the FP64 layers 10.0 -> 9.3 ms)
      std::vector<int> sl(ngroups * 4, 0);
      for (int w = 0; w < nw; ++w) sl[w / WPG * 4 + w % WPG % 4] += load[w];
      auto simd = [&](int w) { return sl[w / WPG * 4 + w % WPG % 4]; };
      for (int w = 0; w < nw; ++w)
        if (cnt[w] < maxpt && (best < 0 || simd(w) < simd(best) ||
                               (simd(w) == simd(best) && load[w] < load[best])))
          best = w;
    } else {
      for (int w = 0; w < nw; ++w)
        if (cnt[w] < maxpt && (best < 0 || load[w] < load[best])) best = w;
    }
    wave_pt[best * maxpt + cnt[best]] = pt;
    wave_mask[best * maxpt + cnt[best]] = ptmask[pt];
    pt_wave[pt] = best; pt_q[pt] = cnt[best];
    cnt[best]++;
    // cost of a tile: forming and splitting its products (about three
    // blocks' worth of MFMA time) plus its output blocks
    load[best] += (ls.mfma_bound ? 1 : 3) + (ls.mfma_bound ? 8 : 1) * __builtin_popcount(ptmask[pt]);
  }
  // Fused layout (one workgroup per CU): the waves of the workgroup are
  // spread over the CU's four SIMDs (wave w on SIMD w % 4), and a SIMD issues
  // its waves' VALU and MFMA work one at a time, so what bounds the group is
  // the busiest SIMD.  Swap tiles (or a tile and an empty slot) between waves
  // of different SIMDs while that lowers the group's (largest SIMD load, sum
  // of squared SIMD loads).  Which wave runs a tile changes no result: its
  // sums are formed in the same order.  (Measured at Ngrid 360, 40 shells:
  // k_xcontract 6.13 -> 5.95 ms; the staged k_contract, several workgroups
  // per CU, ran 4-6 % slower with it and keeps the per-wave balance.)
  if (ls.simd_balance && WPG % 4 == 0) {
    auto tcost = [&](int pt) { return pt < 0 ? 0 : 3 + __builtin_popcount(ptmask[pt]); };
    for (int g = 0; g < ngroups; ++g) {
      const int w0 = g * WPG;
      auto score = [&](long long* sq) {
        int sl[4] = {0, 0, 0, 0};
        for (int w = w0; w < w0 + WPG; ++w) sl[(w - w0) % 4] += load[w];
        *sq = 0;
        int mx = 0;
        for (int s = 0; s < 4; ++s) { mx = std::max(mx, sl[s]); *sq += (long long)sl[s] * sl[s]; }
        return mx;
      };
      long long sq;
      int mx = score(&sq);
      for (bool improved = true; improved;) {
        improved = false;
        for (int a = w0 * maxpt; a < (w0 + WPG) * maxpt; ++a)
          for (int b = a + 1; b < (w0 + WPG) * maxpt; ++b) {
            const int wa = a / maxpt, wb = b / maxpt;
            if ((wa - w0) % 4 == (wb - w0) % 4 || wave_pt[a] == wave_pt[b]) continue;
            const int d = tcost(wave_pt[b]) - tcost(wave_pt[a]);
            load[wa] += d; load[wb] -= d;
            long long sq2;
            const int mx2 = score(&sq2);
            if (mx2 < mx || (mx2 == mx && sq2 < sq)) {
              std::swap(wave_pt[a], wave_pt[b]);
              std::swap(wave_mask[a], wave_mask[b]);
              mx = mx2; sq = sq2; improved = true;
            } else {
              load[wa] -= d; load[wb] += d;
            }
          }
      }
    }
    // slots in use first within each wave (the kernels count a wave's tiles)
    for (int w = 0; w < nw; ++w)
      for (int q = 0; q < maxpt; ++q)
        for (int r = q + 1; r < maxpt && wave_pt[w * maxpt + q] < 0; ++r)
          if (wave_pt[w * maxpt + r] >= 0) {
            std::swap(wave_pt[w * maxpt + q], wave_pt[w * maxpt + r]);
            std::swap(wave_mask[w * maxpt + q], wave_mask[w * maxpt + r]);
          }
    for (int w = 0; w < nw; ++w)
      for (int q = 0; q < maxpt; ++q) {
        const int pt = wave_pt[w * maxpt + q];
        if (pt >= 0) { pt_wave[pt] = w; pt_q[pt] = q; }
      }
  }
  // output slots per group: the blocks that hold a triangle
  std::vector<int>& wave_slot = cl->wave_slot;
  wave_slot.assign(nw * maxpt * 4, -1);
  std::vector<int> gslots(ngroups, 0);
  for (int w = 0; w < nw; ++w)
    for (int q = 0; q < maxpt; ++q) {
      const int pt = wave_pt[w * maxpt + q];
      for (int t = 0; t < 4; ++t)
        if (pt >= 0 && ((ptmask[pt] >> t) & 1)) wave_slot[(w * maxpt + q) * 4 + t] = gslots[w / WPG]++;
    }
  cl->nslot = *std::max_element(gslots.begin(), gslots.end());
  std::vector<int>&tri_loc = cl->tri_loc, &tri_grp = cl->tri_grp;
  tri_loc.assign(ntri, 0);
  tri_grp.assign(ntri, 0);
  for (int t = 0; t < ntri; ++t) {
    const int w = pt_wave[tpt[t]], q = pt_q[tpt[t]];
    const int slot = wave_slot[(w * maxpt + q) * 4 + tlt[t]];
    const int row = trow[t], col = tcol[t];
    // 16x16 MFMA output layout (measured on gfx950): f32 outputs (f32 and bf16
    // inputs) hold row r in lane col + 16*(r/4), register r%4; the f64 MFMA
    // holds it in lane col + 16*(r%4), register r/4.
    const bool f64 = ls.f64;
    const int lane = col + 16 * (f64 ? row % 4 : row / 4);
    const int reg = f64 ? row / 4 : row % 4;
    tri_loc[t] = slot * 256 + lane * 4 + reg;
    tri_grp[t] = w / WPG;
  }
  cl->waves = nw;
  return true;
}

}  // namespace psx
