// Mesh front end of the periodic-box estimator: PCS assignment with
// interlacing, the interlacing/deconvolution combination, and the half <->
// full field conversions.
#include <cstring>

#include "psx_ctx.h"

namespace psx {

// ------------------------------------------------------------ assignment --
// Per-axis PCS stencil of estimator.f:302-378, replayed with the reference's
// float32 operation order (no contraction into FMA): rx = kf_ks*x + 1 + offset
// is the 1-based grid coordinate (offset = 0 for boxes, Ngrid/2 for survey
// coordinates centred on the observer, pyspectrum.py:819); grid A uses rx,
// grid B uses rx + 0.5.  Returns the 0-based base cell (wrapped into [0, N))
// and the four weights (x6) for cells base-1 .. base+2.
// (HIP's __fmul_rn/__fadd_rn are plain operators, so FMA contraction is
// switched off explicitly: the reference multiplies and adds separately.)
__device__ __forceinline__ float pcs_coord(float r, const PcsMap& pm, bool shift, int N, int* c) {
#pragma clang fp contract(off)
  float rx = pm.kf_ks * r + 1.0f;
  rx = rx + pm.offset;
  if (shift) rx = rx + 0.5f;
  const int i1 = (int)rx;  // rx >= 0 for positions inside the clip range: truncation = floor
  const int c0 = i1 - 1;   // in [-1, N]
  *c = c0 < 0 ? c0 + N : (c0 >= N ? c0 - N : c0);
  return rx - (float)i1;  // exact
}

// float32 weights, the reference's operation order
__device__ __forceinline__ void pcs_weights(float h, float* wts) {
#pragma clang fp contract(off)
  const float h2 = h * h;
  const float t = 1.0f - h;
  const float wm2 = (t * t) * t;
  const float wm1 = 4.0f + (3.0f * h - 6.0f) * h2;
  const float wp2 = h2 * h;
  const float wp1 = ((6.0f - wm2) - wm1) - wp2;
  wts[0] = wm2; wts[1] = wm1; wts[2] = wp1; wts[3] = wp2;
}

// float64 weights of the same float32 cell offset (FP64 pipeline)
__device__ __forceinline__ void pcs_weights(float hf, double* wts) {
  const double h = (double)hf;
  const double h2 = h * h;
  const double t = 1.0 - h;
  const double wm2 = t * t * t;
  const double wm1 = 4.0 + (3.0 * h - 6.0) * h2;
  const double wp2 = h2 * h;
  wts[0] = wm2; wts[1] = wm1; wts[2] = 6.0 - wm2 - wm1 - wp2; wts[3] = wp2;
}

template <typename W> __device__ __forceinline__ W wmul(W a, W b);
template <> __device__ __forceinline__ float wmul<float>(float a, float b) { return a * b; }
template <> __device__ __forceinline__ double wmul<double>(double a, double b) { return a * b; }

__device__ __forceinline__ float clip_pos(float v, const PcsMap& pm) {
  // np.clip to [lo, hi]; NaN is sent to lo so no cell index leaves the grid
  v = (v >= pm.lo) ? v : pm.lo;
  return (v <= pm.hi) ? v : pm.hi;
}

// The grid is assigned in tiles of whole x lines: a tile is a ty x tz block
// of (y, z) lines, ty*tz no more than the FFT engine's lines per tile.
// Particles are sorted by the tile of their grid-A base cell; the workgroup
// of a tile visits the particles of every tile whose stencils can reach it
// and adds the contributions to its own cells as int64 fixed point (scale
// 2^e) with LDS atomics -- integer sums, so the grid does not depend on the
// order of the adds -- then converts to the working precision and stores
// each line once (in FFT_periodic after the x pass of the FFT).
struct AssignTiling {
  int ty, tz, nty, ntz;  // lines per tile along y and z; tiles along y and z
};

// At most 8 lines per tile keeps the LDS of a tile (16 B per cell plus the
// complex lines) small enough for several workgroups per CU.
#ifndef PSX_ASSIGN_LINES
#define PSX_ASSIGN_LINES 8
#endif
#ifndef PSX_ASSIGN_TY
#define PSX_ASSIGN_TY 4
#endif
constexpr int ASSIGN_LINES = PSX_ASSIGN_LINES;
template <typename T, int NC>
constexpr int assign_lines_max() {
  return Tile<T, NC>::MAXLINES < ASSIGN_LINES ? Tile<T, NC>::MAXLINES : ASSIGN_LINES;
}

template <typename T>
static AssignTiling assign_tiling(int N) {
  const int tl = std::min(tile_lines_host<T>(N), ASSIGN_LINES);
  AssignTiling a;
  a.ty = tl >= PSX_ASSIGN_TY ? PSX_ASSIGN_TY : tl;
  a.tz = tl / a.ty;
  a.nty = (N + a.ty - 1) / a.ty;
  a.ntz = (N + a.tz - 1) / a.tz;
  return a;
}

// Particles are ordered by assignment tile with a counting sort: count per
// tile (the atomic's return value is the particle's rank in its tile), an
// exclusive scan of the counts, and a scatter of (x, y, z, w) records to
// offset + rank.  The order inside a tile depends on the atomics, which does
// not matter: the tile's workgroup adds integer contributions.
__device__ __forceinline__ unsigned tile_key(float y, float z, int N, const PcsMap& pm, AssignTiling at) {
  int cy, cz;
  pcs_coord(y, pm, false, N, &cy);
  pcs_coord(z, pm, false, N, &cz);
  return (unsigned)(cz / at.tz) * (unsigned)at.nty + (unsigned)(cy / at.ty);
}

__global__ void k_fill_u32(unsigned* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// The boxes of a batched assignment (kernel argument): box b's particles,
// its position map and fixed-point scale, and the offset of its particles
// in the sort buffers.  Tile counts and offsets are per box back to back.
struct AssignBoxes {
  const float* xyz[PSX_MAX_BATCH];
  const float* w[PSX_MAX_BATCH];
  int64_t np[PSX_MAX_BATCH];
  int64_t poff[PSX_MAX_BATCH];
  PcsMap pm[PSX_MAX_BATCH];
  double scale[PSX_MAX_BATCH];
};

__global__ void k_tile_count(const AssignBoxes bs, int N, AssignTiling at,
                             unsigned* __restrict__ count, unsigned* __restrict__ key,
                             unsigned* __restrict__ rank) {
  const int b = blockIdx.y;
  const int64_t np = bs.np[b];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const float* xyz = bs.xyz[b];
  const PcsMap pm = bs.pm[b];
  count += (int64_t)b * at.nty * at.ntz;
  const unsigned k = tile_key(clip_pos(xyz[np + i], pm), clip_pos(xyz[2 * np + i], pm), N, pm, at);
  key[bs.poff[b] + i] = k;
  rank[bs.poff[b] + i] = atomicAdd(count + k, 1u);
}

// Exclusive scan of n counts into off[0..n] (off[n] = total), one workgroup:
// thread t owns the contiguous segment [t*seg, (t+1)*seg) and keeps up to
// SCAN_REG of its counts in registers (one round of loads, no re-read); the
// segment sums are scanned across each wave with shuffles and the 16 wave
// totals once in LDS.  Box blockIdx.y: count [box][n], off [box][n + 1].
constexpr int SCAN_THREADS = 1024, SCAN_WAVES = SCAN_THREADS / 64, SCAN_REG = 32;
__global__ __launch_bounds__(SCAN_THREADS) void k_tile_scan(const unsigned* __restrict__ count,
                                                            int n, unsigned* __restrict__ off) {
  count += (int64_t)blockIdx.y * n;
  off += (int64_t)blockIdx.y * (n + 1);
  __shared__ unsigned wsum[SCAN_WAVES];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int seg = (n + SCAN_THREADS - 1) / SCAN_THREADS;
  const int b = min(n, t * seg), e = min(n, b + seg);
  unsigned c[SCAN_REG];
  unsigned s = 0;
  if (seg <= SCAN_REG) {
#pragma unroll
    for (int k = 0; k < SCAN_REG; ++k) c[k] = b + k < e ? count[b + k] : 0u;
#pragma unroll
    for (int k = 0; k < SCAN_REG; ++k) s += c[k];
  } else {
    for (int i = b; i < e; ++i) s += count[i];
  }
  // inclusive scan of the segment sums across the wave, then across waves
  unsigned inc = s;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned u = __shfl_up(inc, d, 64);
    if (lane >= d) inc += u;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  unsigned before = 0;  // totals of the earlier waves
  for (int w = 0; w < wave; ++w) before += wsum[w];
  unsigned run = before + inc - s;  // exclusive prefix of this segment
  if (seg <= SCAN_REG) {
#pragma unroll
    for (int k = 0; k < SCAN_REG; ++k)
      if (b + k < e) { off[b + k] = run; run += c[k]; }
  } else {
    for (int i = b; i < e; ++i) { off[i] = run; run += count[i]; }
  }
  if (t == SCAN_THREADS - 1) off[n] = before + inc;
}

__global__ void k_tile_scatter(const AssignBoxes bs, const unsigned* __restrict__ key,
                               const unsigned* __restrict__ rank, const unsigned* __restrict__ off,
                               int ntiles, float4* __restrict__ rec) {
  const int b = blockIdx.y;
  const int64_t np = bs.np[b];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const float* xyz = bs.xyz[b];
  const float* w = bs.w[b];
  const PcsMap pm = bs.pm[b];
  const int64_t p = bs.poff[b] + i;
  off += (int64_t)b * (ntiles + 1);
  rec[bs.poff[b] + (int64_t)off[key[p]] + rank[p]] =
      make_float4(clip_pos(xyz[i], pm), clip_pos(xyz[np + i], pm), clip_pos(xyz[2 * np + i], pm),
                  w ? w[i] : 1.0f);
}

// Tiles (width tw) along one axis holding the base cells c in [t0-3, t1]
// (cyclic) whose stencils reach the cells [t0, t1): grid A covers c-1..c+2
// and grid B (base c or c+1) c-1..c+3.  At most t1-t0+4 <= 8 tiles.
__device__ int source_tiles(int t0, int t1, int N, int tw, int* out) {
  int n = 0;
  const int span = min(t1 - t0 + 4, N);
  for (int k = 0; k < span; ++k) {
    const int c = ((t0 - 3 + k) % N + N) % N;
    const int t = c / tw;
    bool seen = false;
    for (int u = 0; u < n; ++u) seen = seen || out[u] == t;
    if (!seen) out[n++] = t;
  }
  return n;
}

__device__ __forceinline__ int wrap1(int c, int N) {
  // c in [-1, 2N): one correction
  return c < 0 ? c + N : (c >= N ? c - N : c);
}

// The rows of work of a tile: entries (record, grid, z stencil row).  A tile
// has at most ASSIGN_TZ z rows, so a particle gives at most that many per grid;
// after a batch (one particle a thread) fewer entries than threads stay.
constexpr int ASSIGN_TZ = ASSIGN_LINES / PSX_ASSIGN_TY < 4 ? ASSIGN_LINES / PSX_ASSIGN_TY : 4;
__host__ __device__ constexpr int assign_queue(int threads) { return threads * (2 * ASSIGN_TZ + 1); }

// LDS: int64 accumulators acc[line][x][grid] (16 B per cell) and the queue of
// entries; with FFTX the same memory then holds the complex lines (row stride
// N+1) and the twiddles.  Box blockIdx.y of a batch: its sorted records (from
// bs.poff), tile offsets [box][ntiles + 1] and grid out [box][N^3].
//
// A tile's workgroup visits the particles of twelve tiles, and of the 32
// stencil rows of a particle about one in twelve is its own: with a thread a
// particle most lanes idle behind masks.  So the workgroup first lists, TH
// particles at a time, the (particle, grid, z row) entries that land in the
// tile, and then works through full rounds of TH entries, each thread
// recomputing its particle's stencil and adding up to four y rows.  Integer
// sums, so neither the order of the list nor that of the atomics matters.
// The lines' part runs on FFT_THREADS threads, whatever TH.
//
// The other half of the kernel is the lines: zeroing, conversion, FFT and
// store.  A thread converts and stores cells of one line, with no index
// division, all of them between two barriers; at compile-time N the FFT's last
// stage stores straight to the grid.  Measured, float, before and
// after: N = 360 with 2e4 points 0.41 -> 0.30 ms, 1e6 0.563 -> 0.463 (0.475
// without the last stage's stores), 4e6 1.19 -> 1.09; N = 512, 4e6 2.16 -> 1.88;
// N = 256, 3e5 0.174 -> 0.151; double, N = 360, 1e6 0.655 -> 0.54.  (Fixed
// point by adding 1.5 * 2^52 instead of the float64 conversion, under a branch on
// the weight's size: 0.51 -> 0.57 at N = 360.)
template <typename T, int NC, bool FFTX, int TH>
__global__ __launch_bounds__(TH) void k_assign_lines(
    const float4* __restrict__ rec, const unsigned* __restrict__ tile_off, const AssignBoxes bs,
    FftShape sh, AssignTiling at, const cplx<T>* __restrict__ tw, cplx<T>* __restrict__ out) {
  const int box = blockIdx.y;
  const int64_t np = bs.np[box];
  const PcsMap pm = bs.pm[box];
  const double scale = bs.scale[box];
  rec += bs.poff[box];
  tile_off += (int64_t)box * (at.nty * at.ntz + 1);
  out += (int64_t)box * n_of<NC>(sh) * n_of<NC>(sh) * n_of<NC>(sh);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  unsigned long long* acc = reinterpret_cast<unsigned long long*>(smem_raw);
  __shared__ int src[64];
  __shared__ unsigned sbeg[64];
  __shared__ int64_t pre[65];
  __shared__ int nsrc_s, nq_s;
  const int N = n_of<NC>(sh);
  const int y0 = (int)(blockIdx.x % at.nty) * at.ty, z0 = (int)(blockIdx.x / at.nty) * at.tz;
  const int y1 = min(y0 + at.ty, N), z1 = min(z0 + at.tz, N);
  const int nl = at.ty * at.tz;
  const int ncell = nl * N;
  unsigned* q_rec = reinterpret_cast<unsigned*>(smem_raw + (size_t)16 * ncell);
  unsigned char* q_row = reinterpret_cast<unsigned char*>(q_rec + assign_queue(TH));
  for (int i = threadIdx.x; i < ncell; i += TH)
    reinterpret_cast<ulonglong2*>(acc)[i] = make_ulonglong2(0ull, 0ull);
  if (threadIdx.x == 0) {
    int sy[8], sz[8];
    const int ny = source_tiles(y0, y1, N, at.ty, sy);
    const int nz = source_tiles(z0, z1, N, at.tz, sz);
    int n = 0;
    for (int b = 0; b < nz; ++b)
      for (int a = 0; a < ny; ++a) src[n++] = sz[b] * at.nty + sy[a];
    nsrc_s = n;
    nq_s = 0;
  }
  __syncthreads();
  const int nsrc = nsrc_s;
  if ((int)threadIdx.x < nsrc) {
    const unsigned key = (unsigned)src[threadIdx.x];
    // records of tile key: [tile_off[key], tile_off[key + 1])
    const unsigned beg = np > 0 ? tile_off[key] : 0u;
    sbeg[threadIdx.x] = beg;
    pre[threadIdx.x + 1] = np > 0 ? (int64_t)(tile_off[key + 1] - beg) : 0;  // length for now
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t s = 0;
    pre[0] = 0;
    for (int u = 0; u < nsrc; ++u) {
      s += pre[u + 1];
      pre[u + 1] = s;
    }
  }
  __syncthreads();
  const int64_t total = pre[nsrc];
  const int lane = (int)(threadIdx.x & 63);
  const unsigned long long below = (1ull << lane) - 1ull;
  auto add_row = [&](const float4& r, int code) {
    const bool shift = (code & 4) != 0;
    const int g = shift ? 1 : 0, c = code & 3;
    int ex, ey, ez;
    T wx[4], wy[4], wz[4];
    pcs_weights(pcs_coord(r.x, pm, shift, N, &ex), wx);
    pcs_weights(pcs_coord(r.y, pm, shift, N, &ey), wy);
    pcs_weights(pcs_coord(r.z, pm, shift, N, &ez), wz);
    const T wzc = c & 2 ? (c & 1 ? wz[3] : wz[2]) : (c & 1 ? wz[1] : wz[0]);
    const int zrow = (wrap1(ez + c - 1, N) - z0) * at.ty;
    const T we = (T)r.w;
    int ix[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) ix[a] = 2 * wrap1(ex + a - 1, N) + g;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int yy = wrap1(ey + b - 1, N);
      if (yy < y0 || yy >= y1) continue;
      unsigned long long* row = acc + 2 * (zrow + yy - y0) * N;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        // estimator.f:380-508: hx*hy*hz*we, left to right
        const T v = wmul(wmul(wmul(wx[a], wy[b]), wzc), we);
        const long long qv = __double2ll_rn((double)v * scale);
        atomicAdd(row + ix[a], (unsigned long long)qv);
      }
    }
  };
  int s = 0;
  unsigned at_rec = 0;  // this thread's record of the batch
  auto locate = [&](int64_t q) {
    while (q >= pre[s + 1]) ++s;
    return sbeg[s] + (unsigned)(q - pre[s]);
  };
  float4 nxt = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if ((int64_t)threadIdx.x < total) nxt = rec[at_rec = locate(threadIdx.x)];
  for (int64_t q0 = 0; q0 < total; q0 += TH) {
    const float4 r = nxt;
    const unsigned my_rec = at_rec;
    const bool has = q0 + threadIdx.x < total;
    if (q0 + TH + threadIdx.x < total) nxt = rec[at_rec = locate(q0 + TH + threadIdx.x)];
    // which of the 2 x 4 z stencil rows land in the tile
    unsigned hits = 0;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      int cy, cz;
      (void)pcs_coord(r.y, pm, g == 1, N, &cy);
      (void)pcs_coord(r.z, pm, g == 1, N, &cz);
      bool hit_y = false;
      unsigned hz = 0;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int yy = wrap1(cy + c - 1, N), zz = wrap1(cz + c - 1, N);
        hit_y = hit_y || (yy >= y0 && yy < y1);
        if (zz >= z0 && zz < z1) hz |= 1u << (4 * g + c);
      }
      if (has && hit_y) hits |= hz;
    }
    // the wave's entries at `base`, stencil row by stencil row
    int n_wave = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) n_wave += __popcll(__ballot((hits >> k) & 1u));
    int base = 0;
    if (lane == 0 && n_wave > 0) base = atomicAdd(&nq_s, n_wave);
    base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const unsigned long long m = __ballot((hits >> k) & 1u);
      if ((hits >> k) & 1u) {
        const int i = base + __popcll(m & below);
        q_rec[i] = my_rec;
        q_row[i] = (unsigned char)k;
      }
      base += __popcll(m);
    }
    __syncthreads();
    const int n = nq_s;
    const int work = q0 + TH < total ? n / TH * TH : n;
    // two rounds at a time, so that their records are loaded together
    for (int i0 = (int)threadIdx.x; i0 < work; i0 += 2 * TH) {
      const int i1 = i0 + TH;
      const float4 r0 = rec[q_rec[i0]];
      float4 r1 = r0;
      if (i1 < work) r1 = rec[q_rec[i1]];
      add_row(r0, q_row[i0]);
      if (i1 < work) add_row(r1, q_row[i1]);
    }
    // the rest (fewer than TH) to the front
    unsigned kr = 0;
    unsigned char kc = 0;
    const bool keep = work + (int)threadIdx.x < n;
    if (keep) { kr = q_rec[work + threadIdx.x]; kc = q_row[work + threadIdx.x]; }
    __syncthreads();
    if (keep) { q_rec[threadIdx.x] = kr; q_row[threadIdx.x] = kc; }
    if (threadIdx.x == 0) nq_s = n - work;
    __syncthreads();
  }
  __syncthreads();
  // The waves past the lines' threads end here, whole waves as TH and FFT_THREADS
  // are multiples of 64, and the barriers below are the others': S_BARRIER waits
  // for the waves of the workgroup that have not ended (CDNA3 and CDNA4 ISA).
  if (TH > FFT_THREADS && threadIdx.x >= FFT_THREADS) return;
  // a thread converts and stores the cells x = x0, x0 + TP, ... of one line
  const double inv = 1.0 / scale;
  const int TP = FFT_THREADS / nl;
  const int line = (int)threadIdx.x / TP, xf = (int)threadIdx.x - line * TP;
  const int ly = line % at.ty, lz = line / at.ty;
  const bool stored = line < nl && y0 + ly < y1 && z0 + lz < z1;
  cplx<T>* dst = out + ((int64_t)(z0 + lz) * N + (y0 + ly)) * N;
  if constexpr (!FFTX) {
    if (stored)
      for (int x = xf; x < N; x += TP) {
        const unsigned long long* a = acc + 2 * (line * N + x);
        dst[x] = mk((T)((double)(long long)a[0] * inv), (T)((double)(long long)a[1] * inv));
      }
  } else {
    // To complex lines of stride N+1 in the same memory.  Compile-time N: all
    // of a thread's cells are in registers between two barriers.  Runtime N:
    // CR rounds of cells at a time; cell e moves from byte 16e to byte
    // sizeof(cplx<T>)*(e + line), for 8-byte complex into cells already read
    // when the batches go up, for 16-byte complex when they go down.
    cplx<T>* lds = reinterpret_cast<cplx<T>*>(smem_raw);
    const int lstride = N + 1;
    auto cell = [&](int e) {
      return mk((T)((double)(long long)acc[2 * e] * inv), (T)((double)(long long)acc[2 * e + 1] * inv));
    };
    if constexpr (NC > 0) {
      constexpr int TPC = FFT_THREADS / assign_lines_max<T, NC>(), U = (NC + TPC - 1) / TPC;
      cplx<T> v[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        v[u] = cell(min(line, nl - 1) * N + min(xf + u * TP, N - 1));
      __syncthreads();
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (line < nl && xf + u * TP < N) lds[line * lstride + xf + u * TP] = v[u];
    } else {
      constexpr int CR = 8, CB = CR * FFT_THREADS;
      const int nbatch = (ncell + CB - 1) / CB;
      for (int bt = 0; bt < nbatch; ++bt) {
        const int e0 = (sizeof(cplx<T>) < 16 ? bt : nbatch - 1 - bt) * CB + (int)threadIdx.x;
        cplx<T> v[CR];
#pragma unroll
        for (int u = 0; u < CR; ++u) v[u] = cell(min(e0 + u * FFT_THREADS, ncell - 1));
        __syncthreads();
#pragma unroll
        for (int u = 0; u < CR; ++u) {
          const int e = e0 + u * FFT_THREADS;
          if (e < ncell) lds[e + e / N] = v[u];
        }
        __syncthreads();
      }
    }
    cplx<T>* twl = lds + nl * lstride;
    stage_twiddles(twl, tw, N);
    __syncthreads();
    if constexpr (NC > 0) {
      fft_tile_store<NC, 1, T, assign_lines_max<T, NC>(), false>(
          lds, nl, lstride, twl, [&](int l, int n, cplx<T> v) {
            const int y = y0 + l % at.ty, zz = z0 + l / at.ty;
            if (y < y1 && zz < z1) out[((int64_t)zz * N + y) * N + n] = v;
          });
    } else {
      fft_tile<NC, 1, T, assign_lines_max<T, NC>()>(lds, sh, nl, lstride, twl);
      if (stored)
        for (int x = xf; x < N; x += TP) dst[x] = lds[line * lstride + x];
    }
  }
}

// Fixed-point exponent: every cell is bounded by 64 * sum|w| (per-axis PCS
// weight <= 4), keep that below 2^62.
int fixed_point_exponent(double wsum_abs) {
  double bound = 64.0 * (wsum_abs > 1.0 ? wsum_abs : 1.0);
  int e = 62 - (int)ceil(log2(bound));
  if (e > 40) e = 40;
  if (e < 0) e = 0;
  return e;
}

template <typename T, int NC, bool FFTX, int TH>
static int assign_lines_th(psx_ctx* ctx, const float4* rec, const unsigned* off,
                           const AssignBoxes& bs, int nbox, int N, AssignTiling at, cplx<T>* grid) {
  const FftPlan* p;
  PSX_TRY(get_fft_plan(ctx, N, &p));
  const size_t nl = (size_t)at.ty * at.tz;
  size_t lds = 16 * nl * N + assign_queue(TH) * (sizeof(unsigned) + 1);
  if (FFTX) lds = std::max(lds, sizeof(cplx<T>) * (nl * (N + 1) + N));
  auto kern = k_assign_lines<T, NC, FFTX, TH>;
  PSX_TRY(set_lds(kern, lds));
  launch_timed(ctx, "k_assign_lines", kern, dim3((unsigned)(at.nty * at.ntz), (unsigned)nbox),
               dim3(TH), lds, rec, off, bs, p->shape, at, plan_tw<T>(p), grid);
  PSX_CHECK_LAUNCH();
  return PSX_OK;
}

// Small grids have fewer workgroups than the chip takes at once, and a wave of
// one waits for its LDS atomics and records: up to two workgroups a CU (512
// tiles, N = 64) they get 16 waves instead of 4.  Measured, float, 256 against
// 1024 threads: N = 40 with 2e4 points 0.030 -> 0.021 ms, 512000 0.358 -> 0.184;
// N = 64, 2e4 0.018 -> 0.017, 2e6 0.60 -> 0.415; above, the wide ones lose what
// is sparse: N = 80 (800 tiles) 2e4 0.026 -> 0.046, 5e5 0.168 -> 0.189, N = 128
// 2e4 0.034 -> 0.056.
//
// The double kernel of a run-time length needs all 128 registers of a thread
// in a workgroup of 1024 and spills (40 bytes a lane), so a CU holds one: past
// 256 tiles a second round starts, which costs more than the wide workgroups
// gain until there is a particle a cell.  Measured, double, the whole field, 256
// against 1024 threads at 0.02, 0.5, 0.9, 1, 2 and 8 particles a cell: N = 50
// (325 tiles) 0.048 / 0.061, 0.106 / 0.111, 0.152 / 0.153, 0.164 / 0.163, 0.281 /
// 0.268, 0.961 / 0.871 ms; N = 60 (450) 0.049 / 0.062, 0.122 / 0.126, 0.181 /
// 0.183, 0.197 / 0.193, 0.339 / 0.325, 1.21 / 1.12.
// Up to 256 tiles, N = 40 (200), at 0.02, 0.5 and 8: 0.042 -> 0.043, 0.079 ->
// 0.069, 0.64 -> 0.49; compile-time N = 64 (512, no spill): 0.038 -> 0.040,
// 0.116 -> 0.106, 1.29 -> 1.11.
constexpr int ASSIGN_WIDE_TILES = 512, ASSIGN_WIDE_THREADS = 1024, ASSIGN_CUS = 256;

template <typename T, int NC>
static int assign_lines_n(psx_ctx* ctx, const float4* rec, const unsigned* off,
                          const AssignBoxes& bs, int nbox, int N, AssignTiling at, cplx<T>* grid,
                          bool fft_x) {
  if (!fft_x)
    return assign_lines_th<T, 0, false, FFT_THREADS>(ctx, rec, off, bs, nbox, N, at, grid);
  if constexpr (NC <= 64) {
    const int64_t tiles = (int64_t)at.nty * at.ntz * nbox;
    int64_t total = 0;
    for (int b = 0; b < nbox; ++b) total += bs.np[b];
    const bool second_round = sizeof(T) == 8 && NC == 0 && tiles > ASSIGN_CUS;
    if (tiles <= ASSIGN_WIDE_TILES && (!second_round || total >= (int64_t)nbox * N * N * N))
      return assign_lines_th<T, NC, true, ASSIGN_WIDE_THREADS>(ctx, rec, off, bs, nbox, N, at, grid);
  }
  return assign_lines_th<T, NC, true, FFT_THREADS>(ctx, rec, off, bs, nbox, N, at, grid);
}

#define PSX_CASE_N(n)                                                                         \
  case n:                                                                                     \
    return assign_lines_n<T, n>(ctx, rec, o, bs, nbox, N, at, grid, fft_x);

// nbox boxes (particles xyz[b], weights w[b] or null, counts np[b], maps
// pm[b], fixed-point scales scale[b]) into nbox grids back to back.
template <typename T>
static int assign_grid_t(psx_ctx* ctx, int nbox, const float* const* xyz, const float* const* w,
                         const int64_t* np, const PcsMap* pm, const double* scale, int N,
                         cplx<T>* grid, bool fft_x) {
  PSX_REQUIRE(nbox >= 1 && nbox <= PSX_MAX_BATCH, "batch of 1 to 16 boxes");
  const AssignTiling at = assign_tiling<T>(N);
  AssignBoxes bs{};
  int64_t total = 0, maxnp = 0;
  for (int b = 0; b < nbox; ++b) {
    PSX_REQUIRE(np[b] >= 0 && np[b] < (int64_t)1 << 32, "more than 2^32 - 1 particles");
    bs.xyz[b] = xyz[b];
    bs.w[b] = w ? w[b] : nullptr;
    bs.np[b] = np[b];
    bs.poff[b] = total;
    bs.pm[b] = pm[b];
    bs.scale[b] = scale[b];
    total += np[b];
    maxnp = std::max(maxnp, np[b]);
  }
  const int64_t ntiles = (int64_t)at.nty * at.ntz;
  const float4* rec = nullptr;
  unsigned* o = nullptr;
  PSX_TRY(ctx_buffer(ctx, "tile_off", (size_t)nbox * (ntiles + 1) * 4, (void**)&o));
  if (total > 0) {
    // counting sort by assignment tile into (x, y, z, w) records, per box
    unsigned *count, *key, *rank;
    float4* r;
    PSX_TRY(ctx_buffer(ctx, "tile_count", (size_t)nbox * ntiles * 4, (void**)&count));
    PSX_TRY(ctx_buffer(ctx, "particle_tile", (size_t)total * 4, (void**)&key));
    PSX_TRY(ctx_buffer(ctx, "particle_rank", (size_t)total * 4, (void**)&rank));
    PSX_TRY(ctx_buffer(ctx, "sorted_particles", (size_t)total * sizeof(float4), (void**)&r));
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)cdiv(nbox * ntiles, 256)), dim3(256), 0,
                       ctx->stream, count, nbox * ntiles);
    PSX_CHECK_LAUNCH();
    const dim3 pgrid((unsigned)cdiv(maxnp, 256), (unsigned)nbox);
    hipLaunchKernelGGL(k_tile_count, pgrid, dim3(256), 0, ctx->stream, bs, N, at, count, key, rank);
    PSX_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_tile_scan, dim3(1, nbox), dim3(SCAN_THREADS), 0, ctx->stream,
                       (const unsigned*)count, (int)ntiles, o);
    PSX_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_tile_scatter, pgrid, dim3(256), 0, ctx->stream, bs, (const unsigned*)key,
                       (const unsigned*)rank, (const unsigned*)o, (int)ntiles, r);
    PSX_CHECK_LAUNCH();
    rec = r;
  }
  // boxes without particles read no records (their np is 0)
  if (!fft_x) return assign_lines_n<T, 0>(ctx, rec, o, bs, nbox, N, at, grid, false);
  switch (N) {
    PSX_FFT_SIZES(PSX_CASE_N)
    default: return assign_lines_n<T, 0>(ctx, rec, o, bs, nbox, N, at, grid, true);
  }
}
#undef PSX_CASE_N

int launch_assign_grid_batch(psx_ctx* ctx, int nbox, const float* const* xyz,
                             const float* const* w, const int64_t* np, const PcsMap* pm,
                             const double* scale, int N, void* grid, int prec, bool fft_x) {
  if (prec == PSX_PREC_F64)
    return assign_grid_t<double>(ctx, nbox, xyz, w, np, pm, scale, N, (cplx<double>*)grid, fft_x);
  return assign_grid_t<float>(ctx, nbox, xyz, w, np, pm, scale, N, (cplx<float>*)grid, fft_x);
}

int launch_assign_grid(psx_ctx* ctx, const float* xyz, const float* w, int64_t np, int N,
                       PcsMap pm, double scale, void* grid, int prec, bool fft_x) {
  return launch_assign_grid_batch(ctx, 1, &xyz, &w, &np, &pm, &scale, N, grid, prec, fft_x);
}

// Unit field delta = 1 (the shell indicators of _counts_Bk123), complex double.
__global__ void k_fill_unit(double* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    p[2 * i] = 1.0;
    p[2 * i + 1] = 0.0;
  }
}

int launch_fill_unit(psx_ctx* ctx, double* half, int64_t n) {
  hipLaunchKernelGGL(k_fill_unit, dim3((unsigned)std::min<int64_t>(cdiv(n, 256), 8192)), dim3(256),
                     0, ctx->stream, half, n);
  PSX_CHECK_LAUNCH();
  return PSX_OK;
}

// --------------------------------------------------------------- fcomb ----
// estimator.f:605-675.  One thread per loop iteration (ix, iy, iz) in
// [0, N/2]^3.  The eight elements {ix,-ix} x {iy,-iy} x {iz,-iz} are read,
// combined, and the eight stores are replayed in the reference's order on a
// register copy in which aliased indices (0 and N/2) share a slot, so the
// value that survives is the reference's.  Only the x <= N/2 elements are
// written (the half field).  rec[n] is the reference's twiddle recurrence
// xrec = recx^n (complex double); W is the per-axis PCS window.
template <typename T> __device__ __forceinline__ T window_val(const float* Wf, const double* Wd, int n);
template <> __device__ __forceinline__ float window_val<float>(const float* Wf, const double*, int n) { return Wf[n]; }
template <> __device__ __forceinline__ double window_val<double>(const float*, const double* Wd, int n) { return Wd[n]; }

template <typename T>
__device__ __forceinline__ cplx<T> slot_get(const cplx<T> (&m)[8], int s) {
  cplx<T> r = m[0];
#pragma unroll
  for (int k = 1; k < 8; ++k) if (s == k) r = m[k];
  return r;
}
template <typename T>
__device__ __forceinline__ void slot_put(cplx<T> (&m)[8], int s, cplx<T> v) {
#pragma unroll
  for (int k = 0; k < 8; ++k) if (s == k) m[k] = v;
}

// Normalisations of the boxes of a batch (kernel argument).
template <typename T> struct FcombCoef {
  T cf[PSX_MAX_BATCH];
};

// Iteration (ix, iy, iz) of estimator.f:646-665: from the eight values v[s]
// at (xs[s>>2], ys[(s>>1)&1], zs[s&1]) (xs = {ix, -ix mod N}, ...) the
// eight stores in the reference's order; m[canon(xb, yb, zb)] is then the
// value the iteration leaves at (xs[xb], ys[yb], zs[zb]) -- where indices
// alias (0 and N/2) the last store wins.
struct FcombSlots {
  bool ax, ay, az;
  __device__ __forceinline__ int canon(int xb, int yb, int zb) const {
    return ((xb && !ax) ? 4 : 0) + ((yb && !ay) ? 2 : 0) + ((zb && !az) ? 1 : 0);
  }
};

template <typename T>
__device__ __forceinline__ void fcomb_iteration(cplx<T> (&m)[8], const FcombSlots& sl, int ix,
                                                int iy, int iz, T cf, const c64* __restrict__ rec,
                                                const float* __restrict__ Wf,
                                                const double* __restrict__ Wd) {
  // twiddles in double (estimator.f:650-653), rounded to T
  const c64 xr = rec[ix], yr = rec[iy], zr = rec[iz];
  const c64 ixr = mk(-xr.im, xr.re);
  const c64 cma = ixr * yr * zr;
  const c64 cmb = ixr * yr * conj(zr);
  const c64 cmc = ixr * conj(yr) * zr;
  const c64 cmd = ixr * conj(yr * zr);
  const cplx<T> one = mk(T(1), T(0));
  auto cv = [](c64 a) { return mk((T)a.re, (T)a.im); };
  const cplx<T> A = cv(cma), B = cv(cmb), C = cv(cmc), D = cv(cmd);
  const T cfac = cf / (window_val<T>(Wf, Wd, ix) * window_val<T>(Wf, Wd, iy) * window_val<T>(Wf, Wd, iz));
  const cplx<T> c000 = m[0] * (one - A) + conj(m[7]) * (one + A);
  const cplx<T> c001 = m[1] * (one - B) + conj(m[6]) * (one + B);
  const cplx<T> c010 = m[2] * (one - C) + conj(m[5]) * (one + C);
  const cplx<T> c011 = m[3] * (one - D) + conj(m[4]) * (one + D);
  slot_put(m, sl.canon(0, 0, 0), c000 * cfac);
  slot_put(m, sl.canon(0, 0, 1), c001 * cfac);
  slot_put(m, sl.canon(0, 1, 0), c010 * cfac);
  slot_put(m, sl.canon(0, 1, 1), c011 * cfac);
  slot_put(m, sl.canon(1, 0, 0), conj(slot_get(m, sl.canon(0, 1, 1))));
  slot_put(m, sl.canon(1, 0, 1), conj(slot_get(m, sl.canon(0, 1, 0))));
  slot_put(m, sl.canon(1, 1, 0), conj(slot_get(m, sl.canon(0, 0, 1))));
  slot_put(m, sl.canon(1, 1, 1), conj(slot_get(m, sl.canon(0, 0, 0))));
}

// The value that iteration leaves at (ix, +-iy, +-iz) (*q = 2 yb + zb) as one
// of its combinations c000, c001, c010, c011 (*q on return) or the conjugate
// of one (*cj): stores 0..3 put c_q, store p >= 4 the conjugate of what slot
// (0, 7 - p) then holds; the last store into a slot decides.
__device__ __forceinline__ void fcomb_survivor(const FcombSlots& sl, int* q, bool* cj) {
  int slot = sl.canon(0, *q >> 1, *q & 1), before = 8;
  bool conjugate = false;
  for (;;) {
    int p = before - 1;
    while (sl.canon(p >> 2, (p >> 1) & 1, p & 1) != slot) --p;  // its own store 0..3 at the latest
    if (p < 4) {
      *q = p;
      *cj = conjugate;
      return;
    }
    slot = sl.canon(0, ((7 - p) >> 1) & 1, (7 - p) & 1);
    before = p;
    conjugate = !conjugate;
  }
}

// Box blockIdx.y of a batch: grid F [box][N^3], half field Hh [box][N^2 (N/2+1)].
template <typename T>
__global__ __launch_bounds__(256) void k_fcomb(const cplx<T>* __restrict__ F, cplx<T>* __restrict__ Hh, int N,
                                               FcombCoef<T> coef, const c64* __restrict__ rec,
                                               const float* __restrict__ Wf,
                                               const double* __restrict__ Wd) {
  const int Nh = N / 2 + 1;
  F += (int64_t)blockIdx.y * N * N * N;
  Hh += (int64_t)blockIdx.y * N * N * Nh;
  const T cf = coef.cf[blockIdx.y];
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (int64_t)Nh * Nh * Nh) return;
  const int ix = (int)(id % Nh);
  const int iy = (int)((id / Nh) % Nh);
  const int iz = (int)(id / ((int64_t)Nh * Nh));
  const int xs[2] = {ix, (N - ix) % N};
  const int ys[2] = {iy, (N - iy) % N};
  const int zs[2] = {iz, (N - iz) % N};
  const FcombSlots sl{xs[0] == xs[1], ys[0] == ys[1], zs[0] == zs[1]};
  cplx<T> m[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int xb = s >> 2, yb = (s >> 1) & 1, zb = s & 1;
    m[s] = F[((int64_t)zs[zb] * N + ys[yb]) * N + xs[xb]];
  }
  fcomb_iteration(m, sl, ix, iy, iz, cf, rec, Wf, Wd);
  // half-field elements owned by this iteration: x = ix, y in {iy,-iy}, z in {iz,-iz}
#pragma unroll
  for (int yb = 0; yb < 2; ++yb) {
#pragma unroll
    for (int zb = 0; zb < 2; ++zb) {
      if ((yb && sl.ay) || (zb && sl.az)) continue;
      Hh[((int64_t)zs[zb] * N + ys[yb]) * Nh + ix] = slot_get(m, sl.canon(0, yb, zb));
    }
  }
}

// The z pass of the backward grid FFT with fcomb as its epilogue.  The
// half-field line (x, y), x <= N/2, is the fcomb of the lines (x, y) and
// (-x, -y) after their z transforms: every value the store order of
// iteration (x, |y|, |z|) reads or leaves at (x, y, z) lies on one of them
// (where x, y or z alias, the other lines of the iteration coincide with
// these two).  A tile holds tp such line pairs, consecutive x at one y; the
// line transforms are those of k_fft_lines.  An element is formed from its two
// values and fcomb_survivor instead of the eight stores that k_fcomb replays.
//
// The lines fill the LDS (two or three workgroups a CU), so between loads and
// stores the kernel is bound by its own instructions and latencies.  A thread
// stays on one line of the loads and on one pair of the epilogue: addresses
// are a base plus a constant stride and the x and y factors of the twiddle and
// the window are formed once (no index divisions, a third of the float64
// products), and nothing is kept in scratch memory.  Measured (float): N = 360
// 0.288 -> 0.254 ms, 16 boxes of 128 0.193 -> 0.127, 300 (runtime N) 0.52 ->
// 0.235, 512 0.98 -> 0.95; reading the grid and writing the half field once
// takes 0.12, 0.09, 0.07 and 0.33 at 4.8 TB/s.  (Several tiles a workgroup with
// the next one's elements loaded ahead into registers: 512 0.83, but 0.151 for
// the 16 boxes and 0.25 -> 0.25 at 360, where the registers cost a workgroup.)
template <typename T, int NC>
__global__ __launch_bounds__(FFT_THREADS) void k_fft_zcomb(const cplx<T>* __restrict__ F,
                                                            cplx<T>* __restrict__ Hh, FftShape sh,
                                                            const cplx<T>* __restrict__ tw,
                                                            FcombCoef<T> coef,
                                                            const c64* __restrict__ rec,
                                                            const float* __restrict__ Wf,
                                                            const double* __restrict__ Wd) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cplx<T>* lds = reinterpret_cast<cplx<T>*>(smem_raw);
  const int N = n_of<NC>(sh), Nh = N / 2 + 1, lstride = N + 1;
  const int64_t NN = (int64_t)N * N;
  F += (int64_t)blockIdx.y * NN * N;
  Hh += (int64_t)blockIdx.y * NN * Nh;
  const T cf = coef.cf[blockIdx.y];
  constexpr int ML = Tile<T, NC>::MAXLINES;
  const int tl = NC > 0 ? ML : tile_lines_for(N, TileCfg<T>::ELEMS, TileCfg<T>::LINES);
  const int tp = tl / 2;  // line pairs per tile
  const int ntx = (Nh + tp - 1) / tp;
  // neighbouring x tiles read the two halves of the same 128-byte lines
  const int bx = xcd_local_block((int)blockIdx.x, (int)gridDim.x);
  const int y = bx / ntx, x0 = (bx - y * ntx) * tp, np = min(tp, Nh - x0);
  // line 2c: (x0 + c, y); line 2c + 1: (-(x0 + c), -y); element n along z: rows
  // n0, n0 + RS, ... of one line, U loads in flight
  {
    constexpr int U = 8;
    const int nl = 2 * tp, RS = FFT_THREADS / nl;
    const int n0 = (int)threadIdx.x / nl, l = (int)threadIdx.x - n0 * nl, c = l >> 1;
    if (n0 < RS && c < np) {
      const int xc = x0 + c;
      const int x = (l & 1) && xc > 0 ? N - xc : xc, ym = y > 0 ? N - y : 0;
      const cplx<T>* src = F + (int64_t)((l & 1) ? ym : y) * N + x;
      cplx<T>* dst = lds + l * lstride;
      for (int nb = n0; nb < N; nb += RS * U) {
        cplx<T> v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = src[(int64_t)min(nb + u * RS, N - 1) * NN];
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (nb + u * RS < N) dst[nb + u * RS] = v[u];
      }
    }
  }
  cplx<T>* twl = lds + tl * lstride;
  stage_twiddles(twl, tw, N);
  __syncthreads();
  fft_tile<NC, 1, T, ML>(lds, sh, 2 * np, lstride, twl);
  // epilogue: pair c, rows z0, z0 + RZ, ...
  const int RZ = FFT_THREADS / tp;
  const int zfirst = (int)threadIdx.x / tp, c = (int)threadIdx.x - zfirst * tp;
  if (zfirst >= RZ || c >= np) return;
  const int yb = y > N / 2 ? 1 : 0, iy = yb ? N - y : y, ix = x0 + c;
  const c64 xr = rec[ix], yr = rec[iy];
  const c64 ixr = mk(-xr.im, xr.re);
  const c64 ixy0 = ixr * yr, ixy1 = ixr * conj(yr);
  const T wxy = window_val<T>(Wf, Wd, ix) * window_val<T>(Wf, Wd, iy);
  const cplx<T> one = mk(T(1), T(0));
  const cplx<T>* la = lds + (2 * c) * lstride;      // (ix, y)
  const cplx<T>* lb = lds + (2 * c + 1) * lstride;  // (-ix, -y)
  cplx<T>* dst = Hh + (int64_t)y * Nh + ix;
  const bool ax = ix == 0 || 2 * ix == N, ay = iy == 0 || 2 * iy == N;
  for (int z = zfirst; z < N; z += RZ) {
    const int zb = z > N / 2 ? 1 : 0, iz = zb ? N - z : z, mz = z > 0 ? N - z : 0;
    // The element is the combination c_q (q = 2 yb + zb) of its iteration,
    // or, where an index aliases, the one whose store survives there (cj:
    // conjugated).
    int q = 2 * yb + zb;
    bool cj = false;
    if (ax || ay || z == mz) fcomb_survivor(FcombSlots{ax, ay, z == mz}, &q, &cj);
    const bool yq = (q & 2) != 0, zq = (q & 1) != 0;
    // c_q = v (1 - t) + conj(v') (1 + t) times cfac, v at (ix, +-iy, +-iz)
    // by q and v' its mirror; both lie on the two lines.  The twiddle t in
    // double (estimator.f:650-653), rounded to T.
    const c64 zr = rec[iz];
    const c64 t64 = q == 3 ? ixr * conj(yr * zr) : (yq ? ixy1 : ixy0) * (zq ? conj(zr) : zr);
    const cplx<T> t = mk((T)t64.re, (T)t64.im);
    const T cfac = cf / (wxy * window_val<T>(Wf, Wd, iz));
    const bool same_y = yq == (yb != 0), same_z = zq == (zb != 0);
    const cplx<T> va = (ay || same_y ? la : lb)[same_z ? z : mz];
    const cplx<T> vm = (ax && (ay || !same_y) ? la : lb)[same_z ? mz : z];
    cplx<T> out = (va * (one - t) + conj(vm) * (one + t)) * cfac;
    if (cj) out = conj(out);
    dst[(int64_t)z * N * Nh] = out;
  }
}

template <typename T, int NC>
static int zcomb_n(psx_ctx* ctx, const FftPlan* p, const cplx<T>* F, cplx<T>* Hh, int nbox,
                   const FcombCoef<T>& c) {
  const int N = p->shape.N, Nh = N / 2 + 1;
  const int tl = tile_lines_host<T>(N), tp = tl / 2;
  const size_t lds = ((size_t)tl * (N + 1) + N) * sizeof(cplx<T>);
  auto kern = k_fft_zcomb<T, NC>;
  PSX_TRY(set_lds(kern, lds));
  const dim3 grid((unsigned)((int64_t)N * ((Nh + tp - 1) / tp)), (unsigned)nbox);
  launch_timed(ctx, "k_fft_zcomb", kern, grid, dim3(FFT_THREADS), lds, F, Hh, p->shape,
               plan_tw<T>(p), c, (const c64*)p->rec, p->Wf, p->Wd);
  PSX_CHECK_LAUNCH();
  return PSX_OK;
}

#define PSX_CASE_N(n) \
  case n: return zcomb_n<T, n>(ctx, p, F, Hh, nbox, c);

template <typename T>
static int zcomb_t(psx_ctx* ctx, const FftPlan* p, const cplx<T>* F, cplx<T>* Hh, int nbox,
                   const FcombCoef<T>& c) {
  switch (p->shape.N) {
    PSX_FFT_SIZES(PSX_CASE_N)
    default: return zcomb_n<T, 0>(ctx, p, F, Hh, nbox, c);
  }
}
#undef PSX_CASE_N

int launch_fft_zcomb_batch(psx_ctx* ctx, const void* F, void* Hh, int N, int nbox,
                           const double* sumw, int prec) {
  PSX_REQUIRE(nbox >= 1 && nbox <= PSX_MAX_BATCH, "batch of 1 to 16 boxes");
  PSX_REQUIRE(tile_lines_host<double>(N) >= 2, "grid too large for the fused z pass");
  const FftPlan* p;
  PSX_TRY(get_fft_plan(ctx, N, &p));
  if (prec == PSX_PREC_F64) {
    FcombCoef<double> c{};
    // cf = 1/(6^3 * 4 * N) with N = sum w as float32 (estimator.f:615)
    for (int b = 0; b < nbox; ++b) c.cf[b] = 1.0 / (216.0 * 4.0 * (double)(float)sumw[b]);
    return zcomb_t<double>(ctx, p, (const cplx<double>*)F, (cplx<double>*)Hh, nbox, c);
  }
  FcombCoef<float> c{};
  for (int b = 0; b < nbox; ++b) c.cf[b] = 1.0f / (864.0f * (float)sumw[b]);
  return zcomb_t<float>(ctx, p, (const cplx<float>*)F, (cplx<float>*)Hh, nbox, c);
}

// nbox grids back to back -> nbox half fields back to back.
int launch_fcomb_batch(psx_ctx* ctx, const void* F, void* Hh, int N, int nbox, const double* sumw,
                       int prec, const void* rec, const float* Wf, const double* Wd) {
  PSX_REQUIRE(nbox >= 1 && nbox <= PSX_MAX_BATCH, "batch of 1 to 16 boxes");
  const int64_t Nh = N / 2 + 1;
  const int64_t n = Nh * Nh * Nh;
  const dim3 grid((unsigned)cdiv(n, 256), nbox);
  if (prec == PSX_PREC_F64) {
    FcombCoef<double> c{};
    // cf = 1/(6^3 * 4 * N) with N = sum w as float32 (estimator.f:615)
    for (int b = 0; b < nbox; ++b) c.cf[b] = 1.0 / (216.0 * 4.0 * (double)(float)sumw[b]);
    hipLaunchKernelGGL(k_fcomb<double>, grid, dim3(256), 0, ctx->stream, (const cplx<double>*)F,
                       (cplx<double>*)Hh, N, c, (const c64*)rec, Wf, Wd);
  } else {
    FcombCoef<float> c{};
    for (int b = 0; b < nbox; ++b) c.cf[b] = 1.0f / (864.0f * (float)sumw[b]);
    hipLaunchKernelGGL(k_fcomb<float>, grid, dim3(256), 0, ctx->stream, (const cplx<float>*)F,
                       (cplx<float>*)Hh, N, c, (const c64*)rec, Wf, Wd);
  }
  PSX_CHECK_LAUNCH();
  return PSX_OK;
}

int launch_fcomb(psx_ctx* ctx, const void* F, void* Hh, int N, double sumw, int prec,
                 const void* rec, const float* Wf, const double* Wd) {
  return launch_fcomb_batch(ctx, F, Hh, N, 1, &sumw, prec, rec, Wf, Wd);
}

// ------------------------------------------------- half <-> full fields ----
// Hermitian part of an arbitrary full field (any strides, element type TI),
// kept on x <= N/2: H(k) = (F(k) + conj F(-k)) / 2.  Re FFT of a field equals
// the FFT of its Hermitian part, so the shell fields of H equal the
// reference's Re(fftn(F * mask)) exactly in exact arithmetic.
template <typename TI, typename T>
__global__ void k_herm_half(const cplx<TI>* __restrict__ F, int64_t sx, int64_t sy, int64_t sz,
                            cplx<T>* __restrict__ Hh, int N) {
  const int Nh = N / 2 + 1;
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (int64_t)Nh * N * N) return;
  const int x = (int)(id % Nh);
  const int y = (int)((id / Nh) % N);
  const int z = (int)(id / ((int64_t)Nh * N));
  const int mx = (N - x) % N, my = (N - y) % N, mz = (N - z) % N;
  const cplx<TI> a = F[x * sx + y * sy + z * sz];
  const cplx<TI> b = F[mx * sx + my * sy + mz * sz];
  Hh[id] = mk((T)(((double)a.re + (double)b.re) * 0.5), (T)(((double)a.im - (double)b.im) * 0.5));
}

// reflect_delta (pyspectrum.py:1134-1157) to a C-order [ix][iy][iz] full field.
template <typename T>
__global__ void k_reflect(const cplx<T>* __restrict__ Hh, cplx<T>* __restrict__ F, int N) {
  const int Nh = N / 2 + 1, hg = N / 2;
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (int64_t)N * N * N) return;
  const int z = (int)(id % N);
  const int y = (int)((id / N) % N);
  const int x = (int)(id / ((int64_t)N * N));
  cplx<T> v;
  if (x < Nh) {
    v = Hh[((int64_t)z * N + y) * Nh + x];
    const bool cx = (x == 0 || x == hg), cy = (y == 0 || y == hg), cz = (z == 0 || z == hg);
    if (cx && cy && cz && !(x == 0 && y == 0 && z == 0)) v.im = T(0);
  } else {
    const int mx = N - x, my = (N - y) % N, mz = (N - z) % N;
    v = conj(Hh[((int64_t)mz * N + my) * Nh + mx]);
  }
  F[id] = v;
}

int launch_herm_half(psx_ctx* ctx, const void* F, int in_prec, int64_t sx, int64_t sy, int64_t sz,
                     void* Hh, int N, int prec) {
  const int64_t n = (int64_t)(N / 2 + 1) * N * N;
  const dim3 grid((unsigned)cdiv(n, 256));
  if (in_prec == PSX_PREC_F64) {
    if (prec == PSX_PREC_F64)
      hipLaunchKernelGGL((k_herm_half<double, double>), grid, dim3(256), 0, ctx->stream,
                         (const cplx<double>*)F, sx, sy, sz, (cplx<double>*)Hh, N);
    else
      hipLaunchKernelGGL((k_herm_half<double, float>), grid, dim3(256), 0, ctx->stream,
                         (const cplx<double>*)F, sx, sy, sz, (cplx<float>*)Hh, N);
  } else {
    if (prec == PSX_PREC_F64)
      hipLaunchKernelGGL((k_herm_half<float, double>), grid, dim3(256), 0, ctx->stream,
                         (const cplx<float>*)F, sx, sy, sz, (cplx<double>*)Hh, N);
    else
      hipLaunchKernelGGL((k_herm_half<float, float>), grid, dim3(256), 0, ctx->stream,
                         (const cplx<float>*)F, sx, sy, sz, (cplx<float>*)Hh, N);
  }
  PSX_CHECK_LAUNCH();
  return PSX_OK;
}

int launch_reflect(psx_ctx* ctx, const void* Hh, void* F, int N, int prec) {
  const int64_t n = (int64_t)N * N * N;
  if (prec == PSX_PREC_F64)
    hipLaunchKernelGGL(k_reflect<double>, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, ctx->stream,
                       (const cplx<double>*)Hh, (cplx<double>*)F, N);
  else
    hipLaunchKernelGGL(k_reflect<float>, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, ctx->stream,
                       (const cplx<float>*)Hh, (cplx<float>*)F, N);
  PSX_CHECK_LAUNCH();
  return PSX_OK;
}

}  // namespace psx
