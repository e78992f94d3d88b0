// k-space binning of |delta|^2: P(k) shells (Pk_periodic), the shell powers
// of the bispectrum (Parseval form of pyspectrum.py:404) and the P_l / P(k,mu)
// estimator of pk_pbox_rsd (estimator.f:155-264).
#include <mutex>

#include "psx_ctx.h"

namespace psx {

// ------------------------------------------------------ runs in a wave ----
// A wave holds 64 consecutive x of one (y, z) row; equal keys form contiguous
// runs of lanes.  First lane of this lane's run, and whether the lane ends it.
struct LaneRun {
  int start;
  bool end;
};

__device__ __forceinline__ LaneRun lane_run(int key, int lane) {
  const int kp = __shfl_up(key, 1, 64);
  const unsigned long long starts = __ballot(lane == 0 || kp != key);
  const unsigned long long upto = starts & (~0ull >> (63 - lane));
  LaneRun r;
  r.start = 63 - __clzll((long long)upto);
  r.end = lane == 63 || ((starts >> (lane + 1 < 64 ? lane + 1 : 63)) & 1ull);
  return r;
}

template <int CTRL, int ROWS> __device__ __forceinline__ double dpp_f64(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// One step of the scan: every lane with `take` adds what the DPP move brings it.
template <int CTRL, int ROWS, int NV>
__device__ __forceinline__ void run_step(double (&v)[NV], bool take) {
#pragma unroll
  for (int e = 0; e < NV; ++e) {
    const double u = dpp_f64<CTRL, ROWS>(v[e]);
    if (take) v[e] += u;
  }
}

// Inclusive scan of v[] over each run in a fixed order: lanes 1, 2, 4 and 8
// below within each row of 16, then the last lane of the previous row into
// rows 1 and 3 and lane 31 into rows 2 and 3.  DPP moves (VALU) instead of
// shuffles, which go through the LDS pipe: that pipe bounded both binning
// kernels.  All 64 lanes must be active.
template <int NV>
__device__ __forceinline__ void run_scan(double (&v)[NV], int lane, int start) {
  const int l = lane & 15;
  run_step<0x111, 0xf, NV>(v, l >= 1 && lane - 1 >= start);
  run_step<0x112, 0xf, NV>(v, l >= 2 && lane - 2 >= start);
  run_step<0x114, 0xf, NV>(v, l >= 4 && lane - 4 >= start);
  run_step<0x118, 0xf, NV>(v, l >= 8 && lane - 8 >= start);
  run_step<0x142, 0xa, NV>(v, (lane & 16) && (lane & 48) - 1 >= start);
  run_step<0x143, 0xc, NV>(v, lane >= 32 && 31 >= start);
}

// ------------------------------------------------------------ bin power ---
// Bins the full field that reflect_delta (pyspectrum.py:1134-1157) builds from
// the half field: 1 <= x < N/2 count twice (the mirror has the same |delta|),
// x = 0 and x = N/2 once, the seven Nyquist corners with Re(delta)^2.
// bin = shell_of_m(|k|^2, step); bins 1..nbins are accumulated (k = kf*|k|).
// Output sums (k, p, n) per bin; the caller divides.
//
// The rows (+-y, +-z) hold the same |k| at each x, so a wave adds the
// |delta|^2 of those (up to four) rows first and bins them once: the bin
// search, the scan and the LDS adds, not the reads of the field, bound the
// kernel.  Measured: Ngrid 512, 256 bins 0.78 -> 0.16 ms; Ngrid 360, 40 bins
// 0.115 -> 0.037 ms (reading the modes inside the last bin at 4.8 TB/s: 0.06 and
// 0.012 ms).
//
// Deterministic: every sum is formed in a fixed order, so the result is
// bit-identical run to run.  A wave takes whole row groups (|y|, |z|), 64
// consecutive x at a time; |k|^2 = x^2 + c grows with x, so the lanes of
// one bin are one contiguous run (and a group or chunk that starts past the
// last bin is skipped with everything after it).  A scan over the lanes sums
// each run, and the run's last lane adds it to the wave's own accumulators
// in LDS (one lane per bin: no two lanes share an address).  The block then
// adds its waves in order and stores a partial per block; k_bin_reduce adds
// the blocks in a fixed order.
constexpr int BP_THREADS = 256, BP_WAVES = BP_THREADS / 64, BP_MAX_BLOCKS = 512;
constexpr int BP_MAX_BINS = 1024;  // LDS: BP_WAVES x 3 x nbins doubles
// Steps above this leave every mode (|k| <= sqrt(3) 512) in shell 0, as this
// one does, and (2b + 3) * step squared stays within 32 bits.
constexpr int BP_MAX_STEP = 2048;

// shell_of_m for m <= 3 * 512^2 and step <= BP_MAX_STEP: an approximate root,
// corrected by the exact bounds ((2b-1) step)^2 <= 4m < ((2b+1) step)^2.
__device__ __forceinline__ int shell_of_m32(int m, int step, float inv_step) {
  int b = (int)(__builtin_amdgcn_sqrtf((float)m) * inv_step + 0.5f);
  const int hi = (2 * b + 1) * step, lo = (2 * b - 1) * step;
  if (4 * m >= hi * hi) ++b;
  else if (b > 0 && 4 * m < lo * lo) --b;
  return b;
}

// The rows of a group: representative (y, z) and its mirrors +-y, +-z.
struct RowGroup {
  int y, z, y2, z2;  // y2 (z2) = y (z) when the row is its own mirror
  __device__ __forceinline__ int rows() const { return (y2 != y ? 2 : 1) * (z2 != z ? 2 : 1); }
};

__device__ __forceinline__ RowGroup row_group(int y, int z, int N, bool fold_y, bool fold_z) {
  RowGroup g;
  g.y = y; g.z = z;
  g.y2 = fold_y && y > 0 ? N - y : y;
  g.z2 = fold_z && z > 0 ? N - z : z;
  return g;
}

// Values x of the group's rows: v[0..3], absent mirrors zero.
template <typename T>
__device__ __forceinline__ void load_group(const cplx<T>* __restrict__ Hh, const RowGroup& g, int N,
                                           int Nh, int x, bool on, cplx<T> (&v)[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = mk(T(0), T(0));
  if (!on) return;
  const bool my = g.y2 != g.y, mz = g.z2 != g.z;
  v[0] = Hh[((int64_t)g.z * N + g.y) * Nh + x];
  if (my) v[1] = Hh[((int64_t)g.z * N + g.y2) * Nh + x];
  if (mz) v[2] = Hh[((int64_t)g.z2 * N + g.y) * Nh + x];
  if (my && mz) v[3] = Hh[((int64_t)g.z2 * N + g.y2) * Nh + x];
}

template <typename T>
__global__ __launch_bounds__(BP_THREADS) void k_bin_power(const cplx<T>* __restrict__ Hh, int N,
                                                          int step, int nbins, double kf,
                                                          int64_t mlast64,
                                                          double* __restrict__ part) {
  // box blockIdx.y of a batch: its half field and its block partials
  Hh += (int64_t)blockIdx.y * N * N * (N / 2 + 1);
  part += (int64_t)blockIdx.y * gridDim.x * 3 * nbins;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double* accw = reinterpret_cast<double*>(smem_raw);  // [BP_WAVES][3][nbins]
  for (int i = threadIdx.x; i < BP_WAVES * 3 * nbins; i += BP_THREADS) accw[i] = 0.0;
  __syncthreads();
  const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
  double* acc = accw + wave * 3 * nbins;
  const int Nh = N / 2 + 1, hg = N / 2, ngroups = Nh * Nh, gstride = (int)gridDim.x * BP_WAVES;
  const float inv_step = 1.0f / (float)step;
  const int mlast = (int)min(mlast64, (int64_t)1 << 30);  // largest |k|^2 of bin nbins
  // the wave's chunks: groups grp, grp + gstride, ..., each 64 x at a time
  int grp = (int)blockIdx.x * BP_WAVES + wave, x0 = 0;
  auto group_c = [&](int g) {
    const int z = g / Nh, y = g - z * Nh;
    return y * y + z * z;
  };
  auto settle = [&]() {  // the next chunk with a mode that is not past the last bin
    while (grp < ngroups) {
      if (x0 < Nh && group_c(grp) + x0 * x0 <= mlast) return;
      grp += gstride;
      x0 = 0;
    }
  };
  cplx<T> nxt[4];
  auto fetch = [&]() {
    const int z = grp / Nh, y = grp - z * Nh;
    load_group(Hh, row_group(y, z, N, y < hg, z < hg), N, Nh, x0 + lane,
               grp < ngroups && x0 + lane < Nh, nxt);
  };
  settle();
  fetch();
  while (grp < ngroups) {
    const int z = grp / Nh, y = grp - z * Nh, xb = x0, x = x0 + lane;
    const RowGroup g = row_group(y, z, N, y < hg, z < hg);
    cplx<T> cur[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) cur[k] = nxt[k];
    x0 += 64;
    settle();
    fetch();
    int key = -1;
    double v[2] = {0.0, 0.0};
    const double nr = (double)g.rows();
    if (x < Nh) {
      const int m = y * y + z * z + x * x;
      const int bin = shell_of_m32(m, step, inv_step);
      if (bin >= 1 && bin <= nbins) {
        const bool xe = (x == 0 || x == hg);
        if (xe && (y == 0 || y == hg) && (z == 0 || z == hg)) cur[0].im = T(0);
        double p = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          p += (double)cur[k].re * (double)cur[k].re + (double)cur[k].im * (double)cur[k].im;
        const double w = xe ? 1.0 : 2.0;
        key = bin - 1;
        v[0] = (w * nr) * (kf * sqrt((double)m));
        v[1] = w * p;
      }
    }
    // keys -1 (outside 1..nbins or x >= Nh) only lead or trail the valid lanes
    if (__ballot(key >= 0) == 0) continue;
    const LaneRun r = lane_run(key, lane);
    run_scan(v, lane, r.start);
    if (key >= 0 && r.end) {
      const int edges = (xb + r.start == 0 ? 1 : 0) + (x == hg ? 1 : 0);
      acc[key] += v[0];
      acc[nbins + key] += v[1];
      acc[2 * nbins + key] += nr * (double)(2 * (lane - r.start + 1) - edges);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 3 * nbins; i += BP_THREADS) {
    double s = accw[i];
#pragma unroll
    for (int w = 1; w < BP_WAVES; ++w) s += accw[w * 3 * nbins + i];
    part[(int64_t)blockIdx.x * 3 * nbins + i] = s;
  }
}

// out[e] = sum over blocks of part[block][e] in a fixed order: a workgroup
// takes 64 entries (coalesced rows of the partials), wave s adds the blocks
// s, s + BIN_RED_SEG, ..., then the waves' sums are added in order.  (One
// wave per entry read 8 bytes of a line at a time: 0.039 -> 0.008 ms for the
// 8100 P_l sums at Ngrid 360.)  Box blockIdx.y of a batch: part
// [box][nblocks][nent], out [box][nent].
constexpr int BIN_RED_SEG = 8;
__global__ __launch_bounds__(64 * BIN_RED_SEG) void k_bin_reduce(const double* __restrict__ part,
                                                                 int nblocks, int nent,
                                                                 double* __restrict__ out) {
  __shared__ double seg_sum[BIN_RED_SEG][64];
  part += (int64_t)blockIdx.y * nblocks * nent;
  out += (int64_t)blockIdx.y * nent;
  const int lane = (int)threadIdx.x & 63, seg = (int)threadIdx.x >> 6;
  const int e = (int)blockIdx.x * 64 + lane;
  double s = 0.0;
  if (e < nent) {
#pragma unroll 8
    for (int b = seg; b < nblocks; b += BIN_RED_SEG) s += part[(int64_t)b * nent + e];
  }
  seg_sum[seg][lane] = s;
  __syncthreads();
  if (seg == 0 && e < nent) {
    double t = seg_sum[0][lane];
#pragma unroll
    for (int k = 1; k < BIN_RED_SEG; ++k) t += seg_sum[k][lane];
    out[e] = t;
  }
}

// Block partials of k_bin_power: one [3][nbins] record per block.
static int bin_power_blocks(int N) {
  const int64_t Nh = N / 2 + 1;
  return (int)std::min<int64_t>(cdiv(Nh * Nh, BP_WAVES), BP_MAX_BLOCKS);
}

static int launch_bin_reduce(psx_ctx* ctx, const void* part, int blocks, int nent, double* out,
                             int nbox) {
  hipLaunchKernelGGL(k_bin_reduce, dim3((unsigned)cdiv(nent, 64), nbox), dim3(64 * BIN_RED_SEG), 0,
                     ctx->stream, (const double*)part, blocks, nent, out);
  PSX_CHECK_LAUNCH();
  return PSX_OK;
}

// k_bin_power + k_bin_reduce with the block partials in `part` (at least
// bin_power_blocks(N) * 3 * nbins doubles; every entry is written before it
// is read, so nothing needs clearing).
// nbox half fields back to back give out3 [nbox][3][nbins].
static int bin_power_into(psx_ctx* ctx, const void* half, int N, int step, int nbins, double kf,
                          int prec, double* out3, void* part, int nbox = 1) {
  const size_t lds = (size_t)BP_WAVES * 3 * nbins * sizeof(double);
  const int blocks = bin_power_blocks(N);
  const int64_t mlast = shell_mmax(nbins, step);
  const int kstep = std::min(step, BP_MAX_STEP);
  if (prec == PSX_PREC_F64) {
    PSX_TRY(set_lds(k_bin_power<double>, lds));
    hipLaunchKernelGGL(k_bin_power<double>, dim3(blocks, nbox), dim3(BP_THREADS), lds, ctx->stream,
                       (const cplx<double>*)half, N, kstep, nbins, kf, mlast, (double*)part);
  } else {
    PSX_TRY(set_lds(k_bin_power<float>, lds));
    hipLaunchKernelGGL(k_bin_power<float>, dim3(blocks, nbox), dim3(BP_THREADS), lds, ctx->stream,
                       (const cplx<float>*)half, N, kstep, nbins, kf, mlast, (double*)part);
  }
  PSX_CHECK_LAUNCH();
  return launch_bin_reduce(ctx, part, blocks, 3 * nbins, out3, nbox);
}

int launch_bin_power(psx_ctx* ctx, const void* half, int N, int step, int nbins, double kf,
                     int prec, double* out3, int nbox) {
  PSX_REQUIRE(nbins >= 1 && nbins <= BP_MAX_BINS, "nbins must be in [1, 1024]");
  void* part = nullptr;
  PSX_TRY(ctx_buffer(ctx, "bin_partials",
                     (size_t)nbox * bin_power_blocks(N) * 3 * nbins * sizeof(double), &part));
  return bin_power_into(ctx, half, N, step, nbins, kf, prec, out3, part, nbox);
}

// ------------------------------------------- bin power without allocation ---
// The block partials of psx_bin_power_noalloc live in this device array
// (NOALLOC_DOUBLES doubles = 6 MiB: 512 blocks x 3 sums x 512 bins), which
// each device holds until the process ends.  Host code never passes the
// array's name to a kernel: its device address is looked up once per device
// with hipGetSymbolAddress and kept in noalloc_ptr[device].  Every call on a
// device shares that device's array, so calls that overlap on one device
// race; each call writes every partial it reads, so nothing needs clearing.
constexpr int NOALLOC_MAX_BINS = 512;
constexpr size_t NOALLOC_DOUBLES = (size_t)BP_MAX_BLOCKS * 3 * NOALLOC_MAX_BINS;
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];

constexpr int NOALLOC_MAX_DEVICES = 64;
static void* noalloc_ptr[NOALLOC_MAX_DEVICES];
static std::mutex noalloc_mu;

// The device address of `scratch` on the context's device (looked up on the
// first call with that device current).
static int noalloc_scratch(psx_ctx* ctx, void** out) {
  const int dev = ctx->device;
  PSX_REQUIRE(dev >= 0 && dev < NOALLOC_MAX_DEVICES, "device index beyond the scratch table");
  std::lock_guard<std::mutex> g(noalloc_mu);
  if (!noalloc_ptr[dev]) {
    int cur = 0;
    PSX_HIP(hipGetDevice(&cur));
    if (cur != dev) PSX_HIP(hipSetDevice(dev));
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != dev) (void)hipSetDevice(cur);
    if (e != hipSuccess || !p)
      return set_error(PSX_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    noalloc_ptr[dev] = p;
  }
  *out = noalloc_ptr[dev];
  return PSX_OK;
}

int launch_bin_power_noalloc(psx_ctx* ctx, const void* half, int N, int step, int nbins, double kf,
                             int prec, double* out3) {
  PSX_REQUIRE(nbins >= 1 && nbins <= NOALLOC_MAX_BINS,
              "psx_bin_power_noalloc: nbins must be in [1, 512] (fixed scratch of 6 MiB)");
  PSX_REQUIRE((size_t)bin_power_blocks(N) * 3 * nbins <= NOALLOC_DOUBLES,
              "psx_bin_power_noalloc: partials exceed the fixed scratch");
  void* part = nullptr;
  PSX_TRY(noalloc_scratch(ctx, &part));
  return bin_power_into(ctx, half, N, step, nbins, kf, prec, out3, part);
}

// p0k[j-1] = sum |delta|^2 / Nk[j] for j = max(j0,1)..nmax (NaN if Nk = 0),
// 0 elsewhere: the shell power of _Bk_periodic (pyspectrum.py:404) by Parseval.
// Box blockIdx.y of a batch: bins3 [box][3][nmax], p0k [box][nmax].
__global__ void k_p0k(const double* __restrict__ bins3, int nmax, int j0, double* __restrict__ p0k) {
  bins3 += (int64_t)blockIdx.y * 3 * nmax;
  p0k += (int64_t)blockIdx.y * nmax;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nmax) return;
  const int j = i + 1;
  p0k[i] = (j >= j0) ? bins3[nmax + i] / bins3[2 * nmax + i] : 0.0;
}

int launch_p0k(psx_ctx* ctx, const double* bins3, int nmax, int j0, double* p0k, int nbox) {
  hipLaunchKernelGGL(k_p0k, dim3((unsigned)cdiv(nmax, 64), nbox), dim3(64), 0, ctx->stream, bins3,
                     nmax, j0, p0k);
  PSX_CHECK_LAUNCH();
  return PSX_OK;
}

// --------------------------------------------------------- pk_pbox_rsd ----
// Restatement of the mode loop of estimator.f:196-244.  The Fortran visits
// the full grid, x > N/2 through the mirrored element; that mode is -k' of
// the half-field mode k' = (N - x, -y, -z), and in its float32 operations
// every sign flip is an exact negation, so it has the same rk, k bin, |mu|,
// mu bin, Legendre weights and |delta|^2.  The kernel therefore visits the
// half field once and counts 0 < x < N/2 twice (x = 0 and x = N/2 map to
// themselves): the same bins and counts, sums equal to round-off.  Except on
// the y or z Nyquist planes: there the mirror's component is +N/2 (index N/2
// maps to itself), not the negation, and the cos(pi/2) residue of the
// float32 line of sight makes its |mu| differ, so that mirror is replayed
// with the Fortran's own frequencies as a second pass over those rows.
// Every float32 operation that decides a bin is replayed in the reference's
// order without contraction (k bin: nint(Nbin*rk/(N/2)); mu bin:
// int((|mu| + dmu)/dmu) in float64 of float32 values).
//
// Row groups: for a line of sight along z, rsd_mode depends on ky and kz
// only through ky^2 and |kz| (its float32 line-of-sight cosines are exactly 0
// and 1, so mu = kz/k), and the Nyquist mirror has the same |mu|: the rows
// (+-y, +-z) share every bin.  Along x it depends on ky through ky^2 only:
// the rows +-y share them.  Along y no two rows do (the cos(pi/2) residue).
// A wave adds the |delta|^2 of such rows and bins them once; the binning
// (roots, divisions, scans, ordered LDS adds), not the reads, bounds the
// kernel.  Measured with the line of sight along z, Ngrid 360, 10 mu bins:
// 0.78 -> 0.147 ms (the modes inside the sphere are read in 0.02 ms).
//
// Deterministic: a wave takes 64 consecutive x of one row group.  The k bin
// depends only on |k|^2 = x^2 + c, so it never decreases along the lanes;
// a scan (fixed order) sums each run of equal keys and the run's last lane
// adds the run to the block's accumulators.  The (k, mu) key is scanned the
// same way; should a key come back after another key within the 64 lanes
// (two run ends with one key, found by a tag written and read back in LDS),
// those run ends are added one lane at a time in lane order.  A mode with a
// (k, mu) bin gives its k, p0 and nk only to that bin (k_rsd_k_sums adds them
// up for the k bin); modes outside the mu bins give them to the k bin.  The
// four waves of a block add their runs in turn, so the order of every
// addition is fixed; k_bin_reduce then adds the block partials in a fixed
// order.
struct RsdConst {
  float kf, mubin, cth, sth, cph, sph;
  int nbin, nmu;
  int64_t mlim;  // no |k|^2 above this has a k bin <= nbin
};

__device__ __forceinline__ int fort_freq(int n, int N) { return n <= N / 2 ? n : n - N; }

// The bins and weights of mode (kx, ky, kz): k bin (0-based, -1 if outside
// 1..nbin), (k, mu) bin (-1 if outside), k, |mu| and the Legendre factors.
// ALONG_Z: line of sight along z, where mu = kz/k exactly.
struct RsdMode {
  int kb, mb;
  double kk, mu, l2, l4;
};

template <bool ALONG_Z>
__device__ __forceinline__ RsdMode rsd_mode(int kx, int ky, int kz, const RsdConst& c, float fnb,
                                            float fh, double md) {
  RsdMode r;
  r.kb = -1;
  r.mb = -1;
  r.kk = r.mu = r.l2 = r.l4 = 0.0;
  float rk, mu32;
  int imk;
  {
#pragma clang fp contract(off)
    const float rkx = (float)kx, rky = (float)ky, rkz = (float)kz;
    rk = cr_sqrtf(rkx * rkx + rky * rky + rkz * rkz);
    imk = (int)roundf(cr_divf(fnb * rk, fh));  // NINT: half away from zero
    if (!(imk <= c.nbin && imk != 0)) return r;
    const float cot1 = cr_divf(rkz, rk);
    if constexpr (ALONG_Z) {
      mu32 = cot1;
    } else {
      const float sit1 = cr_sqrtf(1.0f - cot1 * cot1);
      float cc = 0.0f;
      if (sit1 > 0.0f) {
        const float den = rk * sit1;
        const float cp = cr_divf(rkx, den), sp = cr_divf(rky, den);
        cc = c.sph * sp + c.cph * cp;
      }
      mu32 = c.cth * cot1 + (c.sth * sit1) * cc;
    }
  }
  const double mu = (double)mu32;
  const int imu = (int)((fabs(mu) + md) / md);
  const double mu2 = mu * mu;
  r.l2 = -0.5 + 1.5 * mu2;
  r.l4 = 0.375 - 3.75 * mu2 + 4.375 * (mu2 * mu2);
  r.kk = (double)(c.kf * rk);
  r.mu = fabs(mu);
  r.kb = imk - 1;
  if (imu <= c.nmu && imu > 0) r.mb = r.kb * c.nmu + (imu - 1);
  return r;
}

// Adds each run end's NV sums to acc[e * stride + key]; run ends that share a
// key (a key that came back) are added one lane at a time in lane order.
// The lanes of a wave exchange data through LDS here (the tag written and
// read back, the one-lane-at-a-time adds), so those accesses are volatile:
// issued in program order, never merged or forwarded.
template <int NV>
__device__ __forceinline__ void run_add(bool end, int key, const double* v, double* acc,
                                        int stride, int* tag, int lane) {
  volatile int* vt = tag;
  if (end) vt[key] = lane;
  const bool clash = end && vt[key] != lane;
  if (__ballot(clash) == 0) {
    if (end) {
#pragma unroll
      for (int e = 0; e < NV; ++e) acc[e * stride + key] += v[e];
    }
  } else {
    volatile double* va = acc;
    for (int l = 0; l < 64; ++l) {
      if (lane == l && end) {
#pragma unroll
        for (int e = 0; e < NV; ++e) va[e * stride + key] = va[e * stride + key] + v[e];
      }
    }
  }
}

constexpr int RSD_THREADS = 256, RSD_WAVES = RSD_THREADS / 64, RSD_MAX_BLOCKS = 512;

// LOS 0, 1, 2: line of sight along x, y, z (the rows folded together).
template <typename T, int LOS>
__global__ __launch_bounds__(RSD_THREADS) void k_pk_rsd(const cplx<T>* __restrict__ Hh, int N,
                                                         RsdConst c, double* __restrict__ part) {
  constexpr bool FY = LOS != 1, FZ = LOS == 2;  // fold +-y, +-z
  extern __shared__ __align__(16) unsigned char smem_raw[];
  // layout: [5][nbin] (k, p0, p2, p4, nk) then [4][nbin*nmu] (km, mk, pkm, nkm)
  const int nb = c.nbin, nm = c.nmu, nbm = nb * nm;
  const int ntot = 5 * nb + 4 * nbm;
  double* acc = reinterpret_cast<double*>(smem_raw);
  int* tagk = reinterpret_cast<int*>(acc + ntot);
  int* tagm = tagk + nb;
  for (int i = threadIdx.x; i < ntot; i += RSD_THREADS) acc[i] = 0.0;
  const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
  const int Nh = N / 2 + 1, hN = N / 2;
  const int nyg = FY ? Nh : N, ngroups = nyg * (FZ ? Nh : N);
  const float fnb = (float)nb, fh = (float)hN;
  const double md = (double)c.mubin;
  const int mlim = (int)min(c.mlim, (int64_t)1 << 30);
  // work items of this wave: row groups grp, grp + gstride, ...; each has one
  // pass (two on the y/z Nyquist planes unless the line of sight is along z:
  // the original modes, then the replayed mirrors) of 64-lane chunks
  const int gstride = (int)gridDim.x * RSD_WAVES;
  int grp = (int)blockIdx.x * RSD_WAVES + wave, pass = 0, x0 = 0;
  auto nyquist = [&](int y, int z) { return !FZ && (y == hN || z == hN); };
  // advance to the next chunk that holds a mode below mlim
  auto settle = [&]() {
    while (grp < ngroups) {
      const int z = grp / nyg, y = grp - z * nyg;
      const int npass = nyquist(y, z) ? 2 : 1;
      const int ky = fort_freq(y, N), kz = fort_freq(z, N);
      if (pass < npass && x0 < Nh && ky * ky + kz * kz + x0 * x0 <= mlim) return;
      if (pass + 1 < npass && x0 > 0) { ++pass; x0 = 0; continue; }
      grp += gstride; pass = 0; x0 = 0;
    }
  };
  cplx<T> nxt[4];
  auto group_of = [&](int g) {
    const int z = g / nyg, y = g - z * nyg;
    return row_group(y, z, N, FY && y < hN, FZ && z < hN);
  };
  auto fetch = [&]() {
    load_group(Hh, group_of(grp), N, Nh, x0 + lane, grp < ngroups && x0 + lane < Nh, nxt);
  };
  settle();
  fetch();
  __syncthreads();
  for (;;) {
    const bool has = grp < ngroups;
    if (!__syncthreads_or(has)) break;
    RsdMode m;
    m.kb = -1; m.mb = -1;
    double vk[2] = {0.0, 0.0}, vm[3] = {0.0, 0.0, 0.0}, vo[3] = {0.0, 0.0, 0.0};
    double nmode = 0.0, nedge = 0.0;  // modes per lane, and what an edge lane lacks
    const int xb = x0;
    if (has) {
      const RowGroup g = group_of(grp);
      cplx<T> cur[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) cur[k] = nxt[k];
      const int x = x0 + lane;
      const int ky = fort_freq(g.y, N), kz = fort_freq(g.z, N);
      const bool nyq = nyquist(g.y, g.z);
      const int ps = pass;
      x0 += 64;
      settle();
      fetch();
      const double nr = (double)g.rows();
      // x = 0 and x = N/2 map to themselves; elsewhere the mirror is the
      // exact negation (weight 2) except on the Nyquist planes, where pass 1
      // replays it with the Fortran's frequencies
      nmode = nyq ? nr : 2.0 * nr;
      nedge = nyq ? 0.0 : nr;
      const bool xe = x == 0 || x == hN;
      if (x < Nh && (ps == 0 || !xe)) {
        m = ps == 0 ? rsd_mode<FZ>(x, ky, kz, c, fnb, fh, md)
                    : rsd_mode<FZ>(-x, fort_freq((N - g.y) % N, N), fort_freq((N - g.z) % N, N), c,
                                   fnb, fh, md);
        if (m.kb >= 0) {
          double pk = 0.0;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            if constexpr (sizeof(T) == 8) {
              pk += (double)cur[k].re * (double)cur[k].re + (double)cur[k].im * (double)cur[k].im;
            } else {  // the reference's float32 cabs(ct)**2
              const float a = hypotf(cur[k].re, cur[k].im);
              pk += (double)(a * a);
            }
          }
          const double wn = nmode - (xe ? nedge : 0.0);
          const double p = (xe || nyq ? 1.0 : 2.0) * pk;
          vk[0] = p * 5.0 * m.l2;
          vk[1] = p * 9.0 * m.l4;
          if (m.mb >= 0) { vm[0] = wn * m.kk; vm[1] = wn * m.mu; vm[2] = p; }
          else { vo[0] = wn * m.kk; vo[1] = p; vo[2] = wn; }
        }
      }
    }
    const LaneRun rk = lane_run(m.kb, lane), rm = lane_run(m.mb, lane);
    run_scan(vk, lane, rk.start);
    run_scan(vm, lane, rm.start);
    const bool over = __ballot(m.kb >= 0 && m.mb < 0) != 0;  // modes outside the mu bins
    if (over) run_scan(vo, lane, rk.start);
    const bool endk = m.kb >= 0 && rk.end, endm = m.mb >= 0 && rm.end;
    const double len = (double)(lane - rm.start + 1);
    const int edges = (xb + rm.start == 0 ? 1 : 0) + (xb + lane == hN ? 1 : 0);
    const double va[4] = {vm[0], vm[1], vm[2], nmode * len - nedge * (double)edges};
    for (int w = 0; w < RSD_WAVES; ++w) {
      if (w == wave && has) {
        if (endk) {  // the k bin never decreases along the lanes: one run end per key
          acc[2 * nb + m.kb] += vk[0];
          acc[3 * nb + m.kb] += vk[1];
          if (over) {
            acc[m.kb] += vo[0];
            acc[nb + m.kb] += vo[1];
            acc[4 * nb + m.kb] += vo[2];
          }
        }
        run_add<4>(endm, m.mb, va, acc + 5 * nb, nbm, tagm, lane);
      }
      __syncthreads();
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < ntot; i += RSD_THREADS) part[(int64_t)blockIdx.x * ntot + i] = acc[i];
}

// The k, p0 and nk of each k bin gain those of its (k, mu) bins: rows 0, 1, 4
// of [5][nb] and rows km, pkm, nkm of [4][nb][nm].
__global__ __launch_bounds__(64) void k_rsd_k_sums(double* __restrict__ out, int nb, int nm) {
  const int i = (int)blockIdx.x * 64 + (int)threadIdx.x;
  if (i >= 3 * nb) return;
  const int r = i / nb, kb = i - r * nb;
  const int dst = r == 0 ? 0 : r == 1 ? 1 : 4, src = r == 0 ? 0 : r == 1 ? 2 : 3;
  const double* m = out + 5 * nb + ((int64_t)src * nb + kb) * nm;
  double s = out[dst * nb + kb];
  for (int j = 0; j < nm; ++j) s += m[j];
  out[dst * nb + kb] = s;
}

template <typename T, int LOS>
static int pk_rsd_t(psx_ctx* ctx, const void* half, int N, const RsdConst& c, size_t lds,
                    double* gout) {
  const int Nh = N / 2 + 1;
  const int64_t ngroups = (int64_t)(LOS != 1 ? Nh : N) * (LOS == 2 ? Nh : N);
  const int ntot = 5 * c.nbin + 4 * c.nbin * c.nmu;
  const int blocks = (int)std::min<int64_t>(cdiv(ngroups, RSD_WAVES), RSD_MAX_BLOCKS);
  void* part = nullptr;
  PSX_TRY(ctx_buffer(ctx, "rsd_partials", (size_t)blocks * ntot * sizeof(double), &part));
  auto kern = k_pk_rsd<T, LOS>;
  PSX_TRY(set_lds(kern, lds));
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(RSD_THREADS), lds, ctx->stream, (const cplx<T>*)half,
                     N, c, (double*)part);
  PSX_CHECK_LAUNCH();
  PSX_TRY(launch_bin_reduce(ctx, part, blocks, ntot, gout, 1));
  hipLaunchKernelGGL(k_rsd_k_sums, dim3((unsigned)cdiv(3 * c.nbin, 64)), dim3(64), 0, ctx->stream,
                     gout, c.nbin, c.nmu);
  PSX_CHECK_LAUNCH();
  return PSX_OK;
}

int launch_pk_rsd(psx_ctx* ctx, const void* half, int N, int irsd, int lbox, int nbin, int nmu,
                  int prec, double* gout) {
  PSX_REQUIRE(irsd >= 0 && irsd <= 2, "rsd must be 0, 1 or 2");
  PSX_REQUIRE(nbin >= 1 && nmu >= 1 && lbox > 0, "bad Nbin/Nmu/Lbox");
  RsdConst c;
  const float pi = 3.141592654f;
  const float tpi = 2.0f * pi;
  c.kf = tpi / (float)lbox;
  c.mubin = 1.0f / (float)nmu;
  const float th = irsd == 2 ? 0.0f : 0.5f * pi;
  const float ph = irsd == 1 ? 0.5f * pi : 0.0f;
  // sin/cos of these float32 constants, correctly rounded
  c.cth = (float)cos((double)th); c.sth = (float)sin((double)th);
  c.cph = (float)cos((double)ph); c.sph = (float)sin((double)ph);
  c.nbin = nbin; c.nmu = nmu;
  // imk = nint(nbin*rk/(N/2)) <= nbin needs rk < (nbin + 1/2)(N/2)/nbin; the
  // bound below adds a margin far above float32 rounding
  const double rmax = (nbin + 0.5) * (N / 2) / (double)nbin * (1.0 + 1e-5) + 1e-3;
  c.mlim = (int64_t)std::ceil(rmax * rmax) + 1;
  const int64_t ntot = 5 * (int64_t)nbin + 4 * (int64_t)nbin * nmu;
  const size_t lds = (size_t)ntot * sizeof(double) + (size_t)(nbin + nbin * nmu) * sizeof(int);
  PSX_REQUIRE(lds <= 160 * 1024, "Nbin*Nmu too large for the binning kernel (LDS)");
  const bool f64 = prec == PSX_PREC_F64;
  switch (irsd) {
    case 0: return f64 ? pk_rsd_t<double, 0>(ctx, half, N, c, lds, gout) : pk_rsd_t<float, 0>(ctx, half, N, c, lds, gout);
    case 1: return f64 ? pk_rsd_t<double, 1>(ctx, half, N, c, lds, gout) : pk_rsd_t<float, 1>(ctx, half, N, c, lds, gout);
    default: return f64 ? pk_rsd_t<double, 2>(ctx, half, N, c, lds, gout) : pk_rsd_t<float, 2>(ctx, half, N, c, lds, gout);
  }
}

}  // namespace psx
