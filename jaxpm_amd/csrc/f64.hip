// Float64 CIC paint, CIC read and pm_forces: the reference's computations
// under jax_enable_x64 (its distributed-equivalence tests run in float64,
// tests/test_distributed_pm.py:30).  The corner maths is painting.py's and
// painting_utils.py's in double precision; deposits are summed in float64 (no
// fixed-point mode: a 64-bit fixed point would hold fewer significant bits
// than the double sums), in LDS windows over a tile sort or, for few
// particles, with one global atomic per corner; the transforms are hipFFT D2Z
// / Z2D with the k-space multipliers of kernels.py evaluated in double.
#include "tiles.hpp"

namespace jpm {

namespace {

struct AxisD {
  int i0, i1;       // wrapped indices of the low / high corner
  double w0, w1;    // weights 1 - |x - c| (0 for a dropped relative corner)
};

__device__ __forceinline__ int cell_int_d(double f) {
  return (f >= -2147483648.0 && f < 2147483648.0) ? int(f) : 0;
}

__device__ __forceinline__ int wrap_d(int c, int n) {
  if (uint32_t(c) < uint32_t(n)) return c;
  int r = c % n;
  return r < 0 ? r + n : r;
}

// painting.py:21-37 in double: floor, corner f + o, weight 1 - |x - c|,
// int32 cast then periodic mod.
__device__ __forceinline__ AxisD axis_abs_d(double x, int n) {
  AxisD a;
  const double f = floor(x), f1 = f + 1.0;
  a.w0 = 1.0 - fabs(x - f);
  a.w1 = 1.0 - fabs(x - f1);
  a.i0 = wrap_d(cell_int_d(f), n);
  a.i1 = wrap_d(cell_int_d(f1), n);
  return a;
}

// painting_utils.py:48-69 in double: q = (p + o) mod L (jnp.remainder),
// floor, nd = p - q, nd -= rint(nd / L) L, weight 1 - |nd|; the corner is
// dropped (zero weight at a valid index) unless 0 <= q < L.
__device__ __forceinline__ void corner_rel_d(double p, double o, double L, int &idx, double &w) {
  const double q = floor(jmod(p + o, L));
  const double nd = fold_period(p - q, L);
  const bool ok = (q >= 0.0) && (q < L);
  idx = ok ? int(q) : 0;
  w = ok ? 1.0 - fabs(nd) : 0.0;
}

struct GridD {
  int nx, ny, nz;
  FastDiv div_nz, div_ny;
};

// The corner axes of the particle at (x, y, z), p its index.
template <bool REL>
__device__ __forceinline__ void axes_d(double x, double y, double z, uint32_t p, const GridD &g, AxisD &ax, AxisD &ay,
                                       AxisD &az) {
  if (REL) {
    const uint32_t t = g.div_nz.div(p);
    const uint32_t k = p - t * uint32_t(g.nz);
    const uint32_t i = g.div_ny.div(t);
    const uint32_t j = t - i * uint32_t(g.ny);
    corner_rel_d(double(i) + x, 0.0, double(g.nx), ax.i0, ax.w0);
    corner_rel_d(double(i) + x, 1.0, double(g.nx), ax.i1, ax.w1);
    corner_rel_d(double(j) + y, 0.0, double(g.ny), ay.i0, ay.w0);
    corner_rel_d(double(j) + y, 1.0, double(g.ny), ay.i1, ay.w1);
    corner_rel_d(double(k) + z, 0.0, double(g.nz), az.i0, az.w0);
    corner_rel_d(double(k) + z, 1.0, double(g.nz), az.i1, az.w1);
  } else {
    ax = axis_abs_d(x, g.nx);
    ay = axis_abs_d(y, g.ny);
    az = axis_abs_d(z, g.nz);
  }
}

// The 8 corners (flat index, weight) of the axes: absolute corner order
// 000,100,010,001,110,101,011,111 (painting.py:24-25) or, relative, bit d of
// the corner number along axis d (painting_utils.py:43-45).  A dropped
// relative corner has weight 0 at index 0.
template <bool REL>
__device__ __forceinline__ void corners_of_d(const AxisD &ax, const AxisD &ay, const AxisD &az, const GridD &g,
                                             int64_t idx[8], double w[8]) {
  const int xs[8] = {0, 1, 0, 0, 1, 1, 0, 1};
  const int ys[8] = {0, 0, 1, 0, 1, 0, 1, 1};
  const int zs[8] = {0, 0, 0, 1, 0, 1, 1, 1};
#pragma unroll
  for (int o = 0; o < 8; ++o) {
    const int bx = REL ? (o & 1) : xs[o], by = REL ? ((o >> 1) & 1) : ys[o], bz = REL ? ((o >> 2) & 1) : zs[o];
    const int ix = bx ? ax.i1 : ax.i0, iy = by ? ay.i1 : ay.i0, iz = bz ? az.i1 : az.i0;
    w[o] = (bx ? ax.w1 : ax.w0) * (by ? ay.w1 : ay.w0) * (bz ? az.w1 : az.w0);
    idx[o] = (int64_t(ix) * g.ny + iy) * g.nz + iz;
  }
}

template <bool REL>
__device__ __forceinline__ void corners_d(const double *__restrict__ pos, uint32_t p, const GridD &g, int64_t idx[8],
                                          double w[8]) {
  AxisD ax, ay, az;
  axes_d<REL>(pos[3 * size_t(p)], pos[3 * size_t(p) + 1], pos[3 * size_t(p) + 2], p, g, ax, ay, az);
  corners_of_d<REL>(ax, ay, az, g, idx, w);
}

template <bool REL>
__global__ void __launch_bounds__(256)
paint_f64_kernel(const double *__restrict__ pos, const double *__restrict__ weight, double wscalar, uint32_t n,
                 GridD g, double *__restrict__ mesh) {
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    int64_t idx[8];
    double w[8];
    corners_d<REL>(pos, p, g, idx, w);
    const double wp = weight ? weight[p] : wscalar;
#pragma unroll
    for (int o = 0; o < 8; ++o) unsafeAtomicAdd(&mesh[idx[o]], wp * w[o]);
  }
}

// The paint of many particles: a counting sort into 16^3-cell tiles (count,
// scatter of 32-byte records) and float64 sums of each chunk of a tile in a
// 17^3 LDS window (ds_add_f64), added to the mesh by atomics, rows of
// neighbouring cells.  One global float64 atomic per corner instead runs at some
// 23 G/s (lines shared by the 8 XCDs' L2s).  128^3 displaced particles on 128^3
// cells: 743 us by atomics, 82 with the windows stored for a reduce, now 73; the
// small counts are bound by the launches: 64^3 95, 46 (seven launches), now 28
// (four).
constexpr int kSort64Threads = 256;
constexpr int64_t kPaint64SortMin = 1 << 17;
constexpr uint32_t kMaxTiles64 = 16384;   // the LDS histogram is 64 KiB
// More tiles take the tile table's launch: the scan costs every workgroup, and
// at 160^3 cells, 1000 tiles, 4 million particles in no order took 250 us with
// it and 207 without.
constexpr uint32_t kScanTiles64 = 512;

struct Rec64 {
  double x, y, z;
  uint32_t p, pad;
};

__device__ __forceinline__ uint32_t tile_key_d(const AxisD &ax, const AxisD &ay, const AxisD &az, const TileGrid &t) {
  return (uint32_t(ax.i0 / kTile) * uint32_t(t.ty) + uint32_t(ay.i0 / kTile)) * uint32_t(t.tz) +
         uint32_t(az.i0 / kTile);
}

// The eight deposits of a particle as atomics on the mesh.
template <bool REL>
__device__ __forceinline__ void deposit_d(const AxisD &ax, const AxisD &ay, const AxisD &az, const GridD &g, double wp,
                                          double *__restrict__ mesh) {
  int64_t idx[8];
  double w[8];
  corners_of_d<REL>(ax, ay, az, g, idx, w);
#pragma unroll
  for (int o = 0; o < 8; ++o) unsafeAtomicAdd(&mesh[idx[o]], wp * w[o]);
}

// The eight corner values of three meshes (M apart), weighted.
template <bool REL>
__device__ __forceinline__ void read3_d(const AxisD &ax, const AxisD &ay, const AxisD &az, const GridD &g,
                                        const double *__restrict__ phi3, int64_t M, double s[3]) {
  int64_t idx[8];
  double w[8];
  corners_of_d<REL>(ax, ay, az, g, idx, w);
#pragma unroll
  for (int k = 0; k < 8; ++k)
#pragma unroll
    for (int f = 0; f < 3; ++f) s[f] += phi3[f * M + idx[k]] * w[k];
}

// The tile table as its arrays: the tiles' counts, starts or cursors, chunks.
struct Table64 {
  uint32_t *count, *cursor, *totals;
  ChunkDesc *desc;
  uint32_t chunk;
};

// One pass over the particles, kPer of a thread.  kCount64 adds to the tiles'
// counts and clears mesh[0, zero).  The scatters write the records in tile
// order: kScatter64 from the cursors of a tile table, kScanScatter64 scans the
// counts itself, its cursors counting each tile's records from zero, and its
// first workgroup leaves the chunks and their number (a launch of their own
// otherwise: 64^3 4 us).
enum { kCount64, kScatter64, kScanScatter64 };

template <bool REL, int PASS, int kPer>
__global__ void __launch_bounds__(kSort64Threads)
sort_f64_kernel(const double *__restrict__ pos, uint32_t n, GridD g, TileGrid t, Table64 tab,
                Rec64 *__restrict__ recs, double *__restrict__ mesh, int64_t zero) {
  extern __shared__ uint32_t cur[];
  const uint32_t p0 = blockIdx.x * uint32_t(kSort64Threads * kPer);
  for (uint32_t k = threadIdx.x; k < t.K; k += kSort64Threads) cur[k] = 0;
  double x[kPer], y[kPer], z[kPer];
  uint32_t key[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const uint32_t p = p0 + uint32_t(i) * kSort64Threads + threadIdx.x;
    const size_t at = 3 * size_t(p < n ? p : n - 1);
    x[i] = pos[at];
    y[i] = pos[at + 1];
    z[i] = pos[at + 2];
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const uint32_t p = p0 + uint32_t(i) * kSort64Threads + threadIdx.x;
    AxisD ax, ay, az;
    axes_d<REL>(x[i], y[i], z[i], p < n ? p : n - 1, g, ax, ay, az);
    key[i] = p < n ? tile_key_d(ax, ay, az, t) : 0xffffffffu;
  }
  __syncthreads();
  const int lane = int(threadIdx.x & 63u);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const bool active = key[i] != 0xffffffffu;
    const unsigned long long act = __ballot(active), heads = run_heads(key[i], active);
    if (active && ((heads >> lane) & 1ull)) atomicAdd(&cur[key[i]], run_length(heads, act));
  }
  __syncthreads();
  if constexpr (PASS == kCount64) {
    for (int64_t i = blockIdx.x * int64_t(kSort64Threads) + threadIdx.x; i < zero;
         i += int64_t(gridDim.x) * kSort64Threads)
      mesh[i] = 0.0;
    for (uint32_t k = threadIdx.x; k < t.K; k += kSort64Threads)
      if (cur[k]) atomicAdd(&tab.count[k], cur[k]);
    return;
  }
  if constexpr (PASS == kScatter64) {
    for (uint32_t k = threadIdx.x; k < t.K; k += kSort64Threads)
      if (cur[k]) cur[k] = atomicAdd(&tab.cursor[k], cur[k]);
  } else {
    // particles and chunks of the tiles before this thread's, neighbours each
    constexpr int kOwn = kScanTiles64 / kSort64Threads;
    __shared__ uint32_t first[kScanTiles64], wave_p[kSort64Threads / 64], wave_c[kSort64Threads / 64];
    const uint32_t k0 = threadIdx.x * kOwn;
    uint32_t c[kOwn], np = 0, nc = 0;
#pragma unroll
    for (int i = 0; i < kOwn; ++i) c[i] = k0 + i < t.K ? tab.count[k0 + i] : 0u;
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      np += c[i];
      nc += (c[i] + tab.chunk - 1) / tab.chunk;
    }
    uint32_t xp = np, xc = nc;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t up = __shfl_up(xp, off), uc = __shfl_up(xc, off);
      if (lane >= off) {
        xp += up;
        xc += uc;
      }
    }
    if (lane == 63) {
      wave_p[threadIdx.x >> 6] = xp;
      wave_c[threadIdx.x >> 6] = xc;
    }
    __syncthreads();
    for (uint32_t w = 0; w < threadIdx.x >> 6; ++w) {
      xp += wave_p[w];
      xc += wave_c[w];
    }
    if (blockIdx.x == 0 && threadIdx.x == kSort64Threads - 1) tab.totals[1] = xc;
    uint32_t at = xp - np, ch = xc - nc;
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      first[k0 + i] = at;
      if (blockIdx.x == 0)
        for (uint32_t o = 0; o < c[i]; o += tab.chunk, ++ch)
          tab.desc[ch] = ChunkDesc{k0 + i, at + o, min(tab.chunk, c[i] - o), 0u};
      at += c[i];
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < t.K; k += kSort64Threads)
      if (cur[k]) cur[k] = first[k] + atomicAdd(&tab.cursor[k], cur[k]);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const uint32_t p = p0 + uint32_t(i) * kSort64Threads + threadIdx.x;
    const bool active = key[i] != 0xffffffffu;
    const unsigned long long act = __ballot(active), heads = run_heads(key[i], active);
    uint32_t base = 0;
    if (active && ((heads >> lane) & 1ull)) base = atomicAdd(&cur[key[i]], run_length(heads, act));
    const unsigned long long below = heads & ((2ull << lane) - 1ull);
    const int my_head = below ? 63 - __clzll((long long)below) : 0;
    base = __shfl(base, my_head);
    if (active) recs[base + uint32_t(lane - my_head)] = Rec64{x[i], y[i], z[i], p, 0u};
  }
}

// The corners are the (periodic) 2^3 block at the low corner.
__device__ __forceinline__ bool block_corners(const AxisD &ax, const AxisD &ay, const AxisD &az, const GridD &g) {
  return ax.i1 == (ax.i0 + 1 == g.nx ? 0 : ax.i0 + 1) && ay.i1 == (ay.i0 + 1 == g.ny ? 0 : ay.i0 + 1) &&
         az.i1 == (az.i0 + 1 == g.nz ? 0 : az.i0 + 1);
}

// A particle whose corners are the 2^3 block at its low corner deposits in
// the window; any other (a dropped or doubly rounded relative corner, a
// non-finite position) adds its eight deposits to the mesh itself, as
// paint_f64_kernel does.  The window is then added to the mesh but for its
// zeros, among them the cells past a short tile's halo.
template <bool REL>
__global__ void __launch_bounds__(kWindowThreads)
accum_f64_kernel(const Rec64 *__restrict__ recs, const ChunkDesc *__restrict__ desc,
                 const uint32_t *__restrict__ nchunks, const double *__restrict__ weight, double wscalar, GridD g,
                 TileGrid t, double *__restrict__ mesh) {
  __shared__ double win[kWinCells];
  if (blockIdx.x >= *nchunks) return;
  const ChunkDesc d = desc[blockIdx.x];
  int itx, ity, itz;
  tile_origin(d.tile, t, itx, ity, itz);
  const int ox = itx * kTile, oy = ity * kTile, oz = itz * kTile;
  for (int i = int(threadIdx.x); i < kWinCells; i += kWindowThreads) win[i] = 0.0;
  __syncthreads();
  for (uint32_t q = threadIdx.x; q < d.count; q += kWindowThreads) {
    const Rec64 r = recs[d.start + q];
    const double wp = weight ? weight[r.p] : wscalar;
    AxisD ax, ay, az;
    axes_d<REL>(r.x, r.y, r.z, r.p, g, ax, ay, az);
    if (block_corners(ax, ay, az, g)) {
      double *w0 = win + ((ax.i0 - ox) * kWin + (ay.i0 - oy)) * kWin + (az.i0 - oz);
#pragma unroll
      for (int o = 0; o < 8; ++o) {
        const int bx = o & 1, by = (o >> 1) & 1, bz = (o >> 2) & 1;
        const double w = (bx ? ax.w1 : ax.w0) * (by ? ay.w1 : ay.w0) * (bz ? az.w1 : az.w0);
        unsafeAtomicAdd(w0 + (bx * kWin + by) * kWin + bz, wp * w);
      }
    } else {
      deposit_d<REL>(ax, ay, az, g, wp, mesh);
    }
  }
  __syncthreads();
  for (int i = int(threadIdx.x); i < kWinCells; i += kWindowThreads) {
    const double v = win[i];
    if (v == 0.0) continue;
    const int c = i % kWin, ab = i / kWin, b = ab % kWin, a = ab / kWin;
    const int x = ox + a < t.nx ? ox + a : 0, y = oy + b < t.ny ? oy + b : 0, z = oz + c < t.nz ? oz + c : 0;
    unsafeAtomicAdd(&mesh[(size_t(x) * t.ny + y) * t.nz + z], v);
  }
}

template <bool REL, int NC, bool PAIR>
__global__ void __launch_bounds__(256)
read_f64_kernel(const double *__restrict__ mesh, int64_t cstride, const double *__restrict__ pos, uint32_t n, GridD g,
                double *__restrict__ out, uint32_t per) {
  const uint32_t p = ((blockIdx.x & 7u) * per + (blockIdx.x >> 3)) * blockDim.x + threadIdx.x;
  if (p >= n) return;
  AxisD ax, ay, az;
  axes_d<REL>(pos[3 * size_t(p)], pos[3 * size_t(p) + 1], pos[3 * size_t(p) + 2], p, g, ax, ay, az);
  const uint32_t ix[2] = {uint32_t(ax.i0), uint32_t(ax.i1)}, iy[2] = {uint32_t(ay.i0), uint32_t(ay.i1)},
                 iz[2] = {uint32_t(az.i0), uint32_t(az.i1)};
  // the corner order of corners_of_d
  const int abs_order[8] = {0, 1, 2, 4, 3, 5, 6, 7};
  double v[NC][8];
  load_corners<PAIR, NC>(mesh, size_t(cstride), ix, iy, iz, uint32_t(g.ny), uint32_t(g.nz), v);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int o = REL ? q : abs_order[q];
      s += v[c][o] * (((o & 1) ? ax.w1 : ax.w0) * ((o & 2) ? ay.w1 : ay.w0) * ((o & 4) ? az.w1 : az.w0));
    }
    out[size_t(p) * NC + c] = s;
  }
}

// read_f64_kernel<REL, 3> over a tile sort: each workgroup holds the three
// meshes' 17^3 windows of its tile in LDS (115 KiB, one workgroup of 16 waves
// a CU), so the particles of displaced lattices, whose lanes touch a cache line
// each, read LDS instead.  A particle whose corners are no 2^3 block reads the
// meshes.  The same sums in the same order.  128^3 particles displaced by 3
// cells rms: 46 us, the direct read 122 (173 with single loads).
template <bool REL>
__global__ void __launch_bounds__(1024)
read3_sorted_f64_kernel(const Rec64 *__restrict__ recs, const ChunkDesc *__restrict__ desc,
                        const uint32_t *__restrict__ nchunks, const double *__restrict__ phi3, int64_t M, GridD g,
                        TileGrid t, double *__restrict__ out) {
  extern __shared__ double rwin[];
  if (blockIdx.x >= *nchunks) return;
  const ChunkDesc d = desc[blockIdx.x];
  int itx, ity, itz;
  tile_origin(d.tile, t, itx, ity, itz);
  const int ox = itx * kTile, oy = ity * kTile, oz = itz * kTile;
  constexpr int kPer = (kWinCells + 1023) / 1024;
  double v[3][kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int e0 = int(threadIdx.x) + i * 1024, e = e0 < kWinCells ? e0 : kWinCells - 1;
    const int c = e % kWin, ab = e / kWin, b = ab % kWin, a = ab / kWin;
    const size_t cell = (size_t((ox + a) % t.nx) * t.ny + size_t((oy + b) % t.ny)) * t.nz + size_t((oz + c) % t.nz);
#pragma unroll
    for (int f = 0; f < 3; ++f) v[f][i] = phi3[f * M + cell];
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int e = int(threadIdx.x) + i * 1024;
#pragma unroll
    for (int f = 0; f < 3; ++f)
      if (e < kWinCells) rwin[f * kWinCells + e] = v[f][i];
  }
  __syncthreads();
  const int abs_order[8] = {0, 1, 2, 4, 3, 5, 6, 7};
  for (uint32_t q = threadIdx.x; q < d.count; q += 1024) {
    const Rec64 r = recs[d.start + q];
    AxisD ax, ay, az;
    axes_d<REL>(r.x, r.y, r.z, r.p, g, ax, ay, az);
    double s[3] = {0.0, 0.0, 0.0};
    if (block_corners(ax, ay, az, g)) {
      const double *w0 = rwin + ((ax.i0 - ox) * kWin + (ay.i0 - oy)) * kWin + (az.i0 - oz);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int o = REL ? k : abs_order[k];
        const double w = ((o & 1) ? ax.w1 : ax.w0) * ((o & 2) ? ay.w1 : ay.w0) * ((o & 4) ? az.w1 : az.w0);
        const int off = ((o & 1) * kWin + ((o >> 1) & 1)) * kWin + (o >> 2);
#pragma unroll
        for (int f = 0; f < 3; ++f) s[f] += w0[f * kWinCells + off] * w;
      }
    } else {
      read3_d<REL>(ax, ay, az, g, phi3, M, s);
    }
    double *o3 = out + 3 * size_t(r.p);
    o3[0] = s[0];
    o3[1] = s[1];
    o3[2] = s[2];
  }
}

__global__ void __launch_bounds__(256) zero_f64_kernel(double *__restrict__ p, int64_t m) {
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < m; i += int64_t(gridDim.x) * blockDim.x)
    p[i] = 0.0;
}

// k = 2 pi fftfreq(n)[i] (kernels.py:10-23) in double.
__device__ __forceinline__ double wavenumber(int i, int n) {
  const int f = i <= (n - 1) / 2 ? i : i - n;
  return 2.0 * M_PI * double(f) / double(n);
}

// sinc(t) = sin(pi t) / (pi t), 1 at 0 (jnp.sinc).
__device__ __forceinline__ double sinc_d(double t) {
  if (t == 0.0) return 1.0;
  const double a = M_PI * t;
  return sin(a) / a;
}

// The three force spectra of pm.py:49-56 from the half spectrum of the
// density: F_d = -g_d(k) * invlaplace(k) * longrange(k) * delta(k), with
// g_d the 4-point gradient i (8 sin w - sin 2w) / 6 (order 1) or i k with
// the len//2 entry zeroed (order 0, JPM_K_GRAD_EXACT), invlaplace -1/kk (0 at
// k = 0, times scale; with JPM_K_LAPL_FD, kk from k sinc(k / 2 pi)), longrange
// exp(-kk r^2) (kernels.py:41-115), and with JPM_K_DECONV the CIC
// compensation prod sinc(k / 2 pi)^-2 (kernels.py:118-136).
__global__ void __launch_bounds__(256)
force_f64_kernel(const double2 *__restrict__ dk, int nx, int ny, int nz, double r2, uint32_t kflags, double scale,
                 double2 *__restrict__ out3) {
  const int nzh = nz / 2 + 1;
  const int64_t H = int64_t(nx) * ny * nzh;
  for (int64_t e = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; e < H; e += int64_t(gridDim.x) * blockDim.x) {
    const int kz = int(e % nzh);
    const int64_t r = e / nzh;
    const int ky = int(r % ny), kx = int(r / ny);
    const double k[3] = {wavenumber(kx, nx), wavenumber(ky, ny), wavenumber(kz, nz)};
    const int idx[3] = {kx, ky, kz}, len[3] = {nx, ny, nz};
    double kk = 0.0, kk_plain = 0.0;
    for (int d = 0; d < 3; ++d) {
      kk_plain += k[d] * k[d];
      const double kd = (kflags & JPM_K_LAPL_FD) ? k[d] * sinc_d(k[d] / (2.0 * M_PI)) : k[d];
      kk += kd * kd;
    }
    double pot = kk == 0.0 ? 0.0 : -1.0 / kk;
    if (r2 != 0.0) pot *= exp(-kk_plain * r2);
    if (kflags & JPM_K_DECONV) {
      const double s = sinc_d(k[0] / (2.0 * M_PI)) * sinc_d(k[1] / (2.0 * M_PI)) * sinc_d(k[2] / (2.0 * M_PI));
      pot /= s * s;
    }
    pot *= scale;
    const double2 v = dk[e];
    for (int d = 0; d < 3; ++d) {
      double g;   // gradient_kernel is i * g
      if (kflags & JPM_K_GRAD_EXACT)
        g = (idx[d] == len[d] / 2) ? 0.0 : k[d];
      else
        g = (8.0 * sin(k[d]) - sin(2.0 * k[d])) / 6.0;
      // -(i g) * pot * v
      const double a = -g * pot;
      out3[d * H + e] = make_double2(-a * v.y, a * v.x);
    }
  }
}

GridD make_grid_d(int nx, int ny, int nz) {
  GridD g;
  g.nx = nx;
  g.ny = ny;
  g.nz = nz;
  g.div_nz = FastDiv(uint32_t(nz));
  g.div_ny = FastDiv(uint32_t(ny));
  return g;
}

}  // namespace

int fft_d2z(hipStream_t s, int nx, int ny, int nz, int batch, const double *in, void *out);
int fft_z2d(hipStream_t s, int nx, int ny, int nz, int batch, void *in, double *out);

// Workspace of the sorted paint (byte offsets): the sort, which a read may
// reuse.  total 0 where the atomic form is used instead: few particles, few per
// cell, or more tiles than the LDS histogram holds.
// Paint in us by atomics and sorted, for particles in the order of an
// undisturbed lattice (whose neighbouring lanes share their cells' lines), of a
// smooth displacement of 0.3 and of 3 cells, and in none:
//   51^3, one per cell   11  23  54  53     21  21  23  25
//   64^3                 16  38 100  94     26  27  28  34
//   80^3                 29  69 179 181     34  36  39  46
//   100^3                55 116 297 347     44  47  52  71
//   128^3               114 214 595 725     66  68  73 106
// and in lattice order and in none:
//   256^3, 1/64 a cell  109 111    55  96
//   256^3, 1/128         66  67    49  76
//   400^3, 1/64         430 472   256 380
// (An undisturbed lattice of fewer than some 90^3 particles would be better off
// with atomics, but the least displacement turns that over.)
struct Paint64Ws {
  uint32_t maxchunks, chunk;
  size_t count, tstart, cursor, nchunk, choff, totals, desc, recs, total;
};

static Paint64Ws paint64_ws(int nx, int ny, int nz, int64_t n) {
  Paint64Ws w{};
  if (nx <= 0 || ny <= 0 || nz <= 0 || n < kPaint64SortMin || n > kMaxCells) return w;
  if (n < cells(nx, ny, nz) / 64) return w;
  const TileGrid t = make_tiles(nx, ny, nz);
  if (uint64_t(t.tx) * t.ty * t.tz > kMaxTiles64) return w;
  for (w.chunk = 1024; w.chunk < 8192 && int64_t(w.chunk) * 128 < n;) w.chunk *= 2;
  w.maxchunks = uint32_t((n + w.chunk - 1) / w.chunk + t.K);
  size_t o = 0;
  auto take = [&o](size_t bytes) {
    const size_t at = o;
    o += align_up(bytes);
    return at;
  };
  w.count = take(2 * size_t(t.K) * 4);
  w.cursor = w.count + size_t(t.K) * 4;   // cleared with the counts
  w.tstart = take(size_t(t.K) * 4);
  w.nchunk = take(size_t(t.K) * 4);
  w.choff = take(size_t(t.K) * 4);
  w.totals = take(16);
  w.desc = take(size_t(w.maxchunks) * sizeof(ChunkDesc));
  w.recs = take(size_t(n) * sizeof(Rec64));
  w.total = o;
  return w;
}

size_t cic_paint_f64_ws(int nx, int ny, int nz, int64_t n) { return paint64_ws(nx, ny, nz, n).total; }

template <int PASS>
static int sort_pass(hipStream_t s, const double *pos, uint32_t n, bool rel, const GridD &g, const TileGrid &t,
                     const Table64 &tab, Rec64 *recs, double *mesh, int64_t zero) {
  // Few particles in slices of 1024, so that every CU has one; slices of 2048
  // add less often to the tiles' counters, of which particles in no order meet
  // all (paint in us, slices of 1024 and 2048, lattice and no order: 64^3 25.8
  // and 27.0, 33.6 and 32.4, 80^3 33.6 and 35.0, 54.6 and 46.3)
  const int per = n < (1u << 19) && t.K <= kScanTiles64 ? 4 : 8;
  auto kern = per == 4 ? (rel ? sort_f64_kernel<true, PASS, 4> : sort_f64_kernel<false, PASS, 4>)
                       : (rel ? sort_f64_kernel<true, PASS, 8> : sort_f64_kernel<false, PASS, 8>);
  const uint32_t slice = uint32_t(kSort64Threads * per);
  hipLaunchKernelGGL(kern, dim3((n + slice - 1) / slice), dim3(kSort64Threads), size_t(t.K) * 4, s, pos, n, g, t, tab,
                     recs, mesh, zero);
  JPM_LAUNCHED("sort_f64_kernel");
  return JPM_OK;
}

// mesh (cleared first if `zero`) += the paint.
static int paint_f64_sorted(hipStream_t s, int nx, int ny, int nz, const double *pos, uint32_t n, const double *weight,
                            double wscalar, bool rel, double *mesh, bool zero, char *base, const Paint64Ws &w) {
  const TileGrid t = make_tiles(nx, ny, nz);
  const GridD g = make_grid_d(nx, ny, nz);
  auto u32 = [base](size_t at) { return reinterpret_cast<uint32_t *>(base + at); };
  auto *recs = reinterpret_cast<Rec64 *>(base + w.recs);
  const Table64 tab{u32(w.count), u32(w.cursor), u32(w.totals), reinterpret_cast<ChunkDesc *>(base + w.desc), w.chunk};
  const int64_t m = zero ? cells(nx, ny, nz) : 0;
  int rc = zero_u32(s, tab.count, 2 * t.K);
  if (!rc) rc = sort_pass<kCount64>(s, pos, n, rel, g, t, tab, recs, mesh, m);
  if (rc) return rc;
  if (t.K <= kScanTiles64) {
    rc = sort_pass<kScanScatter64>(s, pos, n, rel, g, t, tab, recs, nullptr, 0);
  } else {
    rc = tile_table(s, tab.count, t.K, w.chunk, u32(w.tstart), tab.cursor, u32(w.nchunk), u32(w.choff), tab.totals,
                    tab.desc);
    if (!rc) rc = sort_pass<kScatter64>(s, pos, n, rel, g, t, tab, recs, nullptr, 0);
  }
  if (rc) return rc;
  hipLaunchKernelGGL(rel ? accum_f64_kernel<true> : accum_f64_kernel<false>, dim3(w.maxchunks), dim3(kWindowThreads), 0,
                     s, recs, tab.desc, tab.totals + 1, weight, wscalar, g, t, mesh);
  JPM_LAUNCHED("accum_f64_kernel");
  return JPM_OK;
}

// The three-component read at the particles of a sort that paint_f64_sorted
// left in base.
static int read3_f64_sorted(hipStream_t s, int nx, int ny, int nz, const double *phi3, bool rel, double *out,
                            const char *base, const Paint64Ws &w) {
  const TileGrid t = make_tiles(nx, ny, nz);
  auto kern = rel ? read3_sorted_f64_kernel<true> : read3_sorted_f64_kernel<false>;
  JPM_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                              int(3 * kWinCells * sizeof(double))));
  hipLaunchKernelGGL(kern, dim3(w.maxchunks), dim3(1024), 3 * kWinCells * sizeof(double), s,
                     reinterpret_cast<const Rec64 *>(base + w.recs), reinterpret_cast<const ChunkDesc *>(base + w.desc),
                     reinterpret_cast<const uint32_t *>(base + w.totals) + 1, phi3, cells(nx, ny, nz),
                     make_grid_d(nx, ny, nz), t, out);
  JPM_LAUNCHED("read3_sorted_f64_kernel");
  return JPM_OK;
}

// ws: cic_paint_f64_ws bytes, or null for the form without one.
int cic_paint_f64(hipStream_t s, int nx, int ny, int nz, const double *pos, int64_t n, const double *weight,
                  double wscalar, double *mesh, uint32_t flags, void *ws, size_t ws_bytes) {
  int rc = check_dims(nx, ny, nz);
  if (rc) return rc;
  JPM_REQUIRE(n >= 0 && n <= kMaxCells, "particle count %lld out of range", (long long)n);
  JPM_REQUIRE(mesh != nullptr, "mesh is null");
  JPM_REQUIRE(!(flags & JPM_DETERMINISTIC),
              "the float64 paint sums in float64; JPM_DETERMINISTIC is a float32 mode");
  const bool rel = flags & JPM_RELATIVE;
  const int64_t m = cells(nx, ny, nz);
  JPM_REQUIRE(!rel || n == m, "relative painting needs one particle per lattice node (n=%lld, mesh %lld)",
              (long long)n, (long long)m);
  const Paint64Ws w = ws ? paint64_ws(nx, ny, nz, n) : Paint64Ws{};
  JPM_REQUIRE(ws_bytes >= w.total, "the float64 paint needs %zu workspace bytes, got %zu", w.total, ws_bytes);
  JPM_REQUIRE(n == 0 || pos != nullptr, "positions are null");
  if (w.total)
    return paint_f64_sorted(s, nx, ny, nz, pos, uint32_t(n), weight, wscalar, rel, mesh, flags & JPM_ZERO_MESH,
                            static_cast<char *>(ws), w);
  if (flags & JPM_ZERO_MESH) {
    hipLaunchKernelGGL(zero_f64_kernel, dim3(grid_for(m, 256)), dim3(256), 0, s, mesh, m);
    JPM_LAUNCHED("zero_f64_kernel");
  }
  if (n == 0) return JPM_OK;
  const GridD g = make_grid_d(nx, ny, nz);
  const unsigned grid = grid_for(n, 256, 256 * 128);
  if (rel)
    hipLaunchKernelGGL(paint_f64_kernel<true>, dim3(grid), dim3(256), 0, s, pos, weight, wscalar, uint32_t(n), g, mesh);
  else
    hipLaunchKernelGGL(paint_f64_kernel<false>, dim3(grid), dim3(256), 0, s, pos, weight, wscalar, uint32_t(n), g,
                       mesh);
  JPM_LAUNCHED("paint_f64_kernel");
  return JPM_OK;
}

int cic_read_f64(hipStream_t s, int nx, int ny, int nz, const double *mesh, int ncomp, int64_t comp_stride,
                 const double *pos, int64_t n, double *out, uint32_t flags) {
  int rc = check_dims(nx, ny, nz);
  if (rc) return rc;
  JPM_REQUIRE(ncomp >= 1 && ncomp <= 4, "ncomp=%d must be 1..4", ncomp);
  JPM_REQUIRE(n >= 0 && n <= kMaxCells, "particle count %lld out of range", (long long)n);
  const int64_t m = cells(nx, ny, nz);
  JPM_REQUIRE(ncomp == 1 || comp_stride >= m, "component stride %lld smaller than the mesh", (long long)comp_stride);
  const bool rel = flags & JPM_RELATIVE;
  JPM_REQUIRE(!rel || n == m, "relative reading needs one particle per lattice node (n=%lld, mesh %lld)",
              (long long)n, (long long)m);
  if (n == 0) return JPM_OK;
  JPM_REQUIRE(mesh && pos && out, "null pointer argument");
  const GridD g = make_grid_d(nx, ny, nz);
  uint32_t per;
  const unsigned grid = xcd_blocks(n, 256, per);
#define JPM_R64(C)                                                                                                  \
  case C: {                                                                                                         \
    auto kern = nz >= 2 ? (rel ? read_f64_kernel<true, C, true> : read_f64_kernel<false, C, true>)                  \
                        : (rel ? read_f64_kernel<true, C, false> : read_f64_kernel<false, C, false>);               \
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, s, mesh, comp_stride, pos, uint32_t(n), g, out, per);        \
    break;                                                                                                          \
  }
  switch (ncomp) {
    JPM_R64(1)
    JPM_R64(2)
    JPM_R64(3)
    JPM_R64(4)
  }
#undef JPM_R64
  JPM_LAUNCHED("read_f64_kernel");
  return JPM_OK;
}

// Workspace of pm_forces_f64: the density mesh, its half spectrum, the three
// force spectra, the three force meshes and, where one particle per cell would
// be painted sorted, that sort, which the read takes up again.
struct Forces64Ws {
  size_t spec, spec3, phi3, sort, sort_bytes, total;
};

static Forces64Ws forces64_ws(int nx, int ny, int nz) {
  const size_t M = size_t(cells(nx, ny, nz)), H = size_t(half_cells(nx, ny, nz));
  Forces64Ws w;
  w.spec = align_up(M * 8);
  w.spec3 = w.spec + align_up(H * 16);
  w.phi3 = w.spec3 + align_up(3 * H * 16);
  w.sort = w.phi3 + align_up(3 * M * 8);
  w.sort_bytes = cic_paint_f64_ws(nx, ny, nz, int64_t(M));
  w.total = w.sort + w.sort_bytes;
  return w;
}

size_t pm_forces_f64_workspace_size(int nx, int ny, int nz) {
  if (nx <= 0 || ny <= 0 || nz <= 0) return 0;
  return forces64_ws(nx, ny, nz).total;
}

int pm_forces_f64(hipStream_t s, int nx, int ny, int nz, const double *pos, int64_t n, const double *delta,
                  double r_split, uint32_t flags, uint32_t kflags, double *out3, void *ws, size_t ws_bytes) {
  int rc = check_dims(nx, ny, nz);
  if (rc) return rc;
  JPM_REQUIRE(n >= 0 && n <= kMaxCells, "particle count %lld out of range", (long long)n);
  JPM_REQUIRE(out3 != nullptr && (n == 0 || pos != nullptr), "null pointer argument");
  const Forces64Ws w = forces64_ws(nx, ny, nz);
  JPM_REQUIRE(ws && ws_bytes >= w.total, "pm_forces_f64 needs %zu workspace bytes, got %zu", w.total, ws_bytes);
  const int64_t M = cells(nx, ny, nz), H = half_cells(nx, ny, nz);
  const bool rel = flags & JPM_RELATIVE;
  char *base = static_cast<char *>(ws);
  double *rho = reinterpret_cast<double *>(base);
  double2 *spec = reinterpret_cast<double2 *>(base + w.spec);
  double2 *spec3 = reinterpret_cast<double2 *>(base + w.spec3);
  double *phi3 = reinterpret_cast<double *>(base + w.phi3);
  const double *field = delta;
  Paint64Ws p{};
  if (!field) {
    p = paint64_ws(nx, ny, nz, n);
    if (p.total > w.sort_bytes) p = Paint64Ws{};
    if (p.total) {
      JPM_REQUIRE(!rel || n == M, "relative painting needs one particle per lattice node (n=%lld, mesh %lld)",
                  (long long)n, (long long)M);
      rc = paint_f64_sorted(s, nx, ny, nz, pos, uint32_t(n), nullptr, 1.0, rel, rho, true, base + w.sort, p);
    } else {
      // too many particles per cell for the sort's share of the workspace:
      // the whole paint where the spectra follow, or atomics
      const bool fits = cic_paint_f64_ws(nx, ny, nz, n) <= w.sort - w.spec;
      rc = cic_paint_f64(s, nx, ny, nz, pos, n, nullptr, 1.0, rho, (flags & JPM_RELATIVE) | JPM_ZERO_MESH,
                         fits ? static_cast<void *>(spec) : nullptr, w.sort - w.spec);
    }
    if (rc) return rc;
    field = rho;
  }
  if ((rc = fft_d2z(s, nx, ny, nz, 1, field, spec))) return rc;
  hipLaunchKernelGGL(force_f64_kernel, dim3(grid_for(H, 256)), dim3(256), 0, s, spec, nx, ny, nz, r_split * r_split,
                     kflags, 1.0 / double(M), spec3);
  JPM_LAUNCHED("force_f64_kernel");
  if ((rc = fft_z2d(s, nx, ny, nz, 3, spec3, phi3))) return rc;
  if (p.total) return read3_f64_sorted(s, nx, ny, nz, phi3, rel, out3, base + w.sort, p);
  return cic_read_f64(s, nx, ny, nz, phi3, 3, M, pos, n, out3, flags & JPM_RELATIVE);
}

}  // namespace jpm
