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
// The exact shortcuts of jmod and fold_period (tiles.hpp) skip fmod's loop
// and the division for nearly every corner.
__device__ __forceinline__ double jmod_d(double x, double L) {
  if (x >= 0.0 && x < L) return x;
  if (x < 0.0 && x > -L) return x + L;
  if (x >= L && x < 2.0 * L) return x - L;
  double m = fmod(x, L);
  if (m != 0.0 && m < 0.0) m = m + L;
  return m;
}

__device__ __forceinline__ double fold_period_d(double nd, double L) {
  const double a = fabs(nd);
  if (a <= 0.25 * L) return nd;
  if (a >= 0.75 * L && a <= 1.25 * L) return nd - copysign(L, nd);
  return nd - rint(nd / L) * L;
}

__device__ __forceinline__ void corner_rel_d(double p, double o, double L, int &idx, double &w) {
  const double q = floor(jmod_d(p + o, L));
  const double nd = fold_period_d(p - q, L);
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
// the tile table, scatter of 32-byte records), float64 sums of each chunk of
// a tile in a 17^3 LDS window (ds_add_f64), and a reduce that adds the
// windows covering each cell to the mesh.  One global float64 atomic per
// corner runs at some 23 G/s (lines shared by the 8 XCDs' L2s).  128^3
// displaced particles on 128^3 cells: 721 -> 87 us.
constexpr int kSort64Threads = 256, kSort64Per = 8;
constexpr uint32_t kSort64Slice = kSort64Threads * kSort64Per;
constexpr uint32_t kChunk64 = 8192;
constexpr int64_t kPaint64SortMin = 1 << 17;
constexpr uint32_t kMaxTiles64 = 16384;   // the LDS histogram is 64 KiB

struct Rec64 {
  double x, y, z;
  uint32_t p, pad;
};

__device__ __forceinline__ uint32_t tile_key_d(const AxisD &ax, const AxisD &ay, const AxisD &az, const TileGrid &t) {
  return (uint32_t(ax.i0 / kTile) * uint32_t(t.ty) + uint32_t(ay.i0 / kTile)) * uint32_t(t.tz) +
         uint32_t(az.i0 / kTile);
}

template <bool REL, bool SCATTER>
__global__ void __launch_bounds__(kSort64Threads)
sort_f64_kernel(const double *__restrict__ pos, uint32_t n, GridD g, TileGrid t, uint32_t *__restrict__ table,
                Rec64 *__restrict__ recs) {
  extern __shared__ uint32_t cur[];
  const uint32_t p0 = blockIdx.x * kSort64Slice;
  for (uint32_t k = threadIdx.x; k < t.K; k += kSort64Threads) cur[k] = 0;
  double x[kSort64Per], y[kSort64Per], z[kSort64Per];
  uint32_t key[kSort64Per];
#pragma unroll
  for (int i = 0; i < kSort64Per; ++i) {
    const uint32_t p = p0 + uint32_t(i) * kSort64Threads + threadIdx.x;
    const size_t at = 3 * size_t(p < n ? p : n - 1);
    x[i] = pos[at];
    y[i] = pos[at + 1];
    z[i] = pos[at + 2];
  }
#pragma unroll
  for (int i = 0; i < kSort64Per; ++i) {
    const uint32_t p = p0 + uint32_t(i) * kSort64Threads + threadIdx.x;
    AxisD ax, ay, az;
    axes_d<REL>(x[i], y[i], z[i], p < n ? p : n - 1, g, ax, ay, az);
    key[i] = p < n ? tile_key_d(ax, ay, az, t) : 0xffffffffu;
  }
  __syncthreads();
  const int lane = int(threadIdx.x & 63u);
#pragma unroll
  for (int i = 0; i < kSort64Per; ++i) {
    const bool active = key[i] != 0xffffffffu;
    const unsigned long long act = __ballot(active), heads = run_heads(key[i], active);
    if (active && ((heads >> lane) & 1ull)) atomicAdd(&cur[key[i]], run_length(heads, act));
  }
  __syncthreads();
  // table: the tile counts, or, for the scatter, the tiles' cursors
  for (uint32_t k = threadIdx.x; k < t.K; k += kSort64Threads)
    if (cur[k]) {
      const uint32_t at = atomicAdd(&table[k], cur[k]);
      if (SCATTER) cur[k] = at;
    }
  if (!SCATTER) return;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSort64Per; ++i) {
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
// paint_f64_kernel does, before the reduce adds the windows.
template <bool REL>
__global__ void __launch_bounds__(kWindowThreads)
accum_f64_kernel(const Rec64 *__restrict__ recs, const ChunkDesc *__restrict__ desc,
                 const uint32_t *__restrict__ nchunks, const double *__restrict__ weight, double wscalar, GridD g,
                 TileGrid t, double *__restrict__ partial, double *__restrict__ mesh) {
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
      int64_t idx[8];
      double w[8];
      corners_of_d<REL>(ax, ay, az, g, idx, w);
#pragma unroll
      for (int o = 0; o < 8; ++o) unsafeAtomicAdd(&mesh[idx[o]], wp * w[o]);
    }
  }
  __syncthreads();
  double *out = partial + size_t(blockIdx.x) * kWinCells;
  for (int i = int(threadIdx.x); i < kWinCells; i += kWindowThreads) out[i] = win[i];
}

// One workgroup per tile: each of its cells adds its tile's windows and, on a
// low face, the +1 halos of the lower neighbours.  1024 threads, four cells
// each, and the sources' chunk ranges in LDS: the loads wait on nothing but
// one another's issue (with 256 threads and the ranges read per cell, 40 us
// whatever the mesh).
__global__ void __launch_bounds__(1024)
reduce_f64_kernel(const double *__restrict__ partial, const uint32_t *__restrict__ choff,
                  const uint32_t *__restrict__ nchunk, TileGrid t, double *__restrict__ mesh) {
  int itx, ity, itz;
  tile_origin(blockIdx.x, t, itx, ity, itz);
  const int Lx = tile_len(itx, t.tx, t.nx), Ly = tile_len(ity, t.ty, t.ny), Lz = tile_len(itz, t.tz, t.nz);
  const int px = itx ? itx - 1 : t.tx - 1, py = ity ? ity - 1 : t.ty - 1, pz = itz ? itz - 1 : t.tz - 1;
  const int PLx = tile_len(px, t.tx, t.nx), PLy = tile_len(py, t.ty, t.ny), PLz = tile_len(pz, t.tz, t.nz);
  __shared__ uint32_t off[8], cnt[8];
  if (threadIdx.x < 8) {
    const int q = int(threadIdx.x);
    const uint32_t src = (uint32_t(q & 4 ? px : itx) * uint32_t(t.ty) + uint32_t(q & 2 ? py : ity)) * uint32_t(t.tz) +
                         uint32_t(q & 1 ? pz : itz);
    off[q] = choff[src];
    cnt[q] = nchunk[src];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kTile * kTile * kTile / 1024; ++i) {
    const int e = int(threadIdx.x) + i * 1024;
    const int a = e >> 8, b = (e >> 4) & 15, c = e & 15;
    if (a >= Lx || b >= Ly || c >= Lz) continue;
    double acc = 0.0;
    for (int q = 0; q < 8; ++q) {
      if (((q & 4) && a) || ((q & 2) && b) || ((q & 1) && c)) continue;
      const int li = ((q & 4 ? PLx : a) * kWin + (q & 2 ? PLy : b)) * kWin + (q & 1 ? PLz : c);
      const double *w = partial + size_t(off[q]) * kWinCells + li;
      for (uint32_t k = 0; k < cnt[q]; ++k) acc += w[size_t(k) * kWinCells];
    }
    mesh[(size_t(itx * kTile + a) * t.ny + size_t(ity * kTile + b)) * t.nz + size_t(itz * kTile + c)] += acc;
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
      int64_t idx[8];
      double w[8];
      corners_of_d<REL>(ax, ay, az, g, idx, w);
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int f = 0; f < 3; ++f) s[f] += phi3[f * M + idx[k]] * w[k];
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

// Workspace of the sorted paint (byte offsets); the sort, which a read may reuse,
// then the windows of the accumulation; total 0 where the atomic form
// is used instead: few particles, or more tiles than the LDS histogram
// holds.  48^3 random particles take 43 us by atomics and 42 us sorted, 64^3
// 94 and 47 us, 128^3 727 and 120 us; in the order of an undisturbed lattice,
// where neighbouring lanes share their cells' lines, 64^3 15 and 44 us, 128^3
// 110 and 75 us.
struct Paint64Ws {
  uint32_t maxchunks;
  size_t count, tstart, cursor, nchunk, choff, totals, desc, recs, sort, partial, total;
};

static Paint64Ws paint64_ws(int nx, int ny, int nz, int64_t n) {
  Paint64Ws w{};
  if (nx <= 0 || ny <= 0 || nz <= 0 || n < kPaint64SortMin || n > kMaxCells) return w;
  const TileGrid t = make_tiles(nx, ny, nz);
  if (uint64_t(t.tx) * t.ty * t.tz > kMaxTiles64) return w;
  w.maxchunks = uint32_t((n + kChunk64 - 1) / kChunk64 + t.K);
  size_t o = 0;
  auto take = [&o](size_t bytes) {
    const size_t at = o;
    o += align_up(bytes);
    return at;
  };
  w.count = take(size_t(t.K) * 4);
  w.tstart = take(size_t(t.K) * 4);
  w.cursor = take(size_t(t.K) * 4);
  w.nchunk = take(size_t(t.K) * 4);
  w.choff = take(size_t(t.K) * 4);
  w.totals = take(16);
  w.desc = take(size_t(w.maxchunks) * sizeof(ChunkDesc));
  w.recs = take(size_t(n) * sizeof(Rec64));
  w.sort = o;
  w.partial = take(size_t(w.maxchunks) * kWinCells * sizeof(double));
  w.total = o;
  return w;
}

size_t cic_paint_f64_ws(int nx, int ny, int nz, int64_t n) { return paint64_ws(nx, ny, nz, n).total; }

// base: w.sort bytes for the sort; partial: the windows.
static int paint_f64_sorted(hipStream_t s, int nx, int ny, int nz, const double *pos, uint32_t n, const double *weight,
                            double wscalar, bool rel, double *mesh, char *base, double *partial, const Paint64Ws &w) {
  const TileGrid t = make_tiles(nx, ny, nz);
  const GridD g = make_grid_d(nx, ny, nz);
  auto u32 = [base](size_t at) { return reinterpret_cast<uint32_t *>(base + at); };
  auto *desc = reinterpret_cast<ChunkDesc *>(base + w.desc);
  auto *recs = reinterpret_cast<Rec64 *>(base + w.recs);
  const unsigned grid = unsigned((uint64_t(n) + kSort64Slice - 1) / kSort64Slice);
  const size_t lds = size_t(t.K) * 4;
  int rc = zero_u32(s, u32(w.count), t.K);
  if (rc) return rc;
  hipLaunchKernelGGL(rel ? (sort_f64_kernel<true, false>) : (sort_f64_kernel<false, false>), dim3(grid),
                     dim3(kSort64Threads), lds, s, pos, n, g, t, u32(w.count), recs);
  JPM_LAUNCHED("sort_f64_kernel");
  rc = tile_table(s, u32(w.count), t.K, kChunk64, u32(w.tstart), u32(w.cursor), u32(w.nchunk), u32(w.choff),
                  u32(w.totals), desc);
  if (rc) return rc;
  hipLaunchKernelGGL(rel ? (sort_f64_kernel<true, true>) : (sort_f64_kernel<false, true>), dim3(grid),
                     dim3(kSort64Threads), lds, s, pos, n, g, t, u32(w.cursor), recs);
  JPM_LAUNCHED("sort_f64_kernel");
  hipLaunchKernelGGL(rel ? accum_f64_kernel<true> : accum_f64_kernel<false>, dim3(w.maxchunks), dim3(kWindowThreads), 0,
                     s, recs, desc, u32(w.totals) + 1, weight, wscalar, g, t, partial, mesh);
  JPM_LAUNCHED("accum_f64_kernel");
  hipLaunchKernelGGL(reduce_f64_kernel, dim3(t.K), dim3(1024), 0, s, partial, u32(w.choff), u32(w.nchunk), t, mesh);
  JPM_LAUNCHED("reduce_f64_kernel");
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
  if (flags & JPM_ZERO_MESH) {
    hipLaunchKernelGGL(zero_f64_kernel, dim3(grid_for(m, 256)), dim3(256), 0, s, mesh, m);
    JPM_LAUNCHED("zero_f64_kernel");
  }
  if (n == 0) return JPM_OK;
  JPM_REQUIRE(pos != nullptr, "positions are null");
  if (w.total)
    return paint_f64_sorted(s, nx, ny, nz, pos, uint32_t(n), weight, wscalar, rel, mesh, static_cast<char *>(ws),
                            reinterpret_cast<double *>(static_cast<char *>(ws) + w.partial), w);
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
// be painted sorted, that sort, which the read takes up again.  The paint's
// windows lie where the spectra follow.
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
  w.sort_bytes = paint64_ws(nx, ny, nz, int64_t(M)).sort;
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
    if (p.total && (p.sort > w.sort_bytes || p.total - p.sort > w.sort - w.spec)) p = Paint64Ws{};
    if (p.total) {
      JPM_REQUIRE(!rel || n == M, "relative painting needs one particle per lattice node (n=%lld, mesh %lld)",
                  (long long)n, (long long)M);
      hipLaunchKernelGGL(zero_f64_kernel, dim3(grid_for(M, 256)), dim3(256), 0, s, rho, M);
      JPM_LAUNCHED("zero_f64_kernel");
      rc = paint_f64_sorted(s, nx, ny, nz, pos, uint32_t(n), nullptr, 1.0, rel, rho, base + w.sort,
                            reinterpret_cast<double *>(spec), p);
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
