// Two-dimensional painting for lens planes: the weighted 2-D CIC paint
// (painting.py:131-158), its adjoint, the density plane of a slab of the box
// (lensing.py:11-44) with its adjoint, and the Gaussian filter of
// utils.gaussian_smoothing (utils.py:208-222) applied between the library's
// 2-D transforms.
//
// A plane is small next to the particle arrays (1024^2 cells are 4 MB, 256^3
// particles 201 MB), so the 2-D paint streams the particles once and adds
// its four deposits with float atomics; so does the density plane of few
// particles.  Many particles go through a counting sort into 64 x 64-pixel
// tiles first and are summed in LDS windows (plane_select_kernel and below).
#include "tiles.hpp"

namespace jpm {

int fft_r2c(hipStream_t s, int nx, int ny, int nz, int batch, const float *in, void *out);
int fft_c2r(hipStream_t s, int nx, int ny, int nz, int batch, void *in, float *out);

// The four corners of a 2-D CIC deposit in the order of painting.py:141
// ((0,0), (1,0), (0,1), (1,1)): weights (1 - |x - cx|)(1 - |y - cy|)
// (painting.py:143-144), derivative factors -sign(x - cx) with sign(0) = +1
// (the derivative jax.grad takes of abs at 0), and cells int32(c) mod n
// (painting.py:148-150).
struct Cic2 {
  uint32_t idx[4];
  float w[4], dx[4], dy[4];
};

__device__ __forceinline__ void cic2(float x, float y, int nx, int ny, Cic2 &c) {
  const float fx = floorf(x), fy = floorf(y);
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    const float cx = fx + float(o & 1), cy = fy + float(o >> 1);
    const float ex = x - cx, ey = y - cy;
    const float kx = 1.0f - fabsf(ex), ky = 1.0f - fabsf(ey);
    c.w[o] = kx * ky;
    c.dx[o] = (ex >= 0.0f ? -1.0f : 1.0f) * ky;
    c.dy[o] = kx * (ey >= 0.0f ? -1.0f : 1.0f);
    c.idx[o] = uint32_t(wrapi(cell_int(cx), nx)) * uint32_t(ny) + uint32_t(wrapi(cell_int(cy), ny));
  }
}

// mesh[nx][ny] += the deposits of particles (pos[p * stride], pos[p * stride
// + 1]), each times weight[p] when weight is given.
__global__ void __launch_bounds__(256)
paint2d_kernel(const float *__restrict__ pos, uint32_t n, uint32_t stride, const float *__restrict__ weight, int nx,
               int ny, float *__restrict__ mesh) {
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    Cic2 c;
    cic2(pos[size_t(p) * stride], pos[size_t(p) * stride + 1], nx, ny, c);
    const float wp = weight ? weight[p] : 1.0f;
#pragma unroll
    for (int o = 0; o < 4; ++o) atomicAdd(&mesh[c.idx[o]], weight ? c.w[o] * wp : c.w[o]);
  }
}

// The adjoint of paint2d for a mesh cotangent g: gpos[p] (2 floats at
// stride gstride) = w_p sum_o g[idx_o] dW_o/dxy, gweight[p] = sum_o g[idx_o]
// W_o.  Either output may be NULL.
__global__ void __launch_bounds__(256)
paint2d_vjp_kernel(const float *__restrict__ pos, uint32_t n, uint32_t stride, const float *__restrict__ weight, int nx,
                   int ny, const float *__restrict__ g, float *__restrict__ gpos, uint32_t gstride,
                   float *__restrict__ gweight) {
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    Cic2 c;
    cic2(pos[size_t(p) * stride], pos[size_t(p) * stride + 1], nx, ny, c);
    float sx = 0.0f, sy = 0.0f, sw = 0.0f;
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      const float v = g[c.idx[o]];
      sx += v * c.dx[o];
      sy += v * c.dy[o];
      sw += v * c.w[o];
    }
    if (gpos) {
      const float wp = weight ? weight[p] : 1.0f;
      gpos[size_t(p) * gstride] = sx * wp;
      gpos[size_t(p) * gstride + 1] = sy * wp;
    }
    if (gweight) gweight[p] = sw;
  }
}

// The plane coordinates of lensing.py:26-29: jnp.mod(x, box_nx) /
// box_nx * res (both axes are wrapped and scaled by box_nx there).
__device__ __forceinline__ float plane_coord(float x, float bnx, float res) { return jmod(x, bnx) / bnx * res; }

// Density plane of the particles pos[n][3] with lo < z <= hi (the weight of
// lensing.py:32-33; the other particles' deposits are zeros and are
// skipped) into plane[res][res].
__global__ void __launch_bounds__(256)
density_plane_kernel(const float *__restrict__ pos, uint32_t n, float bnx, float lo, float hi, float res, int ires,
                     float *__restrict__ plane) {
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    const float d = pos[3 * size_t(p) + 2];
    if (!(d > lo && d <= hi)) continue;
    Cic2 c;
    cic2(plane_coord(pos[3 * size_t(p)], bnx, res), plane_coord(pos[3 * size_t(p) + 1], bnx, res), ires, ires, c);
#pragma unroll
    for (int o = 0; o < 4; ++o) atomicAdd(&plane[c.idx[o]], c.w[o]);
  }
}

// The density plane of many particles, without global atomics on pixels:
//   select   one pass over the particles: those of the slab become records
//            (their plane coordinates, 8 bytes), compacted, and are counted
//            per 64 x 64-pixel tile
//   (tile table: tile starts and chunk descriptors)
//   scatter  the records into tile order
//   accum    one workgroup per chunk of a tile's records: a 65 x 65 window of
//            float64 sums in LDS (ds_add_f64), stored as floats
//   reduce   each pixel sums its tile's windows and, on a low edge, the +1
//            halos of the lower neighbours, and divides by the normalisation
// One float atomic per corner runs at about 25 G/s whatever the order of the
// particles (lines shared by the 8 XCDs' L2s).  256^3 particles, a quarter in
// the slab, 1024^2 pixels, lattice order: 673 -> 134 us, of which the select
// pass over the positions 76.
constexpr int kPt = 64, kPw = kPt + 1, kPwCells = kPw * kPw;
constexpr uint32_t kPlaneSelect = 4096;     // particles per select workgroup, records per scatter workgroup
constexpr uint32_t kPlaneChunk = 8192;      // records per window
constexpr uint32_t kPlaneMaxTiles = 4096;   // 4096^2 pixels: the LDS histogram is 16 KiB
constexpr int64_t kPlaneSortMin = 3 << 18;
// Particles of one sort: more take it in turns, in the workspace of one (2.1 GB
// of records, which all of them may fill), their sums kept in float64.  A turn
// costs 46 us beyond its particles: 2^27 take 1067 us in one and 1113 in two.
constexpr int64_t kPlanePass = 1 << 27;

struct PlaneTiles {
  int res, t;   // pixels and tiles per axis
  FastDiv div_t;
};

__device__ __forceinline__ int plane_cell(float u, int res) { return wrapi(cell_int(floorf(u)), res); }

__device__ __forceinline__ uint32_t plane_tile(float2 r, const PlaneTiles &t) {
  return uint32_t(plane_cell(r.x, t.res) / kPt) * uint32_t(t.t) + uint32_t(plane_cell(r.y, t.res) / kPt);
}

__device__ __forceinline__ int plane_len(int i, const PlaneTiles &t) {
  return i == t.t - 1 ? t.res - i * kPt : kPt;
}

__global__ void __launch_bounds__(64) plane_clear_kernel(uint32_t *__restrict__ a, uint32_t n) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) a[i] = 0u;
}

// nsel[0] selected particles, count[t] of them in tile t (both start at 0).
__global__ void __launch_bounds__(256)
plane_select_kernel(const float *__restrict__ pos, uint32_t n, float bnx, float lo, float hi, PlaneTiles t,
                    uint32_t *__restrict__ nsel, uint32_t *__restrict__ count, float2 *__restrict__ recs) {
  __shared__ float2 stage[kPlaneSelect];
  __shared__ uint32_t cnt, base;
  extern __shared__ uint32_t hist[];
  const uint32_t T = uint32_t(t.t) * uint32_t(t.t);
  if (threadIdx.x == 0) cnt = 0;
  for (uint32_t k = threadIdx.x; k < T; k += 256) hist[k] = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const uint32_t p0 = blockIdx.x * kPlaneSelect;
  constexpr int kPer = 4;   // particles of a thread whose loads are in flight together
  for (uint32_t b = 0; b < kPlaneSelect; b += 256 * kPer) {
    float x[kPer], y[kPer], z[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const uint32_t p = p0 + b + uint32_t(i) * 256 + threadIdx.x;
      const size_t at = 3 * size_t(p < n ? p : n - 1);
      x[i] = pos[at];
      y[i] = pos[at + 1];
      z[i] = p < n ? pos[at + 2] : NAN;
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const bool in = z[i] > lo && z[i] <= hi;
      const unsigned long long act = __ballot(in);
      uint32_t at = 0;
      if (lane == 0 && act) at = atomicAdd(&cnt, uint32_t(__popcll(act)));
      at = __shfl(at, 0) + uint32_t(__popcll(act & ((1ull << lane) - 1ull)));
      if (in) stage[at] = make_float2(plane_coord(x[i], bnx, float(t.res)), plane_coord(y[i], bnx, float(t.res)));
    }
  }
  __syncthreads();
  const uint32_t m = cnt;
  if (threadIdx.x == 0 && m) base = atomicAdd(nsel, m);
  __syncthreads();
  for (uint32_t b = 0; b < m; b += 256) {
    const uint32_t q = b + threadIdx.x;
    const bool active = q < m;
    uint32_t key = 0xffffffffu;
    if (active) {
      const float2 r = stage[q];
      recs[base + q] = r;
      key = plane_tile(r, t);
    }
    const unsigned long long act = __ballot(active);
    const unsigned long long heads = run_heads(key, active);
    if (active && ((heads >> lane) & 1ull)) atomicAdd(&hist[key], run_length(heads, act));
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < T; k += 256)
    if (hist[k]) atomicAdd(&count[k], hist[k]);
}

__global__ void __launch_bounds__(512)
plane_scatter_kernel(const float2 *__restrict__ recs, const uint32_t *__restrict__ nsel, PlaneTiles t,
                     uint32_t *__restrict__ cursor, float2 *__restrict__ sorted) {
  extern __shared__ uint32_t cur[];
  const uint32_t n = *nsel, p0 = blockIdx.x * kPlaneSelect;
  if (p0 >= n) return;
  constexpr int kPer = int(kPlaneSelect) / 512;
  const uint32_t T = uint32_t(t.t) * uint32_t(t.t);
  const int lane = threadIdx.x & 63;
  for (uint32_t k = threadIdx.x; k < T; k += 512) cur[k] = 0;
  float2 r[kPer];
  uint32_t key[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const uint32_t p = p0 + uint32_t(i) * 512 + threadIdx.x;
    r[i] = recs[p < n ? p : n - 1];
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const uint32_t p = p0 + uint32_t(i) * 512 + threadIdx.x;
    key[i] = p < n ? plane_tile(r[i], t) : 0xffffffffu;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const bool active = key[i] != 0xffffffffu;
    const unsigned long long act = __ballot(active);
    const unsigned long long heads = run_heads(key[i], active);
    if (active && ((heads >> lane) & 1ull)) atomicAdd(&cur[key[i]], run_length(heads, act));
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < T; k += 512)
    if (cur[k]) cur[k] = atomicAdd(&cursor[k], cur[k]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const bool active = key[i] != 0xffffffffu;
    const unsigned long long act = __ballot(active);
    const unsigned long long heads = run_heads(key[i], active);
    uint32_t base = 0;
    if (active && ((heads >> lane) & 1ull)) base = atomicAdd(&cur[key[i]], run_length(heads, act));
    const unsigned long long below = heads & ((2ull << lane) - 1ull);
    const int my_head = below ? 63 - __clzll((long long)below) : 0;
    base = __shfl(base, my_head);
    if (active) sorted[base + uint32_t(lane - my_head)] = r[i];
  }
}

// The two corners of a plane coordinate in its tile's window, and their
// weights (Cic2's).  A NaN coordinate has both corners at cell 0, as there.
__device__ __forceinline__ void plane_corners(float u, int origin, int res, int l[2], float w[2]) {
  const float f = floorf(u);
  l[0] = plane_cell(u, res) - origin;
  l[1] = u == u ? l[0] + 1 : l[0];
  w[0] = 1.0f - fabsf(u - f);
  w[1] = 1.0f - fabsf(u - (f + 1.0f));
}

__global__ void __launch_bounds__(512)
plane_accum_kernel(const float2 *__restrict__ sorted, const ChunkDesc *__restrict__ desc,
                   const uint32_t *__restrict__ nchunks, PlaneTiles t, float *__restrict__ partial) {
  __shared__ double win[kPwCells];
  if (blockIdx.x >= *nchunks) return;
  const ChunkDesc d = desc[blockIdx.x];
  const uint32_t tx = t.div_t.div(d.tile), ty = d.tile - tx * uint32_t(t.t);
  for (int i = threadIdx.x; i < kPwCells; i += 512) win[i] = 0.0;
  __syncthreads();
  float2 next = sorted[d.start + (threadIdx.x < d.count ? threadIdx.x : 0u)];
  for (uint32_t q = threadIdx.x; q < d.count; q += 512) {
    const float2 r = next;
    if (q + 512 < d.count) next = sorted[d.start + q + 512];
    int lx[2], ly[2];
    float wx[2], wy[2];
    plane_corners(r.x, int(tx) * kPt, t.res, lx, wx);
    plane_corners(r.y, int(ty) * kPt, t.res, ly, wy);
#pragma unroll
    for (int o = 0; o < 4; ++o)
      unsafeAtomicAdd(&win[lx[o & 1] * kPw + ly[o >> 1]], double(wx[o & 1] * wy[o >> 1]));
  }
  __syncthreads();
  float *out = partial + size_t(blockIdx.x) * kPwCells;
  for (int i = threadIdx.x; i < kPwCells; i += 512) out[i] = float(win[i]);
}

// blockIdx.x: tile; blockIdx.y: 4 of its 64 rows, one pixel per thread.  The
// pixels start from `before` (null: zero) and go to `after` or, when that is
// null, divided by the normalisation to the plane.
__global__ void __launch_bounds__(256)
plane_reduce_kernel(const float *__restrict__ partial, const uint32_t *__restrict__ nchunk,
                    const uint32_t *__restrict__ choff, PlaneTiles t, float norm, const double *before, double *after,
                    float *__restrict__ plane) {
  const int tx = int(t.div_t.div(blockIdx.x)), ty = int(blockIdx.x) - tx * t.t;
  const int a = int(blockIdx.y) * 4 + int(threadIdx.x >> 6), b = int(threadIdx.x & 63u);
  if (a >= plane_len(tx, t) || b >= plane_len(ty, t)) return;
  const int px = tx ? tx - 1 : t.t - 1, py = ty ? ty - 1 : t.t - 1;
  const uint32_t pixel = uint32_t(tx * kPt + a) * uint32_t(t.res) + uint32_t(ty * kPt + b);
  double acc = before ? before[pixel] : 0.0;
  for (int sx = 0; sx <= (a == 0 ? 1 : 0); ++sx)
    for (int sy = 0; sy <= (b == 0 ? 1 : 0); ++sy) {
      const uint32_t src = uint32_t(sx ? px : tx) * uint32_t(t.t) + uint32_t(sy ? py : ty);
      const int la = sx ? plane_len(px, t) : a, lb = sy ? plane_len(py, t) : b;
      const float *w = partial + size_t(choff[src]) * kPwCells + la * kPw + lb;
      const uint32_t n = nchunk[src];
      for (uint32_t k = 0; k < n; ++k) acc += double(w[size_t(k) * kPwCells]);
    }
  if (after)
    after[pixel] = acc;
  else
    plane[pixel] = float(acc) / norm;
}

// Adjoint of the density plane for a plane cotangent g (already divided by
// the normalisation): gpos[p] = (res / box_nx) sum_o g[idx_o] dW_o/dxy for
// the particles in the slab (the mod has derivative 1, the selection 0),
// 0 for the others and for z.
__global__ void __launch_bounds__(256)
density_plane_vjp_kernel(const float *__restrict__ pos, uint32_t n, float bnx, float lo, float hi, float res, int ires,
                         const float *__restrict__ g, float *__restrict__ gpos) {
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    float *o3 = gpos + 3 * size_t(p);
    const float d = pos[3 * size_t(p) + 2];
    float sx = 0.0f, sy = 0.0f;
    if (d > lo && d <= hi) {
      Cic2 c;
      cic2(plane_coord(pos[3 * size_t(p)], bnx, res), plane_coord(pos[3 * size_t(p) + 1], bnx, res), ires, ires, c);
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        const float v = g[c.idx[o]];
        sx += v * c.dx[o];
        sy += v * c.dy[o];
      }
      sx = sx * res / bnx;
      sy = sy * res / bnx;
    }
    o3[0] = sx;
    o3[1] = sy;
    o3[2] = 0.0f;
  }
}

__global__ void __launch_bounds__(256) plane_div_kernel(float *__restrict__ a, uint32_t m, float d) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) a[i] = a[i] / d;
}

__global__ void __launch_bounds__(256) plane_zero_kernel(float *__restrict__ a, uint32_t m) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) a[i] = 0.0f;
}

// fftfreq(n)[i] in float32: i / n for i < (n + 1) / 2, (i - n) / n above.
__device__ __forceinline__ float fftfreq(int i, int n) { return float(i < (n + 1) / 2 ? i : i - n) / float(n); }

// The Gaussian filter of utils.py:213-220 on the half spectrum of an
// [n0][n1] image: exp(-(|k| / s)^2 / 2) with |k| the norm of the two
// fftfreq wave numbers and s = 1 / (2 pi sigma) (norm.pdf(k, 0, s) /
// norm.pdf(0, 0, s)), times 1 / (n0 n1), the normalisation of ifft2.
__global__ void __launch_bounds__(256)
gaussian_filter_kernel(float2 *__restrict__ spec, int n0, int n1, float sd, float inv_m) {
  const int n1h = n1 / 2 + 1;
  const uint32_t H = uint32_t(n0) * uint32_t(n1h);
  for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < H; e += gridDim.x * blockDim.x) {
    const int a = int(e / uint32_t(n1h)), b = int(e % uint32_t(n1h));
    const float u = fftfreq(a, n0), v = fftfreq(b, n1);
    const float k = sqrtf(u * u + v * v);
    const float y = k / sd;
    const float f = expf(-(y * y) * 0.5f) * inv_m;
    const float2 z = spec[e];
    spec[e] = make_float2(z.x * f, z.y * f);
  }
}

int paint_2d(hipStream_t s, int nx, int ny, const float *pos, int64_t n, int stride, const float *weight,
             float *mesh) {
  JPM_REQUIRE(nx > 0 && ny > 0 && int64_t(nx) * ny <= kMaxCells, "plane shape (%d,%d) out of range", nx, ny);
  JPM_REQUIRE(n >= 0 && n <= int64_t(0xffffffffu), "particle count %lld out of range", (long long)n);
  JPM_REQUIRE(stride >= 2, "position stride %d must be at least 2", stride);
  if (n == 0) return JPM_OK;
  JPM_REQUIRE(pos && mesh, "null pointer argument");
  JPM_TIMED(s, "paint2d_kernel");
  hipLaunchKernelGGL(paint2d_kernel, dim3(grid_for(n, 256, 256 * 256)), dim3(256), 0, s, pos, uint32_t(n),
                     uint32_t(stride), weight, nx, ny, mesh);
  JPM_LAUNCHED("paint2d_kernel");
  return JPM_OK;
}

int paint_2d_vjp(hipStream_t s, int nx, int ny, const float *pos, int64_t n, int stride, const float *weight,
                 const float *g, float *gpos, int gstride, float *gweight) {
  JPM_REQUIRE(nx > 0 && ny > 0 && int64_t(nx) * ny <= kMaxCells, "plane shape (%d,%d) out of range", nx, ny);
  JPM_REQUIRE(n >= 0 && n <= int64_t(0xffffffffu), "particle count %lld out of range", (long long)n);
  JPM_REQUIRE(stride >= 2 && (!gpos || gstride >= 2), "strides must be at least 2");
  if (n == 0) return JPM_OK;
  JPM_REQUIRE(pos && g && (gpos || gweight), "null pointer argument");
  hipLaunchKernelGGL(paint2d_vjp_kernel, dim3(grid_for(n, 256, 256 * 256)), dim3(256), 0, s, pos, uint32_t(n),
                     uint32_t(stride), weight, nx, ny, g, gpos, uint32_t(gstride), gweight);
  JPM_LAUNCHED("paint2d_vjp_kernel");
  return JPM_OK;
}

// The slab bounds and the normalisation of lensing.py:32-40, evaluated as
// there: center -+ width / 2 and (box_nx / res)(box_ny / res) width in
// double precision, then rounded to float32 for the float32 comparisons and
// division.
struct PlaneArgs {
  float lo, hi, norm;
};

static PlaneArgs plane_args(int box_nx, int box_ny, double center, double width, int res) {
  PlaneArgs a;
  a.lo = float(center - width / 2.0);
  a.hi = float(center + width / 2.0);
  a.norm = float((double(box_nx) / double(res)) * (double(box_ny) / double(res)) * width);
  return a;
}

// Workspace of the sorted density plane (byte offsets); total 0 where one
// float atomic per corner is used instead: few particles, or more tiles than
// the LDS histogram holds.  A quarter of 64^3 particles takes 14-22 us by
// atomics and 29-45 us sorted, of 96^3 31-67 against 34-55 us, of 128^3
// 63-207 against 40-90 us (128^2 to 1024^2 pixels, both orders).
struct PlaneWs {
  uint32_t T, maxchunks;
  size_t count, nsel, tstart, cursor, nchunk, choff, totals, desc, recs, sorted, partial, sums, total;
};

static PlaneWs plane_ws(int64_t n, int res) {
  PlaneWs w{};
  if (n < kPlaneSortMin || n > int64_t(0xffffffffu) || res <= 0) return w;
  const uint64_t t = uint64_t((res + kPt - 1) / kPt);
  if (t * t > kPlaneMaxTiles) return w;
  w.T = uint32_t(t * t);
  const int64_t one = n < kPlanePass ? n : kPlanePass;
  w.maxchunks = uint32_t((uint64_t(one) + kPlaneChunk - 1) / kPlaneChunk + w.T);
  size_t o = 0;
  auto take = [&o](size_t bytes) {
    const size_t at = o;
    o += align_up(bytes);
    return at;
  };
  w.count = take((size_t(w.T) + 1) * 4);
  w.nsel = w.count + size_t(w.T) * 4;   // cleared with the counts
  w.tstart = take(size_t(w.T) * 4);
  w.cursor = take(size_t(w.T) * 4);
  w.nchunk = take(size_t(w.T) * 4);
  w.choff = take(size_t(w.T) * 4);
  w.totals = take(16);
  w.desc = take(size_t(w.maxchunks) * sizeof(ChunkDesc));
  w.recs = take(size_t(one) * sizeof(float2));
  w.sorted = take(size_t(one) * sizeof(float2));
  w.partial = take(size_t(w.maxchunks) * kPwCells * sizeof(float));
  w.sums = take(one < n ? size_t(res) * size_t(res) * sizeof(double) : 0);
  w.total = o;
  return w;
}

size_t density_plane_ws(int64_t n, int res) { return plane_ws(n, res).total; }

// The n particles of one sort; before, after: as for plane_reduce_kernel.
static int density_plane_sorted(hipStream_t s, const float *pos, uint32_t n, float bnx, const PlaneArgs &a, int res,
                                const double *before, double *after, float *plane, char *base, const PlaneWs &w) {
  PlaneTiles t;
  t.res = res;
  t.t = (res + kPt - 1) / kPt;
  t.div_t = FastDiv(uint32_t(t.t));
  auto *count = reinterpret_cast<uint32_t *>(base + w.count);
  auto *nsel = reinterpret_cast<uint32_t *>(base + w.nsel);
  auto *cursor = reinterpret_cast<uint32_t *>(base + w.cursor);
  auto *nchunk = reinterpret_cast<uint32_t *>(base + w.nchunk);
  auto *choff = reinterpret_cast<uint32_t *>(base + w.choff);
  auto *totals = reinterpret_cast<uint32_t *>(base + w.totals);
  auto *desc = reinterpret_cast<ChunkDesc *>(base + w.desc);
  auto *recs = reinterpret_cast<float2 *>(base + w.recs);
  auto *sorted = reinterpret_cast<float2 *>(base + w.sorted);
  auto *partial = reinterpret_cast<float *>(base + w.partial);
  const unsigned grid = unsigned((uint64_t(n) + kPlaneSelect - 1) / kPlaneSelect);
  hipLaunchKernelGGL(plane_clear_kernel, dim3((w.T + 64) / 64), dim3(64), 0, s, count, w.T + 1);
  JPM_LAUNCHED("plane_clear_kernel");
  hipLaunchKernelGGL(plane_select_kernel, dim3(grid), dim3(256), size_t(w.T) * 4, s, pos, n, bnx, a.lo, a.hi, t, nsel,
                     count, recs);
  JPM_LAUNCHED("plane_select_kernel");
  int rc = tile_table(s, count, w.T, kPlaneChunk, reinterpret_cast<uint32_t *>(base + w.tstart), cursor, nchunk, choff,
                      totals, desc);
  if (rc) return rc;
  hipLaunchKernelGGL(plane_scatter_kernel, dim3(grid), dim3(512), size_t(w.T) * 4, s, recs, nsel, t, cursor, sorted);
  JPM_LAUNCHED("plane_scatter_kernel");
  hipLaunchKernelGGL(plane_accum_kernel, dim3(w.maxchunks), dim3(512), 0, s, sorted, desc, totals + 1, t, partial);
  JPM_LAUNCHED("plane_accum_kernel");
  hipLaunchKernelGGL(plane_reduce_kernel, dim3(w.T, kPt / 4), dim3(256), 0, s, partial, nchunk, choff, t, a.norm,
                     before, after, plane);
  JPM_LAUNCHED("plane_reduce_kernel");
  return JPM_OK;
}

// ws: density_plane_ws(n, res) bytes, or null for the form without one.
int density_plane(hipStream_t s, const float *pos, int64_t n, int box_nx, int box_ny, double center, double width,
                  int res, float *plane, void *ws, size_t ws_bytes) {
  JPM_REQUIRE(box_nx > 0 && box_ny > 0, "box shape must be positive");
  JPM_REQUIRE(res > 0 && int64_t(res) * res <= kMaxCells, "plane resolution %d out of range", res);
  JPM_REQUIRE(n >= 0 && n <= int64_t(0xffffffffu), "particle count %lld out of range", (long long)n);
  JPM_REQUIRE(plane && (n == 0 || pos), "null pointer argument");
  const PlaneArgs a = plane_args(box_nx, box_ny, center, width, res);
  const uint32_t m = uint32_t(res) * uint32_t(res);
  JPM_TIMED(s, "density_plane");
  if (ws) {
    const PlaneWs w = plane_ws(n, res);
    JPM_REQUIRE(ws_bytes >= w.total, "the density plane needs %zu workspace bytes, got %zu", w.total, ws_bytes);
    if (w.total) {
      double *sums = reinterpret_cast<double *>(static_cast<char *>(ws) + w.sums);
      for (int64_t p0 = 0; p0 < n; p0 += kPlanePass) {
        const int64_t left = n - p0;
        const int rc = density_plane_sorted(s, pos + 3 * p0, uint32_t(left < kPlanePass ? left : kPlanePass),
                                            float(box_nx), a, res, p0 ? sums : nullptr,
                                            left > kPlanePass ? sums : nullptr, plane, static_cast<char *>(ws), w);
        if (rc) return rc;
      }
      return JPM_OK;
    }
  }
  hipLaunchKernelGGL(plane_zero_kernel, dim3(grid_for(m, 256, 4096)), dim3(256), 0, s, plane, m);
  JPM_LAUNCHED("plane_zero_kernel");
  if (n > 0) {
    hipLaunchKernelGGL(density_plane_kernel, dim3(grid_for(n, 256, 256 * 256)), dim3(256), 0, s, pos, uint32_t(n),
                       float(box_nx), a.lo, a.hi, float(res), res, plane);
    JPM_LAUNCHED("density_plane_kernel");
  }
  hipLaunchKernelGGL(plane_div_kernel, dim3(grid_for(m, 256, 4096)), dim3(256), 0, s, plane, m, a.norm);
  JPM_LAUNCHED("plane_div_kernel");
  return JPM_OK;
}

int density_plane_vjp(hipStream_t s, const float *pos, int64_t n, int box_nx, int box_ny, double center,
                      double width, int res, float *g, float *gpos) {
  JPM_REQUIRE(box_nx > 0 && box_ny > 0, "box shape must be positive");
  JPM_REQUIRE(res > 0 && int64_t(res) * res <= kMaxCells, "plane resolution %d out of range", res);
  JPM_REQUIRE(n >= 0 && n <= int64_t(0xffffffffu), "particle count %lld out of range", (long long)n);
  if (n == 0) return JPM_OK;
  JPM_REQUIRE(pos && g && gpos, "null pointer argument");
  const PlaneArgs a = plane_args(box_nx, box_ny, center, width, res);
  const uint32_t m = uint32_t(res) * uint32_t(res);
  // the cotangent of the division comes first (g is overwritten with g / norm)
  hipLaunchKernelGGL(plane_div_kernel, dim3(grid_for(m, 256, 4096)), dim3(256), 0, s, g, m, a.norm);
  JPM_LAUNCHED("plane_div_kernel");
  hipLaunchKernelGGL(density_plane_vjp_kernel, dim3(grid_for(n, 256, 256 * 256)), dim3(256), 0, s, pos, uint32_t(n),
                     float(box_nx), a.lo, a.hi, float(res), res, g, gpos);
  JPM_LAUNCHED("density_plane_vjp_kernel");
  return JPM_OK;
}

size_t gaussian_smoothing_ws(int n0, int n1) {
  if (n0 <= 0 || n1 <= 0) return 0;
  return size_t(n0) * size_t(n1 / 2 + 1) * sizeof(float2);
}

// out = Re ifft2(fft2(im) filter) for a real [n0][n1] image: an R2C of the
// image as a 1 x n0 x n1 mesh, the filter, a C2R.  in and out may be the
// same array.
int gaussian_smoothing(hipStream_t s, int n0, int n1, const float *im, float *out, double sigma, void *ws,
                       size_t ws_bytes) {
  JPM_REQUIRE(n0 > 0 && n1 > 0 && int64_t(n0) * n1 <= kMaxCells, "image shape (%d,%d) out of range", n0, n1);
  JPM_REQUIRE(sigma > 0.0, "smoothing scale must be positive");
  JPM_REQUIRE(im && out, "null pointer argument");
  const size_t need = gaussian_smoothing_ws(n0, n1);
  JPM_REQUIRE(ws && ws_bytes >= need, "gaussian smoothing needs %zu workspace bytes, got %zu", need, ws_bytes);
  JPM_TIMED(s, "gaussian_smoothing");
  int rc = fft_r2c(s, 1, n0, n1, 1, im, ws);
  if (rc) return rc;
  const double scale = 1.0 / (2.0 * M_PI * sigma);
  const uint32_t H = uint32_t(n0) * uint32_t(n1 / 2 + 1);
  hipLaunchKernelGGL(gaussian_filter_kernel, dim3(grid_for(H, 256, 4096)), dim3(256), 0, s,
                     static_cast<float2 *>(ws), n0, n1, float(scale), float(1.0 / (double(n0) * double(n1))));
  JPM_LAUNCHED("gaussian_filter_kernel");
  return fft_c2r(s, 1, n0, n1, 1, ws, out);
}

}  // namespace jpm
