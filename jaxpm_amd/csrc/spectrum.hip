// Binned power spectra over R2C half spectra: the mode sums behind jaxpm
// utils.py:76-128 (power_spectrum) and its bin table utils.py:14-73.
//
// The half spectrum is walked flat, 64 consecutive modes a wave (coalesced,
// and no lane idles at the end of a row of nz/2 + 1 modes).  Per mode the
// wave forms |k| exactly as the reference bins it (float64 sum of squares,
// rounded to float32, float32 square root), finds the bin by binary search
// over the edges, and adds the mode and its Hermitian mirror (X(-k) = conj
// X(k), not stored in the half spectrum) to per-bin sums.  |k| grows along a
// row, so the lanes of one bin are neighbours: a segmented scan across the
// wave sums them and the last lane of each run adds the sum to the wave's
// own bins in LDS.  The waves' bins are then added in a fixed order, within
// the workgroup and, by a second kernel, over the workgroups.
//
// Bound by float64 instruction issue (the scans and the divisions by |k|),
// not by the 8 bytes a mode.  256^3, poles 0 2 4: 1671 + 127 us when each
// run of a bin was summed by its own full-wave reductions, the wave numbers
// divided per mode, and the partial sums added by one thread per slot; now
// 123 + 14 us.
#include <cmath>

#include "common.hpp"

namespace jpm {

constexpr int kPkMaxPoles = 8;
constexpr int kPkMaxSlots = 8192;   // accumulators x bins, float64 in LDS (64 KiB)
constexpr int kPkMaxWaves = 4;      // per workgroup, each with its own bins
constexpr int kPkLdsSlots = 4096;   // slots of all waves of a workgroup, when more than one
constexpr int kPkMaxBlocks = 2048;

struct PkParams {
  int nx, ny, nz, nzh;
  uint32_t modes;  // nx ny nzh
  FastDiv div_nzh, div_ny;
  double inv[3];   // 1 / n_d
  double fac[3];   // 2 pi n_d / L_d: cell wave number to h/Mpc
  double los[3];   // unit line of sight (multipoles only)
  int nedges, nbins, nslots, npoles, lmax;
  int poles[kPkMaxPoles];
};

// numpy.fft.fftfreq(n)[i] = i' * (1.0 / n), i' the signed index.
__device__ __forceinline__ double fftfreq(int i, int n, double inv) {
  const int s = i <= (n - 1) / 2 ? i : i - n;
  return double(s) * inv;
}

// (2 l + 1) P_l(mu) of every pole, by Bonnet's recurrence up to the largest.
template <int NP>
__device__ __forceinline__ void legendre_weights(const PkParams &p, double mu, double w[NP]) {
#pragma unroll
  for (int q = 0; q < NP; ++q) w[q] = p.poles[q] == 0 ? 1.0 : 3.0 * mu;
  double p0 = 1.0, p1 = mu;
  for (int n = 1; n < p.lmax; ++n) {
    const double p2 = (double(2 * n + 1) * mu * p1 - double(n) * p0) / double(n + 1);
    p0 = p1;
    p1 = p2;
#pragma unroll
    for (int q = 0; q < NP; ++q)
      if (p.poles[q] == n + 1) w[q] = double(2 * n + 3) * p1;
  }
}

// np.digitize(x, edges) for increasing edges: the number of edges <= x.
__device__ __forceinline__ int digitize(const double *edges, int n, double x) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (edges[mid] <= x)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// v of the lane that the DPP control names (lanes without one keep 0).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
  return __hiloint2double(hi, lo);
}

// Sum of v over the lanes from `head` to this one (head <= lane, the same for
// every lane of a run): row shifts by 1, 2, 4, 8 within rows of 16 lanes,
// then the last lane of row 0 / 2 into row 1 / 3 and of lane 31 into the
// upper half.
__device__ __forceinline__ double segment_scan(double v, int lane, int head) {
  const int r = lane & 15;
  double t;
  t = dpp_move<0x111, 0xf>(v);
  v += (r >= 1 && lane - 1 >= head) ? t : 0.0;
  t = dpp_move<0x112, 0xf>(v);
  v += (r >= 2 && lane - 2 >= head) ? t : 0.0;
  t = dpp_move<0x114, 0xf>(v);
  v += (r >= 4 && lane - 4 >= head) ? t : 0.0;
  t = dpp_move<0x118, 0xf>(v);
  v += (r >= 8 && lane - 8 >= head) ? t : 0.0;
  t = dpp_move<0x142, 0xa>(v);   // row_bcast:15
  v += ((lane & 16) && head < (lane & 48)) ? t : 0.0;
  t = dpp_move<0x143, 0xc>(v);   // row_bcast:31
  v += (lane >= 32 && head < 32) ? t : 0.0;
  return v;
}

// Slots per bin: 0 mode count, 1 sum of |k|, 2+q Re sum for pole q, and for
// cross spectra 2+npoles+q the Im sum.  acc is [wave][slot][bin], then the
// edges.
template <int NP, bool CROSS, bool ANISO>
__global__ __launch_bounds__(kPkMaxWaves * 64) void pk_bin_kernel(const float2 *__restrict__ s1,
                                                                  const float2 *__restrict__ s2,
                                                                  const double *__restrict__ edges, PkParams p,
                                                                  double *__restrict__ partial) {
  extern __shared__ double acc[];
  const int waves = int(blockDim.x >> 6), lane = int(threadIdx.x & 63u), wave = int(threadIdx.x >> 6);
  double *ed = acc + waves * p.nslots;
  for (int e = int(threadIdx.x); e < waves * p.nslots; e += int(blockDim.x)) acc[e] = 0.0;
  for (int e = int(threadIdx.x); e < p.nedges; e += int(blockDim.x)) ed[e] = edges[e];
  __syncthreads();
  double *mine = acc + wave * p.nslots;
  const uint32_t stride = gridDim.x * uint32_t(waves) * 64u;
  for (uint32_t base = (blockIdx.x * uint32_t(waves) + uint32_t(wave)) * 64u; base < p.modes; base += stride) {
    const uint32_t m = base + uint32_t(lane);
    const bool valid = m < p.modes;
    int bin = -1;
    bool pair = false;
    double ks = 0.0, re[NP], im[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) re[q] = im[q] = 0.0;
    if (valid) {
      const float2 a = s1[m];
      const float2 b = CROSS ? s2[m] : a;
      const uint32_t row = p.div_nzh.div(m);
      const int k = int(m - row * uint32_t(p.nzh));
      const uint32_t iu = p.div_ny.div(row);
      const int i = int(iu), j = int(row - iu * uint32_t(p.ny));
      const double kx = p.fac[0] * fftfreq(i, p.nx, p.inv[0]);
      const double ky = p.fac[1] * fftfreq(j, p.ny, p.inv[1]);
      const double kz = p.fac[2] * fftfreq(k, p.nz, p.inv[2]);
      // sqrtf rounds correctly here, as NumPy's float32 root does (with the
      // compiler's default options; the __fsqrt_rn intrinsic does not)
      const float kf = sqrtf(float(kx * kx + ky * ky + kz * kz));
      bin = digitize(ed, p.nedges, double(kf));
      pair = k > 0 && 2 * k != p.nz;   // mirror not stored
      const double xr = double(a.x) * double(b.x) + double(a.y) * double(b.y);
      const double xi = CROSS ? double(a.y) * double(b.x) - double(a.x) * double(b.y) : 0.0;
      ks = (pair ? 2.0 : 1.0) * double(kf);
      // the mirror carries conj: Re adds, Im subtracts
      if (!ANISO) {
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          re[q] = pair ? 2.0 * xr : xr;
          // 0 but for a mode that is not finite, whose imaginary part and its
          // mirror's cancel to NaN
          im[q] = pair ? 0.0 * xi : xi;
        }
      } else {
        const double tx = kx * p.los[0], ty = ky * p.los[1], tz = kz * p.los[2];
        double w[NP], wm[NP];
        legendre_weights<NP>(p, kf == 0.0f ? 0.0 : (tx + ty + tz) / double(kf), w);
        // The mirror of (kx, ky, kz) is its negative, and P_l(-mu) =
        // (-1)^l P_l(mu), except that Nyquist components mirror onto
        // themselves.
        const bool nx2 = 2 * i == p.nx, ny2 = 2 * j == p.ny;
        if (nx2 || ny2) {
          const double numm = (nx2 ? tx : -tx) + (ny2 ? ty : -ty) - tz;
          legendre_weights<NP>(p, kf == 0.0f ? 0.0 : numm / double(kf), wm);
        } else {
#pragma unroll
          for (int q = 0; q < NP; ++q) wm[q] = (p.poles[q] & 1) ? -w[q] : w[q];
        }
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          if (!pair) wm[q] = 0.0;
          re[q] = (w[q] + wm[q]) * xr;
          im[q] = (w[q] - wm[q]) * xi;
        }
      }
    }
    // runs of one bin (neighbouring lanes), each summed into its last lane
    const int prev = __shfl_up(bin, 1);
    const unsigned long long heads = __ballot(lane == 0 || bin != prev) | 1ull;
    const unsigned long long below = heads & ((2ull << lane) - 1ull);
    const int head = 63 - __clzll((long long)below);
    const bool last = lane == 63 || ((heads >> (lane + 1)) & 1ull);
    const unsigned long long run = ((2ull << lane) - 1ull) & ~((1ull << head) - 1ull);
    const unsigned long long pairs = __ballot(pair);
    ks = segment_scan(ks, lane, head);
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      re[q] = segment_scan(re[q], lane, head);
      if (CROSS) im[q] = segment_scan(im[q], lane, head);
    }
    if (last && bin >= 0) {
      unsafeAtomicAdd(&mine[bin], double(__popcll(run) + __popcll(run & pairs)));
      unsafeAtomicAdd(&mine[p.nbins + bin], ks);
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        if (q < p.npoles) {
          unsafeAtomicAdd(&mine[(2 + q) * p.nbins + bin], re[q]);
          if (CROSS) unsafeAtomicAdd(&mine[(2 + p.npoles + q) * p.nbins + bin], im[q]);
        }
      }
    }
  }
  __syncthreads();
  double *out = partial + size_t(blockIdx.x) * size_t(p.nslots);
  for (int e = int(threadIdx.x); e < p.nslots; e += int(blockDim.x)) {
    double v = acc[e];
    for (int w = 1; w < waves; ++w) v += acc[w * p.nslots + e];
    out[e] = v;
  }
}

// out[e] = the sum of slot e over the workgroups: one wave per slot, each lane
// a stride of 64 of them, then a fixed tree.
__global__ void __launch_bounds__(64) pk_reduce_kernel(const double *__restrict__ partial, int blocks, int nslots,
                                                       double *__restrict__ out) {
  const int e = int(blockIdx.x);
  double v = 0.0;
  for (int b = int(threadIdx.x); b < blocks; b += 64) v += partial[size_t(b) * size_t(nslots) + size_t(e)];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if (threadIdx.x == 0) out[e] = v;
}

// Waves of a workgroup: as many as have room for their own bins.
static int pk_waves(int nslots) {
  int w = kPkMaxWaves;
  while (w > 1 && w * nslots > kPkLdsSlots) w >>= 1;
  return w;
}

static int pk_blocks(int nx, int ny, int nz, int nslots) {
  const int64_t per = 64 * pk_waves(nslots);
  const int64_t b = (half_cells(nx, ny, nz) + per - 1) / per;
  return int(b < kPkMaxBlocks ? (b < 1 ? 1 : b) : kPkMaxBlocks);
}

template <int NP>
static auto pk_kernel(bool cross, bool aniso) {
  return cross ? (aniso ? pk_bin_kernel<NP, true, true> : pk_bin_kernel<NP, true, false>)
               : (aniso ? pk_bin_kernel<NP, false, true> : pk_bin_kernel<NP, false, false>);
}

int pk_slots(int nedges, int npoles, int cross) { return (2 + npoles * (cross ? 2 : 1)) * (nedges + 1); }

size_t power_spectrum_ws(int nx, int ny, int nz, int nedges, int npoles, int cross) {
  if (nx <= 0 || ny <= 0 || nz <= 0 || nedges < 0 || npoles < 1) return 0;
  const int nslots = pk_slots(nedges, npoles, cross);
  return size_t(pk_blocks(nx, ny, nz, nslots)) * size_t(nslots) * sizeof(double);
}

int power_spectrum(hipStream_t s, int nx, int ny, int nz, const void *spec1, const void *spec2, double fx, double fy,
                   double fz, const double *edges, int nedges, const int *poles, int npoles, double lx, double ly,
                   double lz, double *out, void *ws, size_t ws_bytes) {
  if (int rc = check_dims(nx, ny, nz)) return rc;
  JPM_REQUIRE(spec1 && out, "power spectrum: null spectrum or output");
  JPM_REQUIRE(nedges >= 0 && (nedges == 0 || edges), "power spectrum: %d edges", nedges);
  JPM_REQUIRE(npoles >= 1 && npoles <= kPkMaxPoles && poles, "power spectrum: 1..%d multipoles, got %d",
              kPkMaxPoles, npoles);
  const int cross = spec2 != nullptr;
  const int nslots = pk_slots(nedges, npoles, cross);
  JPM_REQUIRE(nslots <= kPkMaxSlots, "power spectrum: %d bins x %d sums exceed %d", nedges + 1,
              nslots / (nedges + 1), kPkMaxSlots);
  JPM_REQUIRE(ws_bytes >= power_spectrum_ws(nx, ny, nz, nedges, npoles, cross) && ws,
              "power spectrum: workspace of %zu bytes, need %zu", ws_bytes,
              power_spectrum_ws(nx, ny, nz, nedges, npoles, cross));
  PkParams p{};
  p.nx = nx;
  p.ny = ny;
  p.nz = nz;
  p.nzh = nz / 2 + 1;
  p.modes = uint32_t(half_cells(nx, ny, nz));
  p.div_nzh = FastDiv(uint32_t(p.nzh));
  p.div_ny = FastDiv(uint32_t(ny));
  p.inv[0] = 1.0 / double(nx);
  p.inv[1] = 1.0 / double(ny);
  p.inv[2] = 1.0 / double(nz);
  p.fac[0] = fx;
  p.fac[1] = fy;
  p.fac[2] = fz;
  p.los[0] = lx;
  p.los[1] = ly;
  p.los[2] = lz;
  p.nedges = nedges;
  p.nbins = nedges + 1;
  p.nslots = nslots;
  p.npoles = npoles;
  for (int q = 0; q < npoles; ++q) {
    JPM_REQUIRE(poles[q] >= 0 && poles[q] <= 64, "power spectrum: multipole %d outside [0, 64]", poles[q]);
    p.poles[q] = poles[q];
    if (poles[q] > p.lmax) p.lmax = poles[q];
  }
  const bool aniso = p.lmax > 0;
  const int blocks = pk_blocks(nx, ny, nz, nslots), waves = pk_waves(nslots);
  double *partial = static_cast<double *>(ws);
  const size_t lds = (size_t(waves) * size_t(nslots) + size_t(nedges)) * sizeof(double);
  auto kern = npoles == 1   ? pk_kernel<1>(cross, aniso)
              : npoles == 2 ? pk_kernel<2>(cross, aniso)
              : npoles == 3 ? pk_kernel<3>(cross, aniso)
                            : pk_kernel<kPkMaxPoles>(cross, aniso);
  if (lds > 65536)
    JPM_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(lds)));
  {
    JPM_TIMED(s, "pk_bin_kernel");
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * waves), lds, s, static_cast<const float2 *>(spec1),
                       static_cast<const float2 *>(cross ? spec2 : spec1), edges, p, partial);
    JPM_LAUNCHED("pk_bin_kernel");
  }
  {
    JPM_TIMED(s, "pk_reduce_kernel");
    hipLaunchKernelGGL(pk_reduce_kernel, dim3(nslots), dim3(64), 0, s, partial, blocks, nslots, out);
    JPM_LAUNCHED("pk_reduce_kernel");
  }
  return JPM_OK;
}

}  // namespace jpm
