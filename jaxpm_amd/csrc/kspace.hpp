// Per-axis Fourier multiplier tables and the potential multiplier, shared by
// the k-space passes (kspace.hip) and the FFT pass that applies the
// potential between its forward and inverse column transforms (fftk.hip).
#pragma once

#include "common.hpp"

namespace jpm {

// Per-axis tables, each of length nx + ny + nzh (x entries, then y, then z):
//   k    : wave number 2*pi*fftfreq(n) in radians per cell (fftk)
//   k2   : k^2, or (k sinc(k/2pi))^2 with JPM_K_LAPL_FD (invlaplace_kernel)
//   k2e  : k^2 (longrange_kernel always uses the plain k^2)
//   g    : gradient_kernel coefficient a, the kernel being i*a
//   s    : sinc(k/2pi) (cic_compensation = (sx sy sz)^-2)
struct Tabs {
  const float *k, *k2, *k2e, *g, *s;
  uint32_t oy, oz;  // offsets of the y and z entries
};

// The cached tables of a mesh shape and flags (JPM_K_GRAD_EXACT,
// JPM_K_LAPL_FD select the variants).
int get_tabs(hipStream_t st, int nx, int ny, int nz, uint32_t flags, Tabs &t);

// invlaplace_kernel (kernels.py:90-92): -1/kk, 0 at kk == 0.
__device__ __forceinline__ float green(float kk) { return kk == 0.0f ? 0.0f : -(1.0f / kk); }

// The potential multiplier at mode (i, jy, kz) (table indices, jy and kz
// already offset): scale * G(k) [* exp(-k^2 r2)] [/ (sx sy sz)^2]
// (pm.py:49-52 with kernels.py:69-115).
__device__ __forceinline__ float potential_factor(const Tabs &t, uint32_t i, uint32_t jy, uint32_t kz, float r2,
                                                  int deconv, float scale) {
  float kk = (t.k2[i] + t.k2[jy]) + t.k2[kz];
  float f = green(kk);
  if (r2 != 0.0f) {
    float kke = (t.k2e[i] + t.k2e[jy]) + t.k2e[kz];
    f = f * expf(-kke * r2);
  }
  if (deconv) {
    float p = (t.s[i] * t.s[jy]) * t.s[kz];
    f = f / (p * p);
  }
  return f * scale;
}

// jnp.interp(x, xp, fp) with the default clamping (fp[0] left of xp[0],
// fp[-1] right of xp[-1]).
__device__ __forceinline__ float interp(float x, const float *xp, const float *fp,
                                        int n) {
  // i = clip(searchsorted(xp, x, side='right'), 1, n - 1)
  int lo = 0, hi = n;
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (xp[mid] <= x) lo = mid + 1; else hi = mid;
  }
  int i = lo < 1 ? 1 : (lo > n - 1 ? n - 1 : lo);
  float df = fp[i] - fp[i - 1];
  float dx = xp[i] - xp[i - 1];
  float delta = x - xp[i - 1];
  float f = (fabsf(dx) <= 0.0f) ? fp[i - 1] : fp[i - 1] + (delta / dx) * df;
  if (x < xp[0]) f = fp[0];
  if (x > xp[n - 1]) f = fp[n - 1];
  return f;
}

// The linear field's multiplier (pm.py:137-143): sqrt(P(|k|) M / V) scale.
struct LinearArgs {
  float3 box, nm;
  float mcells, vol, scale;
  const float *ktab, *pktab;
  int ntab;
  const float *boxes;   // per-item boxes (3 floats) and P(k) tables, or null
  __device__ __forceinline__ void item(uint32_t b) {
    if (!boxes) return;
    pktab += size_t(b) * ntab;
    box = make_float3(boxes[3 * b], boxes[3 * b + 1], boxes[3 * b + 2]);
    vol = float(double(box.x) * double(box.y) * double(box.z));
  }
};

__device__ __forceinline__ float linear_factor(const Tabs &t, uint32_t i, uint32_t jy, uint32_t kz,
                                               const LinearArgs &a) {
  // pm.py:137-138: (k_i / L_i * n_i)^2 summed, then ** 0.5
  const float ax = t.k[i] / a.box.x * a.nm.x, ay = t.k[jy] / a.box.y * a.nm.y, az = t.k[kz] / a.box.z * a.nm.z;
  const float kmesh = sqrtf((ax * ax + ay * ay) + az * az);
  const float pk = interp(kmesh, a.ktab, a.pktab, a.ntab);
  return sqrtf(pk * a.mcells / a.vol) * a.scale;
}

}  // namespace jpm
