// Real-space form of the default 4-point gradient.
//
// gradient_kernel(order=1) multiplies by i (8 sin w - sin 2w) / 6
// (kernels.py:63-66), which is exactly the Fourier multiplier of the central
// difference D f(c) = (8 (f(c+1) - f(c-1)) - (f(c+2) - f(c-2))) / 12 along the
// axis (with the forward transform's e^{-ikx} convention, f(c+1) <-> e^{ik}).
// So the three force meshes -IFFT[g_d P] of pm.py:54-56 equal -D_d phi with
// phi = IFFT[P]: one inverse FFT plus this stencil instead of three inverse
// FFTs.  D is antisymmetric (D^T = -D), which gives the adjoint below.
#include "lpt.hpp"

namespace jpm {

struct Mesh3 {
  uint32_t nx, ny, nz;
  FastDiv div_nz, div_ny;
};

// (i + d) mod n for |d| <= 2 and any n >= 1 (two corrections cover n = 1).
__device__ __forceinline__ uint32_t wrap_add(uint32_t i, int d, uint32_t n) {
  int r = int(i) + d;
  if (r < 0) r += int(n);
  if (r < 0) r += int(n);
  if (r >= int(n)) r -= int(n);
  if (r >= int(n)) r -= int(n);
  return uint32_t(r);
}

// -D phi at every cell, from one or two potentials, each workgroup marching
// 256 cells of a (y, z) plane through 8 x planes: the x neighbours move
// through registers, so a plane is read for its own step (and its rows again
// from L2 for the y and z neighbours) instead of once per x offset.
//   MODE 0: the three meshes out + d M of scale * -D phi1
//   MODE 1, 2: the LPT displacement, momentum and force of particles at the
//     lattice nodes (pm.py:79-124), where the CIC read of a force mesh is the
//     node's own value: dx = c0 F1, p = c1 dx, f = c2 F1, and with MODE 2 plus
//     dx2 = c3 F2, c4 dx2 and c5 F2; each (x, y, z) row of three staged in
//     LDS so that the stores are consecutive floats.
// Workgroups run in XCD slabs with neighbouring cells together: the 12 planes
// a plane's workgroups share (3 MB at 256^2) stay in that XCD's L2.
// 256^3: MODE 0 128 -> 46 us.  MODE 2 211 us (738 MB at 3.5 TB/s, limited by
// address and load issue; non-temporal stores of the results, 235 -> 218 us)
// in place of two MODE 0 passes, two force reads and nine elementwise passes,
// 1230 us.
constexpr int kMarch = 8;
typedef float fd4_vec __attribute__((ext_vector_type(4)));

// Orders a wave's LDS writes before its other lanes' reads of them (LDS
// operations of one wave complete in order; this keeps the compiler to it).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int MODE>
__global__ void __launch_bounds__(256)
fd4_march_kernel(const float *__restrict__ phi1, const float *__restrict__ phi2, Mesh3 g, float scale, LptCoef lc,
                 float *__restrict__ out0, float *__restrict__ out1, float *__restrict__ out2, uint32_t nqb,
                 uint32_t nblk, uint32_t per) {
  constexpr int NF = MODE == 2 ? 2 : 1;
  // a wave's own staging rows: no workgroup barrier in the march
  __shared__ __attribute__((aligned(16))) float st[MODE ? 4 * 576 : 4];
  const uint32_t item = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
  if (item >= nblk) return;
  const uint32_t xc = item / nqb, q0 = (item - xc * nqb) * 256u;
  const uint32_t yz = g.ny * g.nz, q = q0 + threadIdx.x;
  const bool valid = q < yz;
  const int lane = int(threadIdx.x & 63u);
  float *sw = st + (MODE ? (threadIdx.x >> 6) * 576 : 0);
  // rows of three floats in 16-byte stores where every plane starts on one
  const bool vec = MODE && (yz & 3u) == 0 &&
                   ((reinterpret_cast<uintptr_t>(out0) | reinterpret_cast<uintptr_t>(out1) |
                     reinterpret_cast<uintptr_t>(out2)) & 15u) == 0;
  const uint32_t w0 = q0 + (threadIdx.x & ~63u);
  const uint32_t cnt = w0 < yz ? 3u * (yz - w0 < 64u ? yz - w0 : 64u) : 0u;   // floats of the wave's cells
  const uint32_t qq = valid ? q : yz - 1;
  const uint32_t j = g.div_nz.div(qq), k = qq - j * g.nz;
  const uint32_t yp1 = wrap_add(j, 1, g.ny) * g.nz + k, ym1 = wrap_add(j, -1, g.ny) * g.nz + k;
  const uint32_t yp2 = wrap_add(j, 2, g.ny) * g.nz + k, ym2 = wrap_add(j, -2, g.ny) * g.nz + k;
  const uint32_t row = j * g.nz;
  const uint32_t zp1 = row + wrap_add(k, 1, g.nz), zm1 = row + wrap_add(k, -1, g.nz);
  const uint32_t zp2 = row + wrap_add(k, 2, g.nz), zm2 = row + wrap_add(k, -2, g.nz);
  const float c8 = scale * (8.0f / 12.0f), c1 = scale * (1.0f / 12.0f);
  const float *phi[2] = {phi1, phi2};
  const uint32_t x0 = xc * kMarch, x1 = x0 + kMarch < g.nx ? x0 + kMarch : g.nx;
  float w[NF][4];   // x - 2, x - 1, x, x + 1
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    w[f][0] = phi[f][size_t(wrap_add(x0, -2, g.nx)) * yz + qq];
    w[f][1] = phi[f][size_t(wrap_add(x0, -1, g.nx)) * yz + qq];
    w[f][2] = phi[f][size_t(x0) * yz + qq];
    w[f][3] = phi[f][size_t(wrap_add(x0, 1, g.nx)) * yz + qq];
  }
  // a plane's loads are all in flight together, and issued before the stores
  // of the plane before it (whose completion they would else wait for)
  float n[NF][9];
  auto load = [&](uint32_t xi) {
    // opaque, so that the loop keeps one base per plane and not 18 advancing
    // 64-bit lane pointers
    uint32_t x = xi;
    asm volatile("" : "+s"(x));
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const float *pl = phi[f] + size_t(x) * yz;
      n[f][0] = phi[f][size_t(wrap_add(x, 2, g.nx)) * yz + qq];
      n[f][1] = pl[yp1];
      n[f][2] = pl[ym1];
      n[f][3] = pl[yp2];
      n[f][4] = pl[ym2];
      n[f][5] = pl[zp1];
      n[f][6] = pl[zm1];
      n[f][7] = pl[zp2];
      n[f][8] = pl[zm2];
    }
  };
  load(x0);
  for (uint32_t x = x0; x < x1; ++x) {
    float F[NF][3];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const float xp2 = n[f][0];
      F[f][0] = -(c8 * (w[f][3] - w[f][1]) - c1 * (xp2 - w[f][0]));
      F[f][1] = -(c8 * (n[f][1] - n[f][2]) - c1 * (n[f][3] - n[f][4]));
      F[f][2] = -(c8 * (n[f][5] - n[f][6]) - c1 * (n[f][7] - n[f][8]));
      w[f][0] = w[f][1];
      w[f][1] = w[f][2];
      w[f][2] = w[f][3];
      w[f][3] = xp2;
    }
    if (x + 1 < x1) load(x + 1);
    if (MODE == 0) {
      const size_t M = size_t(g.nx) * yz, e = size_t(x) * yz + q;
      if (valid) {
        out0[e] = F[0][0];
        out0[M + e] = F[0][1];
        out0[2 * M + e] = F[0][2];
      }
    } else {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        float dx, p, f;
        lpt_combine(lc, F[0][d], MODE == 2, F[NF - 1][d], dx, p, f);
        sw[3 * lane + d] = dx;
        sw[192 + 3 * lane + d] = p;
        sw[384 + 3 * lane + d] = f;
      }
      wave_lds_fence();
      const size_t base = 3 * (size_t(x) * yz + w0);
      if (vec) {
        // 192 floats per array as 48 16-byte stores
        if (4u * uint32_t(lane) < cnt) {
          const int e = 4 * lane;
          __builtin_nontemporal_store(*reinterpret_cast<const fd4_vec *>(sw + e), reinterpret_cast<fd4_vec *>(out0 + base + e));
          __builtin_nontemporal_store(*reinterpret_cast<const fd4_vec *>(sw + 192 + e), reinterpret_cast<fd4_vec *>(out1 + base + e));
          __builtin_nontemporal_store(*reinterpret_cast<const fd4_vec *>(sw + 384 + e), reinterpret_cast<fd4_vec *>(out2 + base + e));
        }
      } else {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const uint32_t e = uint32_t(i) * 64u + uint32_t(lane);
          if (e < cnt) {
            out0[base + e] = sw[e];
            out1[base + e] = sw[192 + e];
            out2[base + e] = sw[384 + e];
          }
        }
      }
      wave_lds_fence();
    }
  }
}

// Adjoint of fd4_march_kernel<0>: out = scale * sum_d (D_d g_d), since
// (-D_d)^T = D_d.
__global__ void __launch_bounds__(256)
fd4_divergence_kernel(const float *__restrict__ g3, size_t chan_stride, Mesh3 g, float scale, float *__restrict__ out,
                      uint32_t per) {
  // blockIdx.y: mesh of a batch of equal shapes (stride M); the three input
  // channels lie chan_stride floats apart
  const uint32_t M = g.nx * g.ny * g.nz;
  g3 += size_t(blockIdx.y) * M;
  out += size_t(blockIdx.y) * M;
  const float c8 = scale * (8.0f / 12.0f), c1 = scale * (1.0f / 12.0f);
  const float *gx = g3, *gy = g3 + chan_stride, *gz = g3 + 2 * chan_stride;
  // workgroup b takes the 256 cells of block (b mod 8) per + b / 8: the
  // dispatcher deals workgroups to the 8 XCDs in turn, so each XCD sweeps one
  // contiguous slab of x planes and the reads at x +- 1, 2 hit its L2
  const uint32_t blk = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
  {
    const uint32_t e = blk * blockDim.x + threadIdx.x;
    if (e >= M) return;
    const uint32_t r = g.div_nz.div(e);
    const uint32_t k = e - r * g.nz;
    const uint32_t i = g.div_ny.div(r);
    const uint32_t j = r - i * g.ny;
    const uint32_t sx = g.ny * g.nz;
    const uint32_t row = e - k;
    const uint32_t plane = e - j * g.nz - k;
    const float dx = c8 * (gx[wrap_add(i, 1, g.nx) * sx + j * g.nz + k] - gx[wrap_add(i, -1, g.nx) * sx + j * g.nz + k]) -
                     c1 * (gx[wrap_add(i, 2, g.nx) * sx + j * g.nz + k] - gx[wrap_add(i, -2, g.nx) * sx + j * g.nz + k]);
    const float dy = c8 * (gy[plane + wrap_add(j, 1, g.ny) * g.nz + k] - gy[plane + wrap_add(j, -1, g.ny) * g.nz + k]) -
                     c1 * (gy[plane + wrap_add(j, 2, g.ny) * g.nz + k] - gy[plane + wrap_add(j, -2, g.ny) * g.nz + k]);
    const float dz = c8 * (gz[row + wrap_add(k, 1, g.nz)] - gz[row + wrap_add(k, -1, g.nz)]) -
                     c1 * (gz[row + wrap_add(k, 2, g.nz)] - gz[row + wrap_add(k, -2, g.nz)]);
    out[e] = (dx + dy) + dz;
  }
}

static Mesh3 make_mesh3(int nx, int ny, int nz) {
  Mesh3 g;
  g.nx = uint32_t(nx);
  g.ny = uint32_t(ny);
  g.nz = uint32_t(nz);
  g.div_nz = FastDiv(g.nz);
  g.div_ny = FastDiv(g.ny);
  return g;
}

template <int MODE>
static int fd4_march(hipStream_t s, int nx, int ny, int nz, const float *phi1, const float *phi2, float scale,
                     const LptCoef &lc, float *o0, float *o1, float *o2) {
  const Mesh3 g = make_mesh3(nx, ny, nz);
  const uint32_t nqb = uint32_t((int64_t(ny) * nz + 255) / 256), nxc = uint32_t((nx + kMarch - 1) / kMarch);
  const uint32_t nblk = nqb * nxc, per = (nblk + 7) / 8;
  hipLaunchKernelGGL(fd4_march_kernel<MODE>, dim3(8 * per), dim3(256), 0, s, phi1, phi2, g, scale, lc, o0, o1, o2,
                     nqb, nblk, per);
  JPM_LAUNCHED("fd4_march_kernel");
  return JPM_OK;
}

int fd4_gradient(hipStream_t s, int nx, int ny, int nz, const float *phi, float scale, float *out3) {
  int rc = check_dims(nx, ny, nz);
  if (rc) return rc;
  JPM_REQUIRE(phi && out3, "null pointer argument");
  JPM_REQUIRE(3 * cells(nx, ny, nz) <= (int64_t(1) << 32), "mesh too large");
  JPM_TIMED(s, "fd4_gradient_kernel");
  return fd4_march<0>(s, nx, ny, nz, phi, nullptr, scale, LptCoef{}, out3, nullptr, nullptr);
}

int lpt_lattice(hipStream_t s, int nx, int ny, int nz, const float *phi1, const float *phi2, const LptCoef &lc,
                float *dx, float *p, float *f) {
  JPM_REQUIRE(phi1 && dx && p && f, "null pointer argument");
  JPM_TIMED(s, "lpt_lattice");
  return phi2 ? fd4_march<2>(s, nx, ny, nz, phi1, phi2, 1.0f, lc, dx, p, f)
              : fd4_march<1>(s, nx, ny, nz, phi1, nullptr, 1.0f, lc, dx, p, f);
}

int fd4_divergence_batch(hipStream_t s, int nx, int ny, int nz, int batch, const float *g3, size_t chan_stride,
                         float scale, float *out) {
  int rc = check_dims(nx, ny, nz);
  if (rc) return rc;
  JPM_REQUIRE(g3 && out, "null pointer argument");
  JPM_REQUIRE(batch >= 1 && batch <= 65535, "batch of %d meshes", batch);
  const int64_t m = cells(nx, ny, nz);
  JPM_REQUIRE(3 * m <= (int64_t(1) << 32), "mesh too large");
  {
    JPM_TIMED(s, "fd4_divergence_kernel");
    const uint32_t blocks = uint32_t((m + 255) / 256), per = (blocks + 7) / 8;
    hipLaunchKernelGGL(fd4_divergence_kernel, dim3(8 * per, batch), dim3(256), 0, s, g3, chan_stride,
                       make_mesh3(nx, ny, nz), scale, out, per);
  }
  JPM_LAUNCHED("fd4_divergence_kernel");
  return JPM_OK;
}

int fd4_divergence(hipStream_t s, int nx, int ny, int nz, const float *g3, float scale, float *out) {
  return fd4_divergence_batch(s, nx, ny, nz, 1, g3, size_t(cells(nx, ny, nz)), scale, out);
}

}  // namespace jpm
