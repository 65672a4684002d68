// The growth-factor products of lpt (pm.py:77-124), shared by its passes.
#pragma once

#include "common.hpp"

namespace jpm {

// dx1 = c[0] F1, p1 = c[1] dx1, f1 = c[2] F1; dx2 = c[3] F2, p2 = c[4] dx2,
// f2 = c[5] F2.
struct LptCoef {
  float c[6];
};

// One component of (dx, p, f), in the reference's order of float32 products
// and sums.
__device__ __forceinline__ void lpt_combine(const LptCoef &lc, float F1, bool second, float F2, float &dx, float &p,
                                            float &f) {
  dx = lc.c[0] * F1;
  p = lc.c[1] * dx;
  f = lc.c[2] * F1;
  if (second) {
    const float dx2 = lc.c[3] * F2;
    dx = dx + dx2;
    p = p + lc.c[4] * dx2;
    f = f + lc.c[5] * F2;
  }
}

// (dx, p, f) at the lattice nodes from the potentials (stencil.hip; phi2 null:
// first order), and at positions from the force meshes (cic.hip; f2 null:
// first order).
int lpt_lattice(hipStream_t s, int nx, int ny, int nz, const float *phi1, const float *phi2, const LptCoef &lc,
                float *dx, float *p, float *f);
int lpt_read(hipStream_t s, int nx, int ny, int nz, const float *f1, const float *f2, const float *pos, int64_t n,
             bool rel, const LptCoef &lc, float *dx, float *p, float *f);

}  // namespace jpm
