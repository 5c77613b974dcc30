#pragma once
// aux_device.hpp — device functions shared by the small kernels: one entry of a phase table and the
// border currents of one flux point.
#include <hip/hip_runtime.h>

#include "../../include/qsf_types.h"
#include "fft_core.hpp"
#include "qsf_launch.hpp"

namespace qsf {

__device__ __forceinline__ double2 axis_table_entry(const AxisTableArgs& a, int64_t i) {
  double h;
  if (a.kind == 0) {  // X: potential (per-axis part) + x·F  (hamiltonian.h:44-79)
    const double x = a.xmin + i * a.dx;
    const double ne = a.use_ne ? a.NE / sqrt(x * x + a.Nsoft) : 0.0;
    h = ne + x * a.C;
  } else {            // P: ½p² + p·A
    const double p = a.dp * (double)(i < a.pn2 ? i : i - a.pn);
    h = (0.5 * p * p) + (p * a.C);
  }
  const double v = a.delta * h;
  double re, im;
  if (a.mode == QSF_MODE_IM) { re = exp(-v); im = 0.0; }
  else { sincos(-v, &im, &re); }
  if (a.kind == 0 && a.apply_abs && a.absorber != QSF_ABS_NONE) {
    const int64_t half = a.n / 2;
    const int64_t nd = i < half ? -i : i - a.n + 1;   // neg_dist_from_edge grid.h:181-185
    const int64_t node = a.nCAP + nd;
    if (node > 0) {
      double f;
      if (a.absorber == QSF_ABS_CAP) {
        const double s4 = (double)(node * (node * (node * node)));
        f = exp(-a.delta * s4 * a.eta);                  // absorbers.h:40-46, one axis
      } else {
        // cos(π/2 · node/nCAP) as the sine of the distance from the edge (never negative)
        const double c = sin(0.5 * M_PI * (double)(a.nCAP - node) / (double)a.nCAP);
        f = pow(pow(c, 0.125), a.delta / a.tau);         // cos^(1/8) per tau of time
      }
      re *= f;
      im *= f;
    }
  }
  re *= a.norm;
  im *= a.norm;
  return double2{re, im};
}

// j[d] of one border point: the probability current from its stencil (grid.h:467-481) with the
// velocity-gauge correction C (propagator.h:249-257). q = [slot_c, slot_plus[D], slot_minus[D]].
template <typename T>
__device__ __forceinline__ void flux_currents(const int32_t* q, const T* g, int D, const double* inv_2dx,
                                              const double* C, double* j) {
  const T c = g[q[0]];
  const double cr = c.x, ci = c.y, nrm = cr * cr + ci * ci;
  for (int d = 0; d < D; ++d) {
    j[d] = 0.0;
    const int32_t sp = q[1 + d], sm = q[1 + D + d];
    if (sp >= 0 && sm >= 0) {
      // inv_2dx * Im(conj(ψ_c) (ψ_+ - ψ_-))
      const double dr = (double)g[sp].x - (double)g[sm].x, di = (double)g[sp].y - (double)g[sm].y;
      j[d] = inv_2dx[d] * (cr * di - ci * dr);
    }
    j[d] += C[d] * nrm;
  }
}

}  // namespace qsf
