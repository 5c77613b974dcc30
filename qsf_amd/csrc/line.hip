// line.hip — launchers around the line kernel (line_impl.hpp): its phase tables for a run of
// steps, the kernel itself by runtime length, and the record rows of the run.
#include <hip/hip_runtime.h>

#include "../../include/qsf_types.h"
#include "aux_device.hpp"
#include "line_impl.hpp"

namespace qsf {

#define QSF_EXTERN_LINE(NN)                                                              \
  extern template int launch_line_size<double, NN, false>(const LineParams&, int, hipStream_t); \
  extern template int launch_line_size<float, NN, false>(const LineParams&, int, hipStream_t);  \
  extern template int launch_line_size<double, NN, true>(const LineParams&, int, hipStream_t);
QSF_SIZES(QSF_EXTERN_LINE)

template <typename Real, bool S32> static int dispatch_line(int64_t n, const LineParams& p, int alt, hipStream_t s) {
  switch (n) {
#define QSF_CASE(NN) case NN: return launch_line_size<Real, NN, S32>(p, alt, s);
    QSF_SIZES(QSF_CASE)
#undef QSF_CASE
    default: return -1;
  }
}

int launch_line(int precision, int64_t n, int variant, const LineParams& p, hipStream_t s) {
  const int alt = variant >= 0 && variant < axis_variants(n) ? var_alt(variant) : 0;
  if (precision == QSF_FP64) return dispatch_line<double, false>(n, p, alt, s);
  if (precision == QSF_FP32_STATE) return dispatch_line<double, true>(n, p, alt, s);
  return dispatch_line<float, false>(n, p, alt, s);
}

// Table blockIdx.y is table (y % per_step) of step y / per_step; its coupling value comes by value
// in the argument block, so a run's couplings need no copy of their own.
__global__ void line_tables_kernel(AxisTableArgs a, LineCouplings c) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  a.C = c.C[blockIdx.y];
  a.delta = c.delta[blockIdx.y % c.per_step];
  reinterpret_cast<double2*>(a.out)[(int64_t)blockIdx.y * a.n + i] = axis_table_entry(a, i);
}

void launch_line_tables(const AxisTableArgs& a, const LineCouplings& c, int tables, hipStream_t s) {
  const int threads = a.n < 256 ? 64 : 256;
  hipLaunchKernelGGL(line_tables_kernel, dim3((unsigned)((a.n + threads - 1) / threads), (unsigned)tables), dim3(threads),
                     0, s, a, c);
}

// One wave per step: the step's sums over the line kernel's waves and its fluxes, in fixed order.
template <typename Real>
__global__ void line_rows_kernel(LineRows a, LineCouplings c) {
  using T = typename cvec<Real>::T;
  const int s = blockIdx.x, lane = threadIdx.x;
  double* rec = a.rec + (int64_t)s * a.rec_width;
  if (lane < 3) {
    const double* w = a.sums + (int64_t)s * a.waves * 3 + lane;
    double x = 0.0;
    for (int k = 0; k < a.waves; ++k) x += w[3 * k];
    rec[lane] = x;
  }
  const T* g = reinterpret_cast<const T*>(a.flux.gathered) + (int64_t)s * a.nvals;
  const double C[3] = {c.C[s], 0.0, 0.0};
  for (int b = 0; b < a.flux.nb; ++b) {
    double x = 0.0;
    for (int64_t k = lane; k < a.flux.npts; k += 64) {
      double j[3];
      flux_currents(a.flux.pts + k * (1 + 2 * a.flux.D), g, a.flux.D, a.flux.inv_2dx, C, j);
      x += j[0] * a.flux.bvec[k * a.flux.nb + b];
    }
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    if (lane == 0) rec[3 + b] = x * a.flux.scale;
  }
}

// The flux time integrals take a run's rows in step order, whatever runs the steps came in.
__global__ void row_integral_kernel(LineRows a, int steps) {
  const int b = threadIdx.x;
  if (b >= a.flux.nb) return;
  double x = a.flux.accum[b];
#pragma unroll 8
  for (int s = 0; s < steps; ++s) x += a.rec[(int64_t)s * a.rec_width + 3 + b] * a.flux.accum_weight;
  a.flux.accum[b] = x;
}

void launch_row_integral(const LineRows& a, int steps, hipStream_t s) {
  hipLaunchKernelGGL(row_integral_kernel, dim3(1), dim3(64), 0, s, a, steps);
}

void launch_line_rows(int precision, const LineRows& a, const LineCouplings& c, int steps, hipStream_t s) {
  if (precision == QSF_FP32_MIXED)
    hipLaunchKernelGGL(line_rows_kernel<float>, dim3((unsigned)steps), dim3(64), 0, s, a, c);
  else
    hipLaunchKernelGGL(line_rows_kernel<double>, dim3((unsigned)steps), dim3(64), 0, s, a, c);
  if (a.flux.nb > 0 && a.flux.accum) launch_row_integral(a, steps, s);
}

}  // namespace qsf
