// rows.hip — record rows of several step boundaries reduced together. A boundary's sums and fluxes
// are small work (a few blocks, each with barriers between its levels): one at a time they cost
// 23 us of a 44 us step of a 256^2 plane (reduction 3.8, flux 9.5, its second level 9.6), and for
// up to kRowSlots boundaries together about the same once. The sums and their order are those of the
// single-boundary kernels, so the rows have the same bits.
#include <hip/hip_runtime.h>

#include "../../include/qsf_types.h"
#include "fft_core.hpp"
#include "rows.hpp"

namespace qsf {

// The first NC sums of slot blockIdx.y: block x takes chunk x of the slot's tiles (one chunk of all
// tiles where they are few).
template <int NC>
__global__ void rows_reduce_kernel(const double* in, int64_t slot_stride, int64_t count, int width, int64_t chunk,
                                   double* out, int64_t out_stride) {
  __shared__ double red[256];
  const double* p = in + (int64_t)blockIdx.y * slot_stride;
  const int64_t lo = (int64_t)blockIdx.x * chunk, hi = lo + chunk < count ? lo + chunk : count;
  for (int c = 0; c < NC; ++c) {
    double acc = 0.0;
    for (int64_t k = lo + threadIdx.x; k < hi; k += 256) acc += p[k * width + c];
    red[threadIdx.x] = acc;
    block_sync();
    for (int s = 128; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
      block_sync();
    }
    if (threadIdx.x == 0) out[(int64_t)blockIdx.y * out_stride + blockIdx.x * NC + c] = red[0];
    block_sync();
  }
}

template <typename Real, int D>
__global__ void rows_flux_kernel(RowSlots r) {
  using T = typename cvec<Real>::T;
  const FluxArgs& a = r.flux;
  const T* g = reinterpret_cast<const T*>(a.gathered) + (int64_t)blockIdx.y * r.nvals;
  const double* C = r.C[blockIdx.y];
  const int nb = a.nb;
  constexpr int stride = 1 + 2 * D;
  double acc[16];
#pragma unroll
  for (int b = 0; b < 16; ++b) acc[b] = 0.0;
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < a.npts;
       p += (int64_t)gridDim.x * blockDim.x) {
    const int32_t* q = a.pts + p * stride;
    const T c = g[q[0]];
    const double cr = c.x, ci = c.y, nrm = cr * cr + ci * ci;
    double j[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      j[d] = 0.0;
      const int32_t sp = q[1 + d], sm = q[1 + D + d];
      if (sp >= 0 && sm >= 0) {
        // inv_2dx * Im(conj(ψ_c) (ψ_+ - ψ_-))  (grid.h:467-481)
        const double dr = (double)g[sp].x - (double)g[sm].x, di = (double)g[sp].y - (double)g[sm].y;
        j[d] = a.inv_2dx[d] * (cr * di - ci * dr);
      }
      j[d] += C[d] * nrm;  // velocityGaugeCorrection (propagator.h:249-257)
    }
    const double* bv = a.bvec + p * nb * D;
#pragma unroll
    for (int b = 0; b < 16; ++b) {
      if (b >= nb) break;
      double s = 0.0;
#pragma unroll
      for (int d = 0; d < D; ++d) s += j[d] * bv[b * D + d];
      acc[b] += s;
    }
  }
  __shared__ double red[256];
#pragma unroll
  for (int b = 0; b < 16; ++b) {
    if (b >= nb) break;
    red[threadIdx.x] = acc[b];
    block_sync();
    for (int s = 128; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
      block_sync();
    }
    if (threadIdx.x == 0) a.partials[((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * nb + b] = red[0];
    block_sync();
  }
}

// One block per slot and border: the fixed tree of flux_finish_kernel over the flux blocks.
__global__ void rows_flux_finish_kernel(RowSlots r, int blocks) {
  __shared__ double red[256];
  const int b = blockIdx.x, nb = r.flux.nb;
  const double* p = r.flux.partials + (int64_t)blockIdx.y * blocks * nb;
  double acc = 0.0;
  for (int64_t k = threadIdx.x; k < blocks; k += blockDim.x) acc += p[k * nb + b];
  red[threadIdx.x] = acc;
  block_sync();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    block_sync();
  }
  if (threadIdx.x == 0) r.rec[(int64_t)blockIdx.y * r.rec_width + 3 + b] = red[0] * r.flux.scale;
}

struct ProductBatch {
  TableProduct p[16];
};
__global__ void table_products_kernel(ProductBatch b) {
  const TableProduct& p = b.p[blockIdx.y];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p.n) return;
  double2 z{1.0, 0.0};
  for (int k = 0; k < p.count; ++k) z = cmul(z, p.in[k][i]);
  p.out[i] = z;
}

void launch_table_products(const TableProduct* p, int count, hipStream_t s) {
  for (int off = 0; off < count; off += 16) {
    ProductBatch b{};
    const int k = count - off < 16 ? count - off : 16;
    int64_t nmax = 0;
    for (int i = 0; i < k; ++i) {
      b.p[i] = p[off + i];
      nmax = p[off + i].n > nmax ? p[off + i].n : nmax;
    }
    hipLaunchKernelGGL(table_products_kernel, dim3((unsigned)((nmax + 255) / 256), (unsigned)k), dim3(256), 0, s, b);
  }
}

__global__ void ground_begin_kernel(double* state, int32_t* flags, double last_energy, int first) {
  if (threadIdx.x) return;
  if (first) state[0] = 1.0;
  state[1] = last_energy;
  flags[0] = flags[1] = 0;
}

// Four sums over [lo, hi) of the boundary pass' blocks followed by the kinetic passes' blocks:
// norm, potential, kinetic of the boundary pass, kinetic of the others.
__device__ __forceinline__ void ground_sums(const GroundRow& g, int64_t lo, int64_t hi, double* out) {
  double a[4] = {0.0, 0.0, 0.0, 0.0};
  for (int64_t k = lo + threadIdx.x; k < hi; k += blockDim.x) {
    if (k < g.tiles) {
      for (int c = 0; c < 3; ++c) a[c] += g.sums[3 * k + c];
    } else {
      a[3] += g.kin[3 * (k - g.tiles) + 2];
    }
  }
  __shared__ double red[4][16];
  for (int c = 0; c < 4; ++c) {
    for (int off = 32; off > 0; off >>= 1) a[c] += __shfl_xor(a[c], off);
    if ((threadIdx.x & 63) == 0) red[c][threadIdx.x >> 6] = a[c];
  }
  block_sync();
  for (int c = 0; c < 4; ++c) {
    out[c] = 0.0;
    for (int w = 0; w < (int)blockDim.x / 64; ++w) out[c] += red[c][w];
  }
}

__global__ void __launch_bounds__(256) ground_chunks_kernel(GroundRow g, int64_t chunk) {
  if (*g.flags) return;
  const int64_t total = g.tiles + g.ktiles, lo = blockIdx.x * chunk, hi = lo + chunk < total ? lo + chunk : total;
  double a[4];
  ground_sums(g, lo, hi, a);
  if (threadIdx.x < 4) g.scratch[4 * blockIdx.x + threadIdx.x] = a[threadIdx.x];
}

__global__ void __launch_bounds__(1024) ground_row_kernel(GroundRow g, int chunks) {
  if (*g.flags) return;
  double a[4];
  if (chunks) {
    // sums of the chunks, in order, by one thread per column
    __shared__ double tot[4];
    if (threadIdx.x < 4) {
      double x = 0.0;
#pragma unroll 8
      for (int k = 0; k < chunks; ++k) x += g.scratch[4 * k + threadIdx.x];
      tot[threadIdx.x] = x;
    }
    block_sync();
    for (int c = 0; c < 4; ++c) a[c] = tot[c];
  } else {
    ground_sums(g, 0, g.tiles + g.ktiles, a);
  }
  if (threadIdx.x) return;
  const double s = sqrt(1.0 / (a[0] * g.dV)), s2 = s * s;
  const double epot = a[1] * s2, ekin = (a[2] + a[3]) * s2;
  g.rec[0] = a[0] * s2;
  g.rec[1] = epot;
  g.rec[2] = ekin;
  g.state[0] = s;
  ++g.flags[1];
  if (g.steers) {
    // shouldContinue (propagator.h:304-309)
    const double curr = __dadd_rn(__dmul_rn(epot, g.dV), __dmul_rn(ekin, g.dVm));
    const double dif = curr - g.state[1];
    g.state[1] = curr;
    if (!(fabs(dif) > g.accuracy)) g.flags[0] = 1;
  }
}

void launch_ground_begin(double* state, int32_t* flags, double last_energy, int first, hipStream_t s) {
  hipLaunchKernelGGL(ground_begin_kernel, dim3(1), dim3(64), 0, s, state, flags, last_energy, first);
}

void launch_ground_row(const GroundRow& g, hipStream_t s) {
  const int64_t total = g.tiles + g.ktiles;
  if (total <= 8192) {
    hipLaunchKernelGGL(ground_row_kernel, dim3(1), dim3(1024), 0, s, g, 0);
    return;
  }
  hipLaunchKernelGGL(ground_chunks_kernel, dim3(256), dim3(256), 0, s, g, (total + 255) / 256);
  hipLaunchKernelGGL(ground_row_kernel, dim3(1), dim3(64), 0, s, g, 256);
}

template <typename T> __global__ void ground_scale_kernel(T* psi, int64_t m, const double* state) {
  const double sc = state[0];
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
    const T v = psi[i];
    psi[i] = T{(decltype(v.x))(v.x * sc), (decltype(v.x))(v.y * sc)};
  }
}

void launch_ground_scale(int precision, void* psi, int64_t m, const double* state, hipStream_t s) {
  const int blocks = (int)((m + 255) / 256 < 8192 ? (m + 255) / 256 : 8192);
  if (precision == QSF_FP64)
    hipLaunchKernelGGL(ground_scale_kernel<double2>, dim3(blocks), dim3(256), 0, s, (double2*)psi, m, state);
  else
    hipLaunchKernelGGL(ground_scale_kernel<float2>, dim3(blocks), dim3(256), 0, s, (float2*)psi, m, state);
}

int flux_blocks(int64_t npts) {
  const int64_t want = (npts + 255) / 256;
  return (int)(want < 1 ? 1 : (want > 1024 ? 1024 : want));
}

template <int NC>
static void reduce_slots(const RowSlots& a, const double* in, int64_t tiles, double* out, int slots, hipStream_t s) {
  if (tiles <= 4096) {
    hipLaunchKernelGGL(rows_reduce_kernel<NC>, dim3(1, (unsigned)slots), dim3(256), 0, s, in, tiles * 3, tiles, 3, tiles,
                       out, a.rec_width);
    return;
  }
  const int64_t chunk = (tiles + 255) / 256;
  hipLaunchKernelGGL(rows_reduce_kernel<NC>, dim3(256, (unsigned)slots), dim3(256), 0, s, in, tiles * 3, tiles, 3, chunk,
                     a.scratch, (int64_t)512);
  hipLaunchKernelGGL(rows_reduce_kernel<NC>, dim3(1, (unsigned)slots), dim3(256), 0, s, (const double*)a.scratch,
                     (int64_t)512, (int64_t)256, NC, (int64_t)256, out, a.rec_width);
}

void launch_rows(int precision, const RowSlots& a, int slots, hipStream_t s) {
  reduce_slots<2>(a, a.partials, a.tiles, a.rec, slots, s);
  if (a.ktiles) reduce_slots<1>(a, a.kin + 2, a.ktiles, a.rec + 2, slots, s);
  if (a.flux.nb <= 0) return;
  const int blocks = flux_blocks(a.flux.npts);
  const dim3 grid((unsigned)blocks, (unsigned)slots);
  const bool f64 = precision == QSF_FP64;
  if (a.flux.D == 2) {
    if (f64) hipLaunchKernelGGL((rows_flux_kernel<double, 2>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((rows_flux_kernel<float, 2>), grid, dim3(256), 0, s, a);
  } else {
    if (f64) hipLaunchKernelGGL((rows_flux_kernel<double, 3>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((rows_flux_kernel<float, 3>), grid, dim3(256), 0, s, a);
  }
  hipLaunchKernelGGL(rows_flux_finish_kernel, dim3((unsigned)a.flux.nb, (unsigned)slots), dim3(256), 0, s, a, blocks);
  if (a.flux.accum) {
    LineRows l{};
    l.rec = a.rec;
    l.rec_width = a.rec_width;
    l.flux = a.flux;
    launch_row_integral(l, slots, s);
  }
}

}  // namespace qsf
