#pragma once
// line_impl.hpp — whole steps of a one-dimensional propagation in one launch (gfx950).
//
// A line of up to 4096 points fits the registers of one block, so the block keeps it there over a
// run of steps: X factor, forward transform, P factor, inverse transform, boundary observation,
// next step (chainEvolve, propagator.h:311-332, and computeEach, :275-300). Nothing of the state
// goes through HBM between steps and nothing is launched between them; per step the block reads
// its phase tables (built for the whole run beforehand by every CU of the device, prefetched
// ahead of the transform they follow) and writes a few sums and the flux stencil, which
// line_rows_kernel turns into record rows after the run.
//
// What bounds it: the one CU that holds the line. Threads per line are therefore as many as the
// plans give with radix-8 stages (512 threads at 4096 points: two waves on each SIMD), exchanges
// alternate between two LDS images of the line (one barrier each instead of two), and the twiddles
// stay in registers, or in LDS where the plan needs more than six records. Measured, a step: 4096
// points FP64, length gauge, energies and flux 49.9 -> 11.1 us (seven single-block launches before);
// 1536 points FP32, norm and flux 29.6 -> 10.9 us; 2560 points FP64 in imaginary time, with its
// four host round trips gone, 197 -> 25.5 us, by the mixed plan (five waves in place of two) 14.7 us.
#include "axis_pass_impl.hpp"

namespace qsf {

// Plan of a line in FP64 arithmetic: eight elements per thread where the length allows it (twelve
// for 3*2^k; the mixed plan for 5*2^k), so the long lines spread over all four SIMDs of the CU. FP32
// arithmetic keeps the plan of the tuned axis pass instead (each factorisation rounds its own way,
// and an FP32 run then gives the values it gives through the passes, whatever the path).
constexpr int line_alt(int n) {
  if (n % 5 == 0) return n >= 80 ? 2 : 0;
  if (n % 3 == 0) return n >= 48 ? 1 : 0;
  return n >= 128 && n != 512 ? 1 : 0;
}

// Exchange layout of a line held by several waves: the padded row layout in one of two images,
// swapped after every exchange. A wave can write image A again only after the barrier of the
// exchange through image B, which every wave reaches after its reads of A.
template <typename T, int STRIDE, bool WAVE> struct LineAddr {
  static constexpr bool kWave = WAVE;
  static constexpr bool kSplitOk = false;
  static constexpr bool kToggle = !WAVE;
  mutable int base;
  __device__ __forceinline__ int operator()(int p) const { return base + p + (p >> RowAddr<T>::SH); }
  __device__ __forceinline__ void flip() const { base = STRIDE - base; }
};

template <typename Real, int N, int LALT> struct LineGeo {
  using T = typename Tr<Real>::T;
  static constexpr int ALT = LALT;
  using PL = PlanOf<N, ALT>;
  static constexpr int TT = PL::T;
  // lines shorter than a wave's 64 threads are held several times over (only copy 0 is stored and
  // counted), so every lane of the wave takes part in the sums; where the line's threads are no whole
  // number of waves (the mixed plan) the lanes left over repeat its first threads, in the same LDS image
  static constexpr int THREADS = (TT + 63) / 64 * 64;
  static constexpr int COPIES = THREADS / TT;
  static constexpr int NWAVES = THREADS / 64;
  static constexpr bool WAVE = TT <= 64;
  static constexpr int STRIDE = row_stride<T, N>();
  static constexpr bool LDS_ROOTS = PL::NST > 1 && !Twiddles<N, ALT, T>::kPreload;
  static constexpr int exchange_bytes = (WAVE ? COPIES : 2) * STRIDE * (int)sizeof(T);
  static constexpr int roots_off = (exchange_bytes + 15) & ~15;
  static constexpr int red_off = roots_off + (LDS_ROOTS ? N * 16 : 0);
  static constexpr int bytes = red_off + 3 * NWAVES * (int)sizeof(double);
};

template <typename Real, int N, int LALT, bool S32>
__global__ void __launch_bounds__((LineGeo<Real, N, LALT>::THREADS)) line_kernel(LineParams p) {
  using G = LineGeo<Real, N, LALT>;
  using T = typename Tr<Real>::T;
  using S = StateOf<Real, S32>;
  using PL = typename G::PL;
  constexpr int ALT = G::ALT, E = PL::E, SLOTS = PL::SLOTS, TT = G::TT;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* lds = reinterpret_cast<T*>(smem_raw);
  double* red = reinterpret_cast<double*>(smem_raw + G::red_off);
  const int tid = threadIdx.x, t = tid % TT, copy = tid / TT, wave = tid >> 6;
  const bool valid = copy == 0;
  S* psi = reinterpret_cast<S*>(p.psi);

  T v[SLOTS];
#pragma unroll
  for (int q = 0; q < SLOTS; ++q) v[q] = from_state<T>(psi[PL::xpos(t, q)]);
  const T* roots = reinterpret_cast<const T*>(p.roots);
  if constexpr (G::LDS_ROOTS) {
    float4* dst = reinterpret_cast<float4*>(smem_raw + G::roots_off);   // 16 bytes per root
    const float4* src = reinterpret_cast<const float4*>(p.roots);
    for (int i = tid; i < N; i += G::THREADS) dst[i] = src[i];
    roots = reinterpret_cast<const T*>(smem_raw + G::roots_off);
    block_sync();
  }
  Twiddles<N, ALT, T> tw;
  tw.load(roots, t);
  LineAddr<T, G::STRIDE, G::WAVE> addr{G::WAVE && !PL::MIXED ? copy * G::STRIDE : 0};
  // the flux stencil slots of this thread's nodes
  const bool epot = p.flags & LINE_EPOT, ekin = p.flags & LINE_EKIN, flux = p.flags & LINE_FLUX;
  const bool obs = p.flags & LINE_OBS, normalise = p.flags & LINE_NORMALIZE;
  const bool formed = ekin || normalise;   // the boundary state itself is needed
  int slot[SLOTS];
  bool any = false;
#pragma unroll
  for (int q = 0; q < SLOTS; ++q) slot[q] = -1;
  if (flux && valid)
    for (int k = 0; k < p.nvals; ++k) {
      const int pos = p.gather_pos[k];
#pragma unroll
      for (int q = 0; q < SLOTS; ++q)
        if (PL::xhas(t, q) && PL::xpos(t, q) == pos) { slot[q] = k; any = true; }
    }

  // The step loop would otherwise hoist every power of the twiddles out of itself (84 registers at
  // 4096 points, all spilled): their values are made opaque before each transform.
  auto transform = [&](T* x, auto dir) {
    if constexpr (Twiddles<N, ALT, T>::kPreload) {
#pragma unroll
      for (int i = 0; i < Twiddles<N, ALT, T>::kTotal; ++i) {
        auto& r = tw.r[i];
        if constexpr (sizeof(T) == 16) asm volatile("" : "+v"(r.x), "+v"(r.y));
        else asm volatile("" : "+v"(r.x), "+v"(r.y), "+v"(r.z), "+v"(r.w));
      }
    }
    int to = t;
    if constexpr (E > 8 || G::NWAVES > 4) asm volatile("" : "+v"(to));   // and its exchange addresses
    fft<N, ALT, decltype(dir)::value>(x, to, lds, addr, roots, tw);
  };
  using FWD = std::integral_constant<int, -1>;
  using INV = std::integral_constant<int, +1>;
  auto wave_sum = [](double x) {
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    return x;
  };
  // sum of a per-wave value over the block, in wave order, known to every thread
  auto block_sum = [&](double x) {
    if constexpr (G::NWAVES == 1) {
      return x;
    } else {
      if ((tid & 63) == 0) red[wave] = x;
      block_sync();
      double a = 0.0;
      for (int k = 0; k < G::NWAVES; ++k) a += red[k];
      block_sync();
      return a;
    }
  };

  double2 za[SLOTS];        // the trailing X factor of the last step, where it is still to be applied
  bool pend = p.za_in != nullptr;
  if (pend) {
#pragma unroll
    for (int q = 0; q < SLOTS; ++q) za[q] = p.za_in[PL::xpos(t, q)];
  }
  double last = p.last_energy;
  int done = 0;
  for (int s = 0; s < p.steps; ++s) {
    const double2* xt = p.xtab + (int64_t)s * p.xtab_step;
    const double2* pt = p.ptab + (int64_t)s * p.ptab_step;
    for (int sub = 0; sub < p.nsub; ++sub) {
      {
        const double2* x = xt + (int64_t)sub * N;
#pragma unroll
        for (int q = 0; q < SLOTS; ++q) {
          double2 z = x[PL::xpos(t, q)];
          if (sub == 0 && pend) z = cmul(za[q], z);
          v[q] = capply(v[q], z);
        }
        pend = false;
      }
      double2 f[E];
#pragma unroll
      for (int q = 0; q < E; ++q) f[q] = pt[(int64_t)sub * N + t + TT * q];
      transform(v, FWD{});
#pragma unroll
      for (int q = 0; q < E; ++q) v[q] = capply(v[q], f[q]);
      if (sub == p.nsub - 1) {
#pragma unroll
        for (int q = 0; q < SLOTS; ++q) za[q] = xt[(int64_t)p.nsub * N + t + (PL::xpos(t, q) - t)];
      }
      transform(v, INV{});
      if constexpr (S32) {
        // the FP32 state is rounded once a substep, as the passes store it: a run's result does
        // not depend on how its steps are split into launches
#pragma unroll
        for (int q = 0; q < SLOTS; ++q) v[q] = from_state<T>(to_state<S>(v[q]));
      }
    }
    pend = true;
    ++done;
    if (!obs) continue;
    // the step boundary: observables weight |psi|^2 by |A|^2 where the state is not formed
    if (formed) {
#pragma unroll
      for (int q = 0; q < SLOTS; ++q) v[q] = capply(v[q], za[q]);
      pend = false;
    }
    if (normalise) {
      double a = 0.0;
#pragma unroll
      for (int q = 0; q < SLOTS; ++q)
        if (PL::xhas(t, q)) a += (double)v[q].x * (double)v[q].x + (double)v[q].y * (double)v[q].y;
      const double nrm = block_sum(wave_sum(valid ? a : 0.0));
      const double sc = sqrt(1.0 / (nrm * p.dV));
#pragma unroll
      for (int q = 0; q < SLOTS; ++q) v[q] = T{(Real)((double)v[q].x * sc), (Real)((double)v[q].y * sc)};
    }
    double nrm = 0.0, ep = 0.0, ek = 0.0;
#pragma unroll
    for (int q = 0; q < SLOTS; ++q) {
      if (!PL::xhas(t, q)) continue;
      double a2 = (double)v[q].x * (double)v[q].x + (double)v[q].y * (double)v[q].y;
      if (!formed) a2 *= cabs2(za[q]);
      nrm += a2;
      if (epot) ep += a2 * p.vtab[PL::xpos(t, q)];
    }
    if (any) {
      T* go = reinterpret_cast<T*>(p.gathered) + (int64_t)s * p.nvals;
#pragma unroll
      for (int q = 0; q < SLOTS; ++q)
        if (slot[q] >= 0) go[slot[q]] = formed ? v[q] : capply(v[q], za[q]);
    }
    if (ekin) {
      T u[SLOTS];
#pragma unroll
      for (int q = 0; q < SLOTS; ++q) u[q] = v[q];
      transform(u, FWD{});
#pragma unroll
      for (int q = 0; q < E; ++q)
        ek += ((double)u[q].x * (double)u[q].x + (double)u[q].y * (double)u[q].y) * p.kin_w[t + TT * q];
    }
    nrm = wave_sum(valid ? nrm : 0.0);
    if (epot) ep = wave_sum(valid ? ep : 0.0);
    if (ekin) ek = wave_sum(valid ? ek : 0.0);
    if ((tid & 63) == 0) {
      double* w = p.sums + ((int64_t)s * G::NWAVES + wave) * 3;
      w[0] = nrm;
      w[1] = ep;
      w[2] = ek;
    }
    if (p.flags & LINE_STOP) {
      // ENERGY_DIFFERENCE steers the loop (shouldContinue, propagator.h:304-309)
      const double curr = __dadd_rn(__dmul_rn(block_sum(ep), p.dV), __dmul_rn(block_sum(ek), p.dVm));
      const double dif = curr - last;
      last = curr;
      if (!(fabs(dif) > p.accuracy)) break;
    }
  }
  // a trailing factor that no observation formed stays pending: it meets the next run's first half
  if (valid) {
#pragma unroll
    for (int q = 0; q < SLOTS; ++q)
      if (PL::xhas(t, q)) psi[PL::xpos(t, q)] = to_state<S>(v[q]);
  }
  if (tid == 0 && p.done) *p.done = done;
}

template <typename Real, int N, int LALT, bool S32>
int launch_line_plan(const LineParams& p, hipStream_t s) {
  using G = LineGeo<Real, N, LALT>;
  static_assert(G::bytes <= 163840, "a line's LDS exceeds the 160 KiB of a CU");
  if (!p.psi) return G::NWAVES;   // geometry only
  static const bool attr_set = [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&line_kernel<Real, N, LALT, S32>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, G::bytes);
    return true;
  }();
  (void)attr_set;
  hipLaunchKernelGGL((line_kernel<Real, N, LALT, S32>), dim3(1), dim3(G::THREADS), G::bytes, s, p);
  return G::NWAVES;
}

// `alt`: the plan of the tuned row pass, for FP32 arithmetic.
template <typename Real, int N, bool S32>
int launch_line_size(const LineParams& p, int alt, hipStream_t s) {
  if constexpr (sizeof(Real) == 8) {
    return launch_line_plan<Real, N, line_alt(N), S32>(p, s);
  } else {
    if constexpr (tuned_length(N)) {
      if (alt) return launch_line_plan<Real, N, 1, S32>(p, s);
    }
    return launch_line_plan<Real, N, 0, S32>(p, s);
  }
}

}  // namespace qsf
