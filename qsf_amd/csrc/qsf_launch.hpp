// qsf_launch.hpp — host-callable launchers of the HIP kernels (internal to libqsf_hip.so).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pass_params.hpp"

namespace qsf {

bool axis_size_supported(int64_t n);
// Launches one fused axis pass with kernel variant v (0 = default; see axis_variants);
// returns the number of blocks (or -1 if n is unsupported).
int launch_axis_pass(int precision, const PassParams& p, hipStream_t s, int v = 0);

// The flux stencil values of an X-representation state ahead of the pass that would gather
// them: out[k] = psi[row[k], pos[k]] times the pending X factor xa at that point (when has_xa),
// the same product the pass forms. Rows run along the last axis.
struct GatherXArgs {
  const void* psi;
  void* out;
  const int32_t* row;
  const int32_t* pos;
  int64_t nvals;
  int64_t n[3];
  int32_t dim;
  int32_t has_xa;
  XFactor xa;
};
void launch_gather_x(int precision, const GatherXArgs& a, hipStream_t s);
int64_t axis_pass_tiles(int precision, const PassParams& p, int v = 0);
// Number of compiled variants for an axis length (tile width x elements per thread).
int axis_variants(int64_t n);
// Fused 2D multigrid transfer into one receiving region (-1 if the length is unsupported).
int launch_transfer(int precision, const TransferParams& p, hipStream_t s);

// Per-axis phase tables of one substep, built on the device from FP64 scalars.
//   X table: expOp(δ·(Ne(x_i)·use_ne + x_i·C)) · absorber(δ, i)
//   P table: expOp(δ·(½p_i² + p_i·C)) · norm
struct AxisTableArgs {
  void* out;             // complex (precision) table of n entries
  int64_t n;
  int32_t kind;          // 0 = X, 1 = P
  int32_t mode;          // QSF_MODE_IM | QSF_MODE_RE
  double delta;
  double C;              // coupling value for this axis (0 if the gauge acts elsewhere)
  // X coordinates / potential / absorber
  double xmin, dx;
  int32_t use_ne;        // add the per-axis electron-nucleus term
  double NE, Nsoft;
  int32_t absorber;      // QSF_ABS_*; applied only when apply_abs
  int32_t apply_abs;
  int64_t nCAP;
  double eta, tau;
  // P coordinates (storage-axis parameters: dp, n, n/2)
  double dp;
  int64_t pn, pn2;
  double norm;
};
void launch_axis_tables(int precision, const AxisTableArgs* a, int count, hipStream_t s);

// Static pair tables exp(-iδ ee): kind PAIR_DIFF (n entries, |i-j|) or PAIR_FULL (n*n1). Model
// QSF_POT_COULOMB: the soft-core attraction over both coordinates (NE, Nsoft).
struct PairTableArgs {
  void* out;
  int64_t n, n1;
  double xmin1, dx1, NE, Nsoft;
  int32_t kind;          // PAIR_DIFF | PAIR_FULL
  int32_t model;         // QSF_POT_EBERLY | QSF_POT_ECKHARDT_SACHA
  int32_t mode;
  double delta, EE, Esoft, xmin, dx;
};
void launch_pair_table(int precision, const PairTableArgs& a, hipStream_t s);

// Potential tables (FP64): model QSF_POT_COULOMB: charge / sqrt(x_i^2 + soft), n entries; Eberly: by
// |i-j|, n entries; Eckhardt-Sacha: n * n1 entries (potential.h:130-179).
void launch_potential(double* out, int64_t n, int64_t n1, int model, double xmin, double dx, double charge, double soft,
                      hipStream_t s);

// psi *= exp(-i delta V) (RE) or exp(-delta V) (IM) with V = NE / sqrt(sum x_d^2 + Nsoft) over the
// bounded coordinates (CoulombInteraction, potential.h:40-44), in place on an X-rep state.
struct RadialArgs {
  void* psi;
  int precision;
  int64_t n[3];
  double xmin[3], dx[3];
  int bounded_mask;
  double NE, Nsoft, delta;
  int mode;
};
void launch_radial_x(const RadialArgs& a, hipStream_t s);

// roots[j] = exp(-2πi j/n), computed in FP64 and rounded to the precision.
void launch_roots(int precision, void* out, int64_t n, hipStream_t s);

// Sum of `count` blocks of `width` doubles into out[width] (fixed order). Large counts use a
// second level through `scratch` (256*width doubles). With ncols >= 0 only the first ncols
// doubles of each block are summed, into out[ncols] (a column reduced on its own: pass the
// partials from that column on).
void launch_reduce_partials(const double* partials, int64_t count, int width, double* out, double* scratch,
                            hipStream_t s, int ncols = -1);

// Flux through border families from gathered boundary values.
struct FluxArgs {
  const void* gathered;  // complex (precision)
  int32_t precision;
  const int32_t* pts;    // per point: [slot_c, slot_plus[d], slot_minus[d] for d < D] (1 + 2D ints)
  const double* bvec;    // per point: nb * D border components
  int64_t npts;
  int32_t D, nb;
  double inv_2dx[3];
  double vgC[3];         // velocity-gauge correction (0 if not velocity gauge)
  double scale;          // dV / dx0
  double* partials;      // per block: nb sums
  double* out;           // nb sums (after reduction), may be accumulated into
  double* accum;         // if non-null: accum[b] += out[b] * accum_weight
  double accum_weight;
};
void launch_flux(const FluxArgs& a, hipStream_t s);

// ---- lines: whole steps of a 1D propagation in one launch (line_impl.hpp) ----
enum LineFlags : uint32_t {
  LINE_OBS = 1u << 0,        // boundary observables of every step
  LINE_EPOT = 1u << 1,
  LINE_EKIN = 1u << 2,
  LINE_FLUX = 1u << 3,       // gather the flux stencil of every step
  LINE_NORMALIZE = 1u << 4,  // scale to unit norm at every boundary, before the observables
  LINE_STOP = 1u << 5        // stop once the energy difference is within `accuracy`
};
struct LineParams {
  void* psi;                 // in: step-boundary state, or (za_in) before its trailing X factor;
                             // out: the latter, or with LINE_EKIN or LINE_NORMALIZE the former
  const double2* za_in;      // trailing X factor of the step before the run, still to be applied
  const void* roots;
  int32_t steps, nsub;       // P substeps per step
  uint32_t flags;
  const double2* xtab;       // [step][nsub + 1][n] X factors, xtab_step elements per step (0: static)
  const double2* ptab;       // [step][nsub][n] P factors
  int64_t xtab_step, ptab_step;
  const double* vtab;        // potential of the nodes
  const double* kin_w;       // 1/2 p^2 of the nodes
  const int32_t* gather_pos; // node of each flux stencil value
  int32_t nvals;
  void* gathered;            // [step][nvals]
  double* sums;              // [step][wave][3]: norm, potential, kinetic
  double dV, dVm, last_energy, accuracy;
  int32_t* done;             // steps taken
};
// Launches the run; returns the waves per block (the layout of `sums`), also without launching
// when p.psi is null; -1: unsupported length. `variant`: the tuned variant of the length's row pass.
int launch_line(int precision, int64_t n, int variant, const LineParams& p, hipStream_t s);

constexpr int kLineTables = 320, kLineSteps = 128;   // tables and steps of one run
struct LineCouplings {
  double C[kLineTables];
  double delta[9];
  int32_t per_step;          // tables per step
};
// `tables` tables of a.n entries at a.out, table k with coupling c.C[k] and substep length
// c.delta[k % c.per_step].
void launch_line_tables(const AxisTableArgs& a, const LineCouplings& c, int tables, hipStream_t s);
struct LineRows {
  const double* sums;
  int32_t waves, nvals;
  double* rec;               // [step][rec_width]: norm, epot, ekin, fluxes
  int64_t rec_width;
  FluxArgs flux;             // nb = 0: no fluxes
};
// c.C[s] is the velocity-gauge correction of step s's fluxes.
void launch_line_rows(int precision, const LineRows& a, const LineCouplings& c, int steps, hipStream_t s);
// The flux time integrals of `steps` rows, added in step order.
void launch_row_integral(const LineRows& a, int steps, hipStream_t s);

// Element-wise multiply of a complex (precision) array by a real FP64 table value per point.
void launch_scale(int precision, void* psi, int64_t m, double s, hipStream_t st);
void launch_copy_convert(int from_prec, const void* src, int to_prec, void* dst, int64_t m, hipStream_t s);

}  // namespace qsf

namespace qsf {
// 2D multigrid transfer pieces (multigrid.h:454-616): gather + mask the edge slice of the
// source into `slice` (zero elsewhere), and dst += slice.
struct SliceArgs {
  const void* src;
  void* slice;
  int64_t n0, n1, n2;    // n2 = 1 for 2D
  int32_t dirFree;       // 0, 1 (2D, 3D) or 2 (3D)
  int64_t nCAP;
  const double* inv_tab; // inv_mask(node) for node in [0, nCAP]
  const double* corr_tab;// 2D: mask_correction by the other axis' node, or nullptr (not group 1)
  const double* m1_tab;  // 3D: mask(node) for node in [0, nCAP] when the receiver is group 1
};
void launch_slice_2d(int precision, const SliceArgs& a, hipStream_t s);
// 3D slices of every box at once: the boxes of multigrid.h:454-569 tile the sliding axis, and
// the transform along the freed axis never crosses them.
void launch_slice_3d(int precision, const SliceArgs& a, hipStream_t s);
void launch_add(int precision, void* dst, const void* src, int64_t m, hipStream_t s);
}  // namespace qsf

namespace qsf {
// ---- batched solves (one launch covers every solve of a size group; blockIdx.y = solve) ----
struct BatchTableArgs {       // P tables of one solve for the current device step
  void* out[2];
  int64_t n[2], pn[2], pn2[2];
  double dp[2];
  double delta;               // dt of the P substep
  const double* coupling;     // [total_steps][3]: A per axis of each step's P substep
  int64_t total_steps;
  int32_t storage_axis[2];    // coupling / P coordinates of the reference's storage axis
};
void launch_batch_ptables(int precision, const BatchTableArgs* dev_args, int nsolves, int64_t nmax,
                          const int64_t* step_ctr, hipStream_t s);

struct BatchObsArgs {         // observables of one solve at the boundary the pass observed
  const double* partials;
  int64_t tiles;
  const void* gathered;
  const double* coupling;     // [total_steps][3]
  int64_t total_steps;
  double* rec;                // [total_steps + 1][1 + nb]: norm, flux[nb]
  double* flux_int;           // [nb]
  double dV;
};
struct BatchFluxGeo {
  const int32_t* pts;
  const double* bvec;
  int64_t npts;
  int32_t D, nb, precision;
  double inv_2dx[3], scale, dt;
};
// Observes the boundary after step *step_ctr (called before the counter advances).
void launch_batch_obs(const BatchObsArgs* dev_args, int nsolves, const BatchFluxGeo& geo,
                      const int64_t* step_ctr, hipStream_t s);
void launch_step_increment(int64_t* step_ctr, hipStream_t s);
}  // namespace qsf
