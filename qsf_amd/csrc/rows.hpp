#pragma once
// rows.hpp — record rows of several step boundaries reduced together (rows.hip).
#include <hip/hip_runtime.h>

#include "qsf_launch.hpp"

namespace qsf {

constexpr int kRowSlots = 32;   // boundaries one reduction takes
struct RowSlots {
  const double* partials;    // [slot][tiles][3] block sums of the observing passes
  int64_t tiles;
  const double* kin;         // [slot][ktiles][3] block sums of the kinetic passes (third sum)
  int64_t ktiles;            // 0: no kinetic energy
  double* rec;               // [slot][rec_width]: norm, potential and kinetic sums, fluxes
  int64_t rec_width;
  double* scratch;           // [slot][256 * 2] second reduction level (more than 4096 tiles)
  FluxArgs flux;             // nb = 0: no fluxes; gathered: [slot][nvals]; partials: [slot][blocks * nb]
  int64_t nvals;
  double C[kRowSlots][3];    // velocity-gauge correction of each boundary
};
// out[i] = product of up to kFactors tables of n entries.
struct TableProduct {
  static constexpr int kFactors = 19;
  double2* out;
  int64_t n;
  int32_t count;
  const double2* in[kFactors];
};
void launch_table_products(const TableProduct* p, int count, hipStream_t s);

// The row of one step boundary in imaginary time, from the block sums of the passes that read the
// (not yet normalised) boundary state, and the scale that the next pass normalises it with.
struct GroundRow {
  const double* sums;        // [tiles][3]: norm, potential, kinetic sum of the last axis
  int64_t tiles;
  const double* kin;         // [ktiles][3]: kinetic sums of the other axes (third sum)
  int64_t ktiles;
  double* scratch;           // 256 * 4: second level (more than 8192 tiles)
  double dV, dVm, accuracy;
  int32_t steers;            // the energy difference ends the run (sets flags[0])
  double* state;             // [0] scale, [1] energy of the row before
  int32_t* flags;            // [0] halted, [1] rows taken
  double* rec;               // norm, potential and kinetic sums of the normalised state
};
void launch_ground_begin(double* state, int32_t* flags, double last_energy, int first, hipStream_t s);
void launch_ground_row(const GroundRow& g, hipStream_t s);
// psi *= state[0] (the scale of the last row)
void launch_ground_scale(int precision, void* psi, int64_t m, const double* state, hipStream_t s);

int flux_blocks(int64_t npts);
void launch_rows(int precision, const RowSlots& a, int slots, hipStream_t s);

}  // namespace qsf
