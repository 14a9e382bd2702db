// Real-space (short-range) part of P3M Coulomb on the device: every pair of
// charged particles closer than r_cut (minimum image) contributes the pair
// force and energy of CoulombP3M::pair_force / pair_energy (p3m.hpp:146-180,
// A&S erfc of AS_erfc_part.hpp:29-40), as the reference's short-range loop
// applies them over its cell system (forces.cpp:178-208).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace espresso_amd {

struct ShortRangeParams {
  double box[3] = {0., 0., 0.};
  double prefactor = 0.;
  double alpha = 0.;
  double r_cut = 0.;
  int subdivision = 0; // cells per r_cut: 0 or 2 = two, 1 = one
  // ELC dielectric contrasts: each pair within r_cut also gets the terms of
  // add_pair_force_corrections / pair_energy_correction (elc.hpp:250-296),
  // particle i against the image of itself in the layer it sits in
  bool elc_images = false;
  double elc_h = 0.;  // L_z - gap
  double elc_sl = 0.; // space layer
  double elc_dt = 0., elc_db = 0.;
};

struct ShortRangeResult {
  double energy = 0.;    // sum over pairs of the pair energy
  double virial[9] = {}; // sum over pairs of F_ij (x) d_ij, d_ij = r_i - r_j (row-major)
};

/** Cell-list pair solver.  Charged particles are counting-sorted into columns
 *  along z of edge >= r_cut (>= r_cut / 2 along an axis that holds fewer than
 *  three of those), cut into z bins; groups of 64 particles of a column take
 *  the particles of the columns around them (k_sr_columns).  With ELC images
 *  the sort is into cells of edge >= r_cut / s, s = 2 (or 1), at most 64 per
 *  dimension, and one workgroup per cell takes its particles against the
 *  (2 s + 1)^3 neighbour cells, staged through LDS with the periodic shift
 *  applied.  Forces accumulate in registers (FP64).  With fewer than 3 cells
 *  along a dimension it falls back to all pairs with the minimum-image
 *  displacement. */
class ShortRange {
public:
  explicit ShortRange(int device);
  ~ShortRange();
  ShortRange(ShortRange const &) = delete;
  ShortRange &operator=(ShortRange const &) = delete;

  /** Adds the pair forces to force (device arrays of n particles, stream
   *  st).  With out != nullptr the energy and virial are reduced and the
   *  call synchronises the stream. */
  void compute(hipStream_t st, ShortRangeParams const &p, int64_t n, double const *pos,
               double const *q, double *force, ShortRangeResult *out);

  /** Cells of edge >= r_cut / s, s = 1 with subdivision 1, else 2, that the
   *  box of the last call holds per dimension (1 1 1: all pairs).  The search
   *  with ELC images runs over these; the column search has a grid of its own
   *  and goes by them only for whether the box is wide enough. */
  void cells(int out[3]) const;

  /** Dipolar real space (DipolarP3M::pair_force / pair_energy,
   *  dp3m.hpp:160-235) over the same columns, for particles with a
   *  non-zero dipole: adds forces and torques ([n][3] device arrays, either
   *  may be null) and, with energy != null, returns the pair energy (the
   *  call then synchronises).  exact_erfc selects libm erfc for B_r (the
   *  reference's choice at accuracy <= 5e-6).  Returns false, doing
   *  nothing, when the box is narrower than five cells of edge r_cut / 2
   *  (three of r_cut with subdivision 1). */
  bool compute_dipolar(hipStream_t st, ShortRangeParams const &p, bool exact_erfc, int64_t n,
                       double const *pos, double const *dip, double *force, double *torque,
                       double *energy);

private:
  struct Impl;
  Impl *m;
};

} // namespace espresso_amd
