/* Generated by geos-chem_amd/mechgen/emit_rates.py from mech/carbon.json -- do not edit. */
#pragma once
#include "species_carbon.h"

namespace gckpp {
// Update_RCONST of mechanism carbon: rc[r*rs] for r = 0..7, in parts
constexpr int RATE_PARTS_carbon = 1;
template <int P>
__device__ void rates_carbon(const rl::RateEnv &E, double *__restrict__ rc, int64_t rs);
template <>
__device__ __forceinline__ void rates_carbon<0>(const rl::RateEnv &E, double *__restrict__ rc,
    int64_t rs) {
  rc[0 * rs] = (2.45e-12*exp(-1775.0e0/E.TEMP)*E.TROP);
  rc[1 * rs] = (9.60e-12*exp(-1360.0e0/E.TEMP)*E.TROP);
  rc[2 * rs] = (E.K_TROP(0));
  rc[3 * rs] = (E.K_TROP(1));
  rc[4 * rs] = (E.K_TROP(2));
  rc[5 * rs] = (E.K_STRAT(0));
  rc[6 * rs] = (E.K_STRAT(1));
  rc[7 * rs] = (E.K_STRAT(2));
}
}  // namespace gckpp
