// Update_RCONST on the GPU (KPP/fullchem/gckpp_Rates.F90:408-1503): one lane
// per cell and part evaluates that part of the mechanism's generated rate
// program (gen/rates_<mech>.h) against the cell's inputs, read field-major
// with cells fastest.  The derived temperature terms and RELHUM are formed as
// Set_Kpp_GridBox_Values does (GeosCore/fullchem_mod.F90:2089-2167).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "cell_fields.h"
#include "gckpp_internal.h"
#include "hetlaws.h"
#include "ratelaws.h"
#include "gen/rates_fullchem.h"
#include "hglaws.h"
#include "gen/rates_Hg.h"
#include "gen/rates_carbon.h"

#define NSPEC_FULLCHEM species_fullchem::NSPEC

namespace gckpp {

__device__ inline rl::RateEnv make_env(const RatesArgs &a, int64_t cell, int nspec) {
  using namespace rl;
  RateEnv E;
  const int64_t n = a.ncell;
  E.met = a.met + cell;
  E.mstride = n;
  E.photol = a.photol + cell;
  E.pstride = n;
  E.het = a.het + (a.het_stride ? cell : 0);
  E.hstride = a.het_stride ? a.het_stride : 1;
  E.conc_p = a.conc + cell;
  E.cstride = n;
  E.consts = a.consts;
  E.nspec = nspec;
  const double T = E.met[(int64_t)MET_TEMP * n];
  E.TEMP = T;
  E.PRESS = E.met[(int64_t)MET_PRESS * n];
  E.NUMDEN = E.met[(int64_t)MET_NUMDEN * n];
  E.H2O = E.met[(int64_t)MET_H2O * n];
  E.SUNCOS = E.met[(int64_t)MET_SUNCOS * n];
  E.H_PLUS_G = E.met[(int64_t)MET_H_PLUS * n];
  E.SRHOBr = E.met[(int64_t)MET_SRHOBr * n];
  E.SRHOCl = E.met[(int64_t)MET_SRHOCl * n];
  E.SRO3 = E.met[(int64_t)MET_SRO3 * n];
  E.TROP = E.met[(int64_t)MET_TROP * n];
  E.INV_TEMP = 1.0 / T;
  E.TEMP_OVER_K300 = T / 300.0;
  E.K300_OVER_TEMP = 300.0 / T;
  E.SR_TEMP = sqrt(T);
  E.FOUR_R_T = 4.0 * kConR * T;
  E.FOUR_RGASLATM_T = 4.0 * kRgasLatm * T;
  E.EIGHT_RSTARG_T = 8.0 * kRstarG * T;
  double consexp = 17.2693882 * (T - 273.16) / (T - 35.86);
  double vpresh2o = kConsvap * exp(consexp) / T;
  E.RELHUM = (E.H2O / vpresh2o) * 100.0;
  return E;
}

// Block (x, y): part y for 64 cells; the blocks of a part run side by side, so
// that its code stays in the instruction caches (parts side by side for a
// cell: 1.08 -> 1.18 ms).  Bound by FP64 instructions (66k a cell, half of
// them exp, log and pow; 0.44 ms at full rate) beside 3.45 GB (0.6 ms).  As one
// function of 1,058 statements that reread its environment from scratch after
// every store (the coefficients might alias it: no exponential was shared) it
// took 111k instructions and 168 registers, 3,072 of a grid's 3,726 waves at a
// time.  Inlined by part, the output restrict, four waves a SIMD: 238,464
// cells 1.88 -> 0.86 ms.
#define GCKPP_RATES_KERNEL(NAME, NSPEC)                                        \
  template <int P>                                                             \
  __device__ __forceinline__ void part_##NAME(const RatesArgs &a, int64_t cell) { \
    if constexpr (P < RATE_PARTS_##NAME) {                                     \
      if ((int)blockIdx.y != P) return part_##NAME<P + 1>(a, cell);            \
      const rl::RateEnv E = make_env(a, cell, NSPEC);                          \
      rates_##NAME<P>(E, a.rconst + cell, a.ncell);                            \
    }                                                                          \
  }                                                                            \
  __global__ __launch_bounds__(64, 4) void k_rates_##NAME(RatesArgs a) {       \
    const int64_t cell = (int64_t)blockIdx.x * 64 + threadIdx.x;               \
    if (cell < a.ncell) part_##NAME<0>(a, cell);                               \
  }
GCKPP_RATES_KERNEL(fullchem, NSPEC_FULLCHEM)
GCKPP_RATES_KERNEL(Hg, species_Hg::NSPEC)
GCKPP_RATES_KERNEL(carbon, species_carbon::NSPEC)

bool rates_available(int mech) {
  return mech == MECH_FULLCHEM || mech == MECH_HG || mech == MECH_CARBON;
}

void launch_rates_mech(int mech, const RatesArgs &a, hipStream_t s) {
  auto grid = [&](int parts) { return dim3((unsigned)((a.ncell + 63) / 64), (unsigned)parts); };
  if (mech == MECH_FULLCHEM)
    hipLaunchKernelGGL(k_rates_fullchem, grid(RATE_PARTS_fullchem), dim3(64), 0, s, a);
  else if (mech == MECH_HG)
    hipLaunchKernelGGL(k_rates_Hg, grid(RATE_PARTS_Hg), dim3(64), 0, s, a);
  else if (mech == MECH_CARBON)
    hipLaunchKernelGGL(k_rates_carbon, grid(RATE_PARTS_carbon), dim3(64), 0, s, a);
}

}  // namespace gckpp
