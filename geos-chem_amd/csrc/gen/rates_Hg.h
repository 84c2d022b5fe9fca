/* Generated by geos-chem_amd/mechgen/emit_rates.py from mech/Hg.json -- do not edit. */
#pragma once
#include "species_Hg.h"

namespace gckpp {
// Update_RCONST of mechanism Hg: rc[r*rs] for r = 0..93, in parts
constexpr int RATE_PARTS_Hg = 1;
template <int P>
__device__ void rates_Hg(const rl::RateEnv &E, double *__restrict__ rc, int64_t rs);
template <>
__device__ __forceinline__ void rates_Hg<0>(const rl::RateEnv &E, double *__restrict__ rc,
    int64_t rs) {
  rc[0 * rs] = (rl::GCARR_ab(E, 1.46e-32,1.86e0)*E.NUMDEN);
  rc[1 * rs] = (rl::GCARR_abc(E, 1.6e-9,1.86e0,-7801.0e0)*E.NUMDEN);
  rc[2 * rs] = (3.9e-11);
  rc[3 * rs] = (3.0e-12);
  rc[4 * rs] = (rl::GCJPLPR_abab(E, 4.3e-30,5.9e0,1.2e-10,1.90e0,0.6e0));
  rc[5 * rs] = (rl::GCJPLPR_abab(E, 4.3e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[6 * rs] = (rl::GCJPLPR_abab(E, 4.3e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[7 * rs] = (rl::GCJPLPR_abab(E, 4.3e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[8 * rs] = (rl::GCJPLPR_abab(E, 4.3e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[9 * rs] = (3.0e-11);
  rc[10 * rs] = (rl::GCARR_ac(E, 4.1e-12,-856.0e0));
  rc[11 * rs] = (rl::GCARR_ac(E, 6.0e-11,-550.0e0));
  rc[12 * rs] = (3.0e-11);
  rc[13 * rs] = (rl::GCARR_ac(E, 2.25e-33,680.0e0)*E.NUMDEN);
  rc[14 * rs] = (3.9e-11);
  rc[15 * rs] = (3.0e-12);
  rc[16 * rs] = (rl::GCJPLPR_abab(E, 4.3e-30,5.9e0,1.2e-10,1.90e0,0.6e0));
  rc[17 * rs] = (rl::GCJPLPR_abab(E, 4.3e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[18 * rs] = (rl::GCJPLPR_abab(E, 4.3e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[19 * rs] = (rl::GCJPLPR_abab(E, 4.3e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[20 * rs] = (3.0e-11);
  rc[21 * rs] = (3.0e-11);
  rc[22 * rs] = (3.0e-11);
  rc[23 * rs] = (rl::GCARR_ac(E, 4.1e-12,-856.0e0));
  rc[24 * rs] = (rl::GCARR_ac(E, 6.0e-11,-550.0e0));
  rc[25 * rs] = (rl::GCARR_ac(E, 3.34e-33,43.0e0)*E.NUMDEN);
  rc[26 * rs] = (rl::GCARR_ac(E, 1.22e-9,-5720.0e0)*E.NUMDEN);
  rc[27 * rs] = (rl::GCJPLPR_abab(E, 4.1e-30,5.9e0,1.2E-10,1.90e0,0.6e0));
  rc[28 * rs] = (rl::GCJPLPR_abab(E, 4.1e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[29 * rs] = (rl::GCJPLPR_abab(E, 4.1e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[30 * rs] = (rl::GCJPLPR_abab(E, 4.1e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[31 * rs] = (rl::GCJPLPR_abab(E, 4.1e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[32 * rs] = (rl::GCJPLPR_abab(E, 4.1e-30,5.9e0,6.9e-11,2.40e0,0.6e0));
  rc[33 * rs] = (3.0e-11);
  rc[34 * rs] = (rl::GCARR_ac(E, 4.1e-12,-856.0e0));
  rc[35 * rs] = (rl::GCARR_ac(E, 6.0e-11,-550.0e0));
  rc[36 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgBrNO2)));
  rc[37 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgBrHO2)));
  rc[38 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgBrOH)));
  rc[39 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgBrBrO)));
  rc[40 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgBrClO)));
  rc[41 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgBr2)));
  rc[42 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgClNO2)));
  rc[43 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgClHO2)));
  rc[44 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgClOH)));
  rc[45 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgClBrO)));
  rc[46 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgClClO)));
  rc[47 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgClBr)));
  rc[48 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgCl2)));
  rc[49 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgOHNO2)));
  rc[50 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgOHHO2)));
  rc[51 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgOHOH)));
  rc[52 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgOHBrO)));
  rc[53 * rs] = (rl::Het_HgIIP_Org(E, 0.1e0,E.srmw(species_Hg::HgOHClO)));
  rc[54 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgBrNO2)));
  rc[55 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgBrHO2)));
  rc[56 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgBrOH)));
  rc[57 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgBrBrO)));
  rc[58 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgBrClO)));
  rc[59 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgBr2)));
  rc[60 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgClNO2)));
  rc[61 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgClHO2)));
  rc[62 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgClOH)));
  rc[63 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgClBrO)));
  rc[64 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgClClO)));
  rc[65 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgClBr)));
  rc[66 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgOHNO2)));
  rc[67 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgOHHO2)));
  rc[68 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgOHOH)));
  rc[69 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgOHBrO)));
  rc[70 * rs] = (rl::Het_HgIIP_Inorg(E, 0.1e0,E.srmw(species_Hg::HgOHClO)));
  rc[71 * rs] = (E.PHOTOL(24));
  rc[72 * rs] = (E.PHOTOL(25));
  rc[73 * rs] = (E.PHOTOL(26));
  rc[74 * rs] = (E.PHOTOL(3));
  rc[75 * rs] = (E.PHOTOL(6));
  rc[76 * rs] = (E.PHOTOL(7));
  rc[77 * rs] = (E.PHOTOL(8));
  rc[78 * rs] = (E.PHOTOL(9));
  rc[79 * rs] = (E.PHOTOL(10));
  rc[80 * rs] = (E.PHOTOL(11));
  rc[81 * rs] = (E.PHOTOL(13));
  rc[82 * rs] = (E.PHOTOL(14));
  rc[83 * rs] = (E.PHOTOL(15));
  rc[84 * rs] = (E.PHOTOL(16));
  rc[85 * rs] = (E.PHOTOL(17));
  rc[86 * rs] = (E.PHOTOL(18));
  rc[87 * rs] = (E.PHOTOL(5));
  rc[88 * rs] = (E.PHOTOL(19));
  rc[89 * rs] = (E.PHOTOL(20));
  rc[90 * rs] = (E.PHOTOL(4));
  rc[91 * rs] = (E.PHOTOL(22));
  rc[92 * rs] = (E.PHOTOL(23));
  rc[93 * rs] = (E.PHOTOL(12));
}
}  // namespace gckpp
