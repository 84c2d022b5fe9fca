// The integrator state of one cell and its step control (ros_Integrator,
// KPP/fullchem/gckpp_Integrator.F90:578-786), for the solvers that keep it in
// registers.
#pragma once
#include "gckpp_internal.h"

namespace gckpp {

struct RosState {
  double T, H, Hnew, Hexit, Texit, HnewAcc;
  int st[8];
  int ierr, tries;
  bool rejLast, rejMore, newStep;
};

// The integrator state at the start of a cell's integration.
__device__ __forceinline__ void state_begin(const IntegrateArgs &a, int64_t cell, bool cold,
                                            RosState &S) {
  const RosParams &P = a.prm;
  const double hs = (a.hstart && !cold) ? a.hstart[cell] : 0.0;
  double Hstart = P.Hstart_default;
  if (hs > 0.0) Hstart = min_f(fabs(hs), fabs(P.Tend - P.Tstart));
  S.T = P.Tstart;
  double H = min_f(max_f(fabs(P.Hmin), fabs(Hstart)), fabs(P.Hmax));
  if (fabs(H) <= 10.0 * P.roundoff) H = P.DeltaMin;
  S.H = P.direction * H;
  S.Hnew = S.H;
  S.Hexit = S.Texit = S.HnewAcc = 0.0;
  for (int k = 0; k < 8; ++k) S.st[k] = 0;
  S.ierr = 1;
  S.rejLast = S.rejMore = false;
  S.newStep = true;
}

// Before a new step: true when the integration is over (S.ierr then holds
// IERR), else H is cut to what is left.
__device__ __forceinline__ bool state_done(const RosParams &P, RosState &S) {
  const bool more = (P.direction > 0) ? ((S.T - P.Tend) + P.roundoff <= 0.0)
                                      : ((P.Tend - S.T) + P.roundoff <= 0.0);
  if (!more) return true;
  if (S.st[2] > P.max_steps) { S.ierr = -6; return true; }
  if ((S.T + 0.1 * S.H) == S.T || S.H <= P.roundoff) { S.ierr = -7; return true; }
  S.H = min_f(S.H, fabs(P.Tend - S.T));
  return false;
}

// After an attempt with error norm err: the next step size and the counters;
// true when the step is accepted.
__device__ __forceinline__ bool state_step(const RosParams &P, double err, RosState &S) {
  const double H = S.H;
  const double fac = min_f(P.FacMax, max_f(P.FacMin, P.FacSafe / pow(err, 1.0 / kRosELO)));
  S.Hnew = H * fac;
  S.st[2] += 1;
  const bool ok = err <= 1.0 || H <= P.Hmin;
  if (ok) {
    S.st[3] += 1;
    S.T = S.T + P.direction * H;
    S.Hnew = max_f(P.Hmin, min_f(S.Hnew, P.Hmax));
    if (S.rejLast) S.Hnew = min_f(S.Hnew, H);
    S.Hexit = H;
    S.Texit = S.T;
    S.HnewAcc = S.Hnew;
    S.rejLast = S.rejMore = false;
  } else {
    if (S.rejMore) S.Hnew = H * P.FacRej;
    S.rejMore = S.rejLast;
    S.rejLast = true;
    if (S.st[3] >= 1) S.st[4] += 1;
  }
  S.H = S.Hnew;
  S.newStep = ok;
  return ok;
}

}  // namespace gckpp
