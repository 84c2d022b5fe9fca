// Persistent lane-per-cell Rodas3 solver for a small mechanism: one lane's
// whole cell in registers, its Fun, Jacobian, LU and substitutions straight-line
// code (gen/unroll_<mech>.h, mechgen/unroll.py).  The operations and their
// order are those of k_persist's table walk, so the results are bit-identical.
//
// The table walk reads every operand from the wave's slot block in memory, a
// wait every few FMAs; a Hg cell is 161 LU entries and 32 species, and an
// attempt about 4,000 FP64 instructions.  Here they are that many instructions
// on values that mostly stay on the CU: the diagonal and the vectors in 512
// registers, the other LU entries and the fixed species in 80 KB of LDS a wave.
// What does not fit goes to memory: the state and 74 rate constants to the slot
// block, 162 of the values between the partials and the LU to scratch (376
// bytes a lane).  So two waves a CU; with four (40 KB each, the LU in registers)
// the compiler spilled 200 to 500 values and the spills' way to memory bounded
// the kernel (21.6 ms of the step below).  Lanes take new cells from the counter sixteen at a time: a
// refill's loads wait once for all of them.
// Measured on the 72x46x72 grid (238,464 Hg cells, cold step): 38.1 ms with the
// table walk, 11.9 ms here, 70 us an attempt and wave, two thirds of it waiting
// for the rate constants and state from L2 and for divisions in the backward
// substitution.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstdint>

#include "gckpp_internal.h"
#include "mech_traits.h"
#include "ros_state.h"

namespace gckpp {
namespace {

#include "gen/unroll_Hg.h"

template <class M> struct Unrolled;
template <> struct Unrolled<Traits_Hg> {
  static constexpr int NG = unroll_Hg::NLU_LDS, NL = unroll_Hg::NRATE_LDS;
  static constexpr int LDS_FIELDS = unroll_Hg::LDS_FIELDS;
  template <class... A>
  static __device__ __forceinline__ void fun(A &&...a) { unroll_Hg::fun(a...); }
  template <class... A>
  static __device__ __forceinline__ void fun_partials(A &&...a) { unroll_Hg::fun_partials(a...); }
  template <class... A>
  static __device__ __forceinline__ bool lu(A &&...a) { return unroll_Hg::lu(a...); }
  template <class... A>
  static __device__ __forceinline__ void solve(A &&...a) { unroll_Hg::solve(a...); }
};
static_assert(Unrolled<Traits_Hg>::LDS_FIELDS * 64 * sizeof(double) == kUnrolledLds, "LDS of a wave");

typedef __attribute__((address_space(3))) double lds_double;
typedef unsigned int u32x2 __attribute__((__vector_size__(8)));
constexpr int kRefill = 16;  // idle lanes that start a refill

// k_persist's loop with the state in registers; a workgroup is one wave with
// kUnrolledLds of LDS and its slot block.
template <class M>
__global__ __launch_bounds__(64, 1) void k_lane_unrolled(PersistArgs pa) {
  using U = Unrolled<M>;
  constexpr int N = M::NVAR, NF = M::NFIX, NG = U::NG, NL = U::NL;
  extern __shared__ double un_lds[];
  const int lane = threadIdx.x;
  const int64_t wave = blockIdx.x;
  lds_double *const own = (lds_double *)un_lds + lane;
  // the wave's slot block: the rate constants past LDS, then Y, a field of 64
  // doubles at a constant offset from a buffer resource
  constexpr int SY = M::NREACT - NL;
  const __amdgpu_buffer_rsrc_t slot = __builtin_amdgcn_make_buffer_rsrc(
      pa.work + wave * (64 * pa.slot_fields), (short)0, (int)(64 * pa.slot_fields * 8), 0x00020000);
  auto get = [&](int f) -> double {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(slot, lane * 8, f * 512, 0));
  };
  auto put = [&](int f, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), slot, lane * 8, f * 512, 0);
  };
  const IntegrateArgs &a = pa.q[0];
  const RosParams &P = a.prm;
  const int64_t total = pa.qend[0];
  // LDS fields: LU entries, fixed species, rate constants
  auto lds = [&](int k) -> double { return own[k * 64]; };
  auto put_lds = [&](int k, double v) { own[k * 64] = v; };
  auto fix = [&](int s) -> double { return own[(NG + s) * 64]; };
  auto rate = [&](int r) -> double { return r < NL ? own[(NG + NF + r) * 64] : get(r - NL); };
  // (no value of LDS or the slot block is kept in a register across this)
  auto reread = [] { asm volatile("" ::: "memory"); };

  RosState S{};
  int64_t cell = -1;
  bool first = true, drained = false;
  auto load = [&]() {
#pragma unroll
    for (int i = 0; i < N; ++i) put(SY + i, a.conc[(int64_t)i * a.cstride + cell]);
  };
  for (;;) {
    const unsigned long long idle = __ballot(cell < 0 && !drained);
    const unsigned long long busy = __ballot(cell >= 0);
    if (!idle && !busy) break;
    if (idle && (!busy || __popcll(idle) >= kRefill)) {
      if (cell < 0 && !drained) {
        int64_t c;
        if (pa.counter) c = (int64_t)atomicAdd(pa.counter, 1u);
        else c = first ? wave * 64 + lane : total;
        first = false;
        if (c >= total) {
          drained = true;
        } else {
          cell = a.order ? a.order[c] : c;
#pragma unroll
          for (int r = 0; r < M::NREACT; ++r) {
            const double k = a.rconst[(int64_t)r * a.rstride + cell];
            if (r < NL) own[(NG + NF + r) * 64] = k;
            else put(r - NL, k);
          }
#pragma unroll
          for (int s = 0; s < NF; ++s) own[(NG + s) * 64] = a.conc[(int64_t)(N + s) * a.cstride + cell];
          load();
          state_begin(a, cell, false, S);
          S.tries = 0;
        }
      }
      continue;
    }
    bool done = false;
    if (cell >= 0 && S.newStep) {
      // tail hand-off (see k_persist): T, H, the counters and Y to the list
      if (pa.ho.cap > 0 &&
          (P.direction > 0 ? (S.T - P.Tend) + P.roundoff <= 0.0 : (P.Tend - S.T) + P.roundoff <= 0.0) &&
          total - (int64_t)__hip_atomic_load(pa.ho.done, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT) <= pa.ho.cap) {
        const int64_t idx = (int64_t)atomicAdd(pa.ho.count, 1u);
        const int64_t cap = pa.ho.cap;
        if (idx < cap) {
          double *const r = pa.ho.rec + idx;
          r[0] = S.T;
          r[cap] = S.H;
          r[2 * cap] = S.Hexit;
          r[3 * cap] = S.Texit;
          r[4 * cap] = S.HnewAcc;
          for (int k = 0; k < 8; ++k) r[(5 + k) * cap] = (double)S.st[k];
          r[13 * cap] = (double)S.tries;
          r[14 * cap] = 0.0;
#pragma unroll
          for (int i = 0; i < N; ++i) r[(HO_FIELDS + i) * cap] = get(SY + i);
          pa.ho.cell[idx] = (int32_t)cell;
          atomicAdd(pa.ho.done, 1u);
          cell = -1;
        }
      }
      if (cell >= 0) done = state_done(P, S);
    }
    if (cell >= 0 && !done) {
      double D[N], K0[N], K1[N], K2[N], v[N];
      if (S.newStep) {
        S.st[0] += P.autonomous ? 1 : 2;
        S.st[1] += 1;
      }
      // Fcn0 (again in a rejected step's next attempt: the same value), the
      // matrix and its LU; H halved while a pivot is below TINY
      int nconsec = 0;
      bool singular = true;
      while (singular) {
        double y[N], b[M::NPART];
        reread();
#pragma unroll
        for (int i = 0; i < N; ++i) y[i] = get(SY + i);
        U::fun_partials(y, rate, fix, v, b);
        singular = U::lu(b, 1.0 / (P.direction * S.H * kRosGamma1), D, lds, put_lds);
        S.st[5] += 1;
        if (singular) {
          S.st[7] += 1;
          if (++nconsec <= 5) S.H *= 0.5;
          else break;
        }
      }
      if (singular) {
        S.ierr = -8;
        done = true;
      } else {
        const double dH = P.direction * S.H, c0 = 4.0 / dH, c1 = 1.0 / dH, c2 = -1.0 / dH,
                     c3 = -(8.0 / 3.0) / dH;
        // solves for K0..K3 (K3 in v); a loop, so that Fun and the substitutions
        // are inlined once.  Fcn0 waits in K1 for stage 1.
#pragma unroll
        for (int i = 0; i < N; ++i) {
          K1[i] = v[i];
          K0[i] = K2[i] = 0.0;
        }
#pragma unroll 1
        for (int s = 0; s < 4; ++s) {
          reread();
          if (s == 1) {
#pragma unroll
            for (int i = 0; i < N; ++i) v[i] = fma(c0, K0[i], K1[i]);
          } else if (s >= 2) {
            double y[N];
#pragma unroll
            for (int i = 0; i < N; ++i) {
              y[i] = fma(2.0, K0[i], get(SY + i));
              if (s == 3) y[i] = fma(1.0, K2[i], y[i]);
            }
            U::fun(y, rate, fix, v);
            S.st[0] += 1;
#pragma unroll
            for (int i = 0; i < N; ++i) {
              v[i] = fma(c2, K1[i], fma(c1, K0[i], v[i]));
              if (s == 3) v[i] = fma(c3, K2[i], v[i]);
            }
          }
          U::solve(D, lds, v);
          S.st[6] += 1;
#pragma unroll
          for (int i = 0; i < N; ++i) {
            if (s == 0) K0[i] = v[i];
            else if (s == 1) K1[i] = v[i];
            else if (s == 2) K2[i] = v[i];
          }
        }
        // Ynew into K0 and the error norm in species order
        double err = 0.0;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const double y0 = get(SY + i), y1 = fma(1.0, v[i], fma(1.0, K2[i], fma(2.0, K0[i], y0)));
          const double ye = fma(1.0, v[i], 0.0);
          K0[i] = y1;
          const double ymax = max_f(fabs(y0), fabs(y1));
          const int k = P.vectol ? i : 0;
          const double q = ye / (a.atol[k] + a.rtol[k] * ymax);
          err = fma(q, q, err);
        }
        err = max_f(sqrt(err / N), 1.0e-10);
        if (a.hlog && S.st[2] < a.hlog_n) {
          a.hlog[(int64_t)(2 * S.st[2]) * a.ncell + cell] = (float)S.H;
          a.hlog[(int64_t)(2 * S.st[2] + 1) * a.ncell + cell] = (float)err;
        }
        if (state_step(P, err, S)) {
#pragma unroll
          for (int i = 0; i < N; ++i) put(SY + i, P.clip_negative ? max_f(K0[i], 0.0) : K0[i]);
        }
      }
    }
    if (done) {
      if (S.ierr < 0 && a.retry && S.tries == 0) {
        load();
        state_begin(a, cell, true, S);
        S.tries = 1;
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const double c = get(SY + i);
          a.conc[(int64_t)i * a.cstride + cell] = a.clip_out ? (c > 0.0 ? c : 0.0) : c;
        }
        if (a.clip_out) {
#pragma unroll
          for (int s = 0; s < NF; ++s) {
            const double f = fix(s);
            a.conc[(int64_t)(N + s) * a.cstride + cell] = f > 0.0 ? f : 0.0;
          }
        }
        if (a.istatus)
#pragma unroll
          for (int k = 0; k < 20; ++k) a.istatus[(int64_t)k * a.sstride + cell] = k < 8 ? S.st[k < 8 ? k : 0] : 0;
        if (a.rstatus) {
          for (int k = 3; k < 20; ++k) a.rstatus[(int64_t)k * a.sstride + cell] = 0.0;
          a.rstatus[cell] = S.Texit;
          a.rstatus[a.sstride + cell] = S.Hexit;
          a.rstatus[2 * a.sstride + cell] = S.HnewAcc;
        }
        if (a.hnew) a.hnew[cell] = S.HnewAcc;
        if (a.ierr) a.ierr[cell] = S.ierr;
        if (pa.ho.cap > 0) atomicAdd(pa.ho.done, 1u);
        cell = -1;
      }
    }
  }
}

}  // namespace

const void *unrolled_kernel(int qset) {
  return qset == PQ_HG ? (const void *)k_lane_unrolled<Traits_Hg> : nullptr;
}

}  // namespace gckpp
