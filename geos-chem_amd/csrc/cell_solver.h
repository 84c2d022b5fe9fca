// The cell-per-wave Rodas3 attempt on cell programs (mechgen/cell_sched.py):
// one wavefront integrates one cell whose LU and solve vector live in LDS
// (fullchem: 53 KB, three cells per CU) and whose state, rate constants,
// stage vectors and the LU's tail block live in the lanes' registers.
//
// What bounds it: the LDS round trips of the levels in front of the tail block
// and the operand reads, two per FMA (about 2,100 LDS reads an attempt), with
// one wave per SIMD to hide them.  Hence straight-line programs (no flags, no
// loop control: 14.0k instructions, the operands of seven steps in flight), sums
// cut into 32-term chunks so that a 384-term row is not one lane's serial
// chain, the last 34 rows -- a chain of pivots -- in registers, and the
// reaction products in LDS over the tail block's slots (gathered from L2 they
// cost 64 cache lines a step), and the LU laid out in the order in which the
// substitutions read it, a step's lanes side by side (112 ms without).
// Measured on the 24x23x72 grid, cold step of 39,744 cells: 537 ms with the
// block programs of wave_sched.py, 101 ms here; 55 us an attempt and wave where
// it was 280 us; one cell's Integrate 9.1 ms and 2.2 ms.
//
// Included by wave_solver.hip inside namespace gckpp.
#pragma once

typedef __attribute__((address_space(3))) double lds_double;

// One wave's LDS block by byte offset; own: the block plus the lane's double.
struct CellLds {
  unsigned base, own, coef;
  int lane;
  __amdgpu_buffer_rsrc_t words;  // the programs' words
};
__device__ __forceinline__ double cell_ld(unsigned off) { return *(const lds_double *)off; }
__device__ __forceinline__ void cell_st(unsigned off, double v) { *(lds_double *)off = v; }

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
// Block k of the programs' words (four words a lane, 1 KB a block), through a
// buffer resource: the block's offset is a constant, so no load needs an
// address register (a base address for every four blocks had pushed the
// kernel's registers into scratch).
__device__ __forceinline__ u32x4 cell_word(const CellLds &c, int k) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                       c.words, c.lane * 16 + (k & 3) * 1024, (k >> 2) * 4096, 0));
}
// True on the lanes of a constant mask.  (The asm keeps the masks out of
// registers: hoisted from the attempt loop as constants, they spilled.)
template <unsigned LO, unsigned HI>
__device__ __forceinline__ bool lanes_of() {
  unsigned lo, hi;
  asm volatile("s_mov_b32 %0, %1" : "=s"(lo) : "i"(LO));
  asm volatile("s_mov_b32 %0, %1" : "=s"(hi) : "i"(HI));
  return __builtin_amdgcn_inverse_ballot_w64((uint64_t)hi << 32 | lo);
}
// x = fma(-t, s, x) on the lanes of a constant mask, s the same on every lane
// (the wave runs with all lanes on).  One FMA on the chain x -> s -> x; a
// select would put two more instructions there.
template <unsigned LO, unsigned HI>
__device__ __forceinline__ void fma_on(double &x, double t, double s) {
  asm volatile(
      "s_mov_b32 exec_lo, %3\n\ts_mov_b32 exec_hi, %4\n\tv_fma_f64 %0, -%1, %2, %0\n\t"
      "s_mov_b64 exec, -1"
      : "+v"(x)
      : "v"(t), "s"(s), "i"(LO), "i"(HI));
}
// Lane l's value on every lane.
__device__ __forceinline__ double bcast(double v, int l) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint64_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, l);
  const uint64_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l);
  return __builtin_bit_cast(double, hi << 32 | lo);
}
// x / d from y = 1 / d (correctly rounded): Markstein's two-step quotient
// (IBM J. Res. Dev. 34(1), 1990), the same double as x / d for finite
// operands away from underflow, in three dependent FMAs where the division
// sequence takes eleven instructions.
__device__ __forceinline__ double cell_div(double x, double d, double y) {
  const double q = x * y;
  return fma(fma(-d, q, x), y, q);
}

#define LD(off) cell_ld(c.base + (off))
#define ST(off, v) cell_st(c.base + (off), v)
#define CF(off) cell_ld(c.coef + (off))
#define LDL(off) cell_ld(c.own + (off))
#define STL(off, v) cell_st(c.own + (off), v)
#include "gen/cell_fullchem.h"

// The cell programs of a mechanism that has them (Traits::TAIL > 0).
template <class M> struct CellProg;
template <> struct CellProg<Traits_fullchem> {
  static constexpr int TAIL = cell_fullchem::TAIL, ROWS = cell_fullchem::ROWS;
  static constexpr int NCOEF = cell_fullchem::NCOEF, SIZE = cell_fullchem::SIZE;
  static constexpr int X0 = cell_fullchem::X0, CELLS = cell_fullchem::CELLS;
  static __device__ __forceinline__ void fun(const CellLds &c, const double (&R)[ROWS]) {
    cell_fullchem::cell_fun(c, R);
  }
  static __device__ __forceinline__ void jac(const CellLds &c, const double (&R)[ROWS], double diag,
                                             bool &bad) {
    cell_fullchem::cell_jac(c, R, diag, bad);
  }
  static __device__ __forceinline__ void lu(const CellLds &c, double (&T)[TAIL], double &ud,
                                            double &yd) {
    cell_fullchem::cell_lu(c, T, ud, yd);
  }
  static __device__ __forceinline__ void solve(const CellLds &c, const double (&T)[TAIL], double ud,
                                               double yd) {
    cell_fullchem::cell_solve(c, T, ud, yd);
  }
  // the same with no read of an LU position that is not the sum's own
  static __device__ __forceinline__ void solve_apart(const CellLds &c, const double (&T)[TAIL],
                                                     double ud, double yd) {
    cell_fullchem::cell_solve_apart(c, T, ud, yd);
  }
  static __device__ __forceinline__ __amdgpu_buffer_rsrc_t words() {
    return brsrc(cell_fullchem::words, (int)sizeof(cell_fullchem::words));
  }
  static __device__ int rx(int i) { return cell_fullchem::rx[i]; }
  static __device__ double coef(int i) { return cell_fullchem::coef[i]; }
  static __device__ __forceinline__ void constants(const CellLds &c) {
    if (c.lane == 0) {
      ST(8 * cell_fullchem::ZERO, 0.0);
      ST(8 * cell_fullchem::ONE, 1.0);
      ST(8 * cell_fullchem::NEG, -1.0);
    }
  }
};

// What a lane keeps of its wave's cell between attempts: the rate constants
// of its reactions, and of species lane + 64 k the concentration and Fcn0.
template <class M>
struct CellState {
  static constexpr int KS = (M::NVAR + 63) / 64;
  double R[CellProg<M>::ROWS], Y[KS], F0[KS];
};

// Fixed species and rate constants of the cell; Y is the
// caller's.
template <class M>
__device__ __forceinline__ void cell_load(const IntegrateArgs &a, const CellLds &c, int64_t cell,
                                          CellState<M> &s) {
  using P = CellProg<M>;
  wave_sync();
  P::constants(c);
  if (c.lane < M::NFIX)
    STL(8 * (P::X0 + M::NVAR), a.conc[(int64_t)(M::NVAR + c.lane) * a.cstride + cell]);
#pragma unroll
  for (int u = 0; u < P::ROWS; ++u)
    s.R[u] = a.rconst[(int64_t)P::rx(u * 64 + c.lane) * a.rstride + cell];
  wave_sync();
}

template <class M>
__device__ __forceinline__ void cell_begin(const IntegrateArgs &a, const CellLds &c, int64_t cell,
                                           CellState<M> &s) {
  cell_load<M>(a, c, cell, s);
#pragma unroll
  for (int k = 0; k < CellState<M>::KS; ++k) {
    const int i = c.lane + 64 * k < M::NVAR ? c.lane + 64 * k : M::NVAR - 1;
    s.Y[k] = a.conc[(int64_t)i * a.cstride + cell];
  }
}

// Continues a handed-off cell (see state_resume).
template <class M>
__device__ __forceinline__ void cell_resume(const IntegrateArgs &a, const Handoff &ho,
                                            const CellLds &c, int64_t cell, int64_t idx,
                                            CellState<M> &s) {
  cell_load<M>(a, c, cell, s);
#pragma unroll
  for (int k = 0; k < CellState<M>::KS; ++k) {
    const int i = c.lane + 64 * k < M::NVAR ? c.lane + 64 * k : M::NVAR - 1;
    s.Y[k] = ho.rec[(HO_FIELDS + i) * ho.cap + idx];
  }
}

template <class M>
__device__ __forceinline__ void cell_finish(const IntegrateArgs &a, const CellLds &c, int64_t cell,
                                            const CellState<M> &s) {
#pragma unroll
  for (int k = 0; k < CellState<M>::KS; ++k) {
    const int i = c.lane + 64 * k;
    const double v = a.clip_out ? (s.Y[k] > 0.0 ? s.Y[k] : 0.0) : s.Y[k];
    if (i < M::NVAR) a.conc[(int64_t)i * a.cstride + cell] = v;
  }
  if (a.clip_out && c.lane < M::NFIX) {
    const double v = LDL(8 * (CellProg<M>::X0 + M::NVAR));
    a.conc[(int64_t)(M::NVAR + c.lane) * a.cstride + cell] = v > 0.0 ? v : 0.0;
  }
}

// One Rodas3 attempt of the wave's cell (lane_attempt's algorithm and order
// of operations): CELL_DONE when the cell is done (S.ierr then holds IERR),
// CELL_AGAIN when it has to be made again with APART.  P::solve lets a lane
// whose terms have ended read another row's factor times 0, which an infinite
// factor turns into a NaN of a row that has nothing to do with it.  A stage
// vector's NaN reaches the error norm; so an attempt whose norm is NaN is made
// again with P::solve_apart, and a row is NaN only where its own terms make it
// so.  (As a second copy of the attempt: a branch around the solve costs every
// attempt 1 %, its first loads no longer start before it.)
enum { CELL_MORE = 0, CELL_DONE = 1, CELL_AGAIN = 2 };
template <class M, bool APART>
__device__ __forceinline__ int cell_attempt(const IntegrateArgs &a, const CellLds &c, int64_t cell,
                                            RosState &S, CellState<M> &cs) {
  using P = CellProg<M>;
  constexpr int N = M::NVAR, KS = CellState<M>::KS;
  const RosParams &prm = a.prm;
  const double dir = prm.direction;
  // the lane's species of a vector to X and back
  auto put = [&](const double (&v)[KS]) {
    wave_sync();
#pragma unroll
    for (int k = 0; k < KS; ++k)
      if (64 * (k + 1) <= N || c.lane + 64 * k < N) STL(8 * (P::X0 + 64 * k), v[k]);
    wave_sync();
  };
  auto get = [&](double (&v)[KS]) {
    wave_sync();
#pragma unroll
    for (int k = 0; k < KS; ++k)
      v[k] = 64 * (k + 1) <= N || c.lane + 64 * k < N ? LDL(8 * (P::X0 + 64 * k)) : 0.0;
    wave_sync();
  };
  if (!APART && S.newStep && state_done(prm, S)) return CELL_DONE;
  double K0[KS], K1[KS], K2[KS], K3[KS], T[P::TAIL], ud = 1.0, yd = 1.0, dH = 0.0;
#pragma unroll
  for (int k = 0; k < KS; ++k) K0[k] = K1[k] = K2[k] = K3[k] = 0.0;
#pragma unroll
  for (int k = 0; k < P::TAIL; ++k) T[k] = 0.0;
  // s = -1: Fcn0 of a new step; s = 0: the matrix and its LU; s = 0..3: the
  // stages.  A loop, so that the programs are inlined once.
#pragma unroll 1
  for (int s = !APART && S.newStep ? -1 : 0; s < 4; ++s) {
    double v[KS];
    if (s < 0 || s >= 2) {
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        v[k] = cs.Y[k];
        if (s >= 2) v[k] = fma(2.0, K0[k], v[k]);
        if (s == 3) v[k] = fma(1.0, K2[k], v[k]);
      }
      put(v);
      P::fun(c, cs.R);
      get(v);
      S.st[0] += s >= 0 || prm.autonomous ? 1 : 2;
      if (s < 0) {
        S.st[1] += 1;
#pragma unroll
        for (int k = 0; k < KS; ++k) cs.F0[k] = v[k];
        continue;
      }
    } else {
      if (s == 0) {
        int nconsec = 0;
        bool singular = true;
        while (singular) {
          put(cs.Y);
          bool bad = false;
          P::jac(c, cs.R, 1.0 / (dir * S.H * kRosGamma1), bad);
          const bool ising = __ballot(bad) != 0;
          if (!ising) P::lu(c, T, ud, yd);
          S.st[5] += 1;
          if (!ising) {
            singular = false;
          } else {
            S.st[7] += 1;
            ++nconsec;
            if (nconsec <= 5) S.H *= 0.5;
            else break;
          }
        }
        if (singular) { S.ierr = -8; return CELL_DONE; }
        dH = dir * S.H;
      }
#pragma unroll
      for (int k = 0; k < KS; ++k) v[k] = cs.F0[k];
    }
    if (s > 0) {
      const double c0 = (s == 1 ? 4.0 : 1.0) / dH, c1 = -1.0 / dH, c2 = -(8.0 / 3.0) / dH;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        v[k] = fma(c0, K0[k], v[k]);
        if (s >= 2) v[k] = fma(c1, K1[k], v[k]);
        if (s == 3) v[k] = fma(c2, K2[k], v[k]);
      }
    }
    put(v);
    if constexpr (APART) P::solve_apart(c, T, ud, yd);
    else P::solve(c, T, ud, yd);
    get(v);
    S.st[6] += 1;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      if (s == 0) K0[k] = v[k];
      else if (s == 1) K1[k] = v[k];
      else if (s == 2) K2[k] = v[k];
      else K3[k] = v[k];
    }
  }
  const double H = S.H;
  // Ynew and the error norm: a lane's terms in species order, then the 64
  // lanes' sums in lane order
  double yn[KS], at[KS], rt[KS], part = 0.0;
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    const int i = prm.vectol ? (c.lane + 64 * k < N ? c.lane + 64 * k : N - 1) : 0;
    at[k] = a.atol[i];
    rt[k] = a.rtol[i];
  }
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    yn[k] = fma(1.0, K3[k], fma(1.0, K2[k], fma(2.0, K0[k], cs.Y[k])));
    const double ye = fma(1.0, K3[k], 0.0);
    const double ymax = max_f(fabs(cs.Y[k]), fabs(yn[k]));
    const double q = ye / (at[k] + rt[k] * ymax);
    if (64 * (k + 1) <= N || c.lane + 64 * k < N) part = fma(q, q, part);
  }
  wave_sync();
  STL(8 * P::X0, part);
  wave_sync();
  double err = 0.0;
#pragma unroll 1
  for (int l = 0; l < 64; l += 16) {
    double q[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) q[u] = LD(8 * (P::X0 + l + u));
#pragma unroll
    for (int u = 0; u < 16; ++u) err += q[u];
  }
  if (!APART && __any(err != err)) {
    S.st[0] -= 2;  // (counted again: the stages' Fun, the LU, the substitutions)
    S.st[5] -= 1;
    S.st[6] -= 4;
    return CELL_AGAIN;
  }
  err = max_f(sqrt(err / N), 1.0e-10);
  if (a.hlog && S.st[2] < a.hlog_n && c.lane == 0) {
    a.hlog[(int64_t)(2 * S.st[2]) * a.ncell + cell] = (float)H;
    a.hlog[(int64_t)(2 * S.st[2] + 1) * a.ncell + cell] = (float)err;
  }
  if (state_step(prm, err, S)) {
#pragma unroll
    for (int k = 0; k < KS; ++k) cs.Y[k] = prm.clip_negative ? max_f(yn[k], 0.0) : yn[k];
  }
  return CELL_MORE;
}

#undef LD
#undef ST
#undef CF
#undef LDL
#undef STL
