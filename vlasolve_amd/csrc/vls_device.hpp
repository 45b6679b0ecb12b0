// Device helpers shared by the kernels of the forward step.
#pragma once
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include "vls_internal.hpp"

namespace vls {

// Slices per chunk of the moment's sum over j, and head rows of the pivot
// tables (past them the pivots are at their fixed point).
constexpr int kJC = 20, kHead = 16;
// Rows of a segment of the streaming line solves (vls_stream.hip).
constexpr int kSegRows = 16;

__device__ __forceinline__ double BV2(double x) { return x * x * x; }
__device__ __forceinline__ double BV1(double x) {
  return 1.0 + 3.0 * x + 3.0 * x * x - 3.0 * x * x * x;
}

// modf for the finite, non-negative coordinates used here: integer part by
// truncation, exact fractional remainder (localSpline::pos2Coord,
// src/localSpline.hxx:352-358).
__device__ __forceinline__ void split(double x, int &n, double &t) {
  double ip = trunc(x);
  t = x - ip;
  n = (int)ip;
}

__device__ __forceinline__ double lane_next(double x) {  // lane i gets lane i+1's x
  int lo = __double2loint(x), hi = __double2hiint(x);
  lo = __builtin_amdgcn_mov_dpp(lo, 0x130 /* wave_shl:1 */, 0xf, 0xf, true);
  hi = __builtin_amdgcn_mov_dpp(hi, 0x130, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

struct MomentArgs {
  const double *Ct1, *dU, *dR, *gfac;
  double *P, *dM, *Mx, *acc, *mTot;
  unsigned *cnt;
};

// The kick's value of a point from the four column-spline coefficients of
// its target rows n..n+3 and its offset y in the cell (evaluateNxPy,
// src/localSpline.hxx:423-441, in the column form)
__device__ __forceinline__ double kick_value(double y, double d0, double d1, double d2, double d3) {
  double result = 1.0 / 6.0;
  result *= BV2(1. - y) * d0 + BV1(1. - y) * d1 + BV1(y) * d2 + BV2(y) * d3;
  return result;
}

// the head rows of an axis's pivot table (u, RN(1/d) and its remainder)
struct HeadTab {
  double u[kHead + 1], rd[kHead + 1], rl[kHead + 1];
};

// localSpline::evaluateC(Nx,x,Ny,y), src/localSpline.hxx:381-398
__device__ __forceinline__ double eval_c(const double *d, int64_t st, double xr, double xu) {
  int Nx, Ny;
  double x, y;
  split(xr, Nx, x);
  split(xu, Ny, y);
  Nx++;
  Ny++;
  const double *p0 = d + Nx + (int64_t)(Ny - 1) * st;
  const double *p1 = p0 + st;
  const double *p2 = p1 + st;
  const double *p3 = p2 + st;
  const double b2xI = BV2(1. - x);
  const double b1xI = BV1(1. - x);
  const double b2x = BV2(x);
  const double b1x = BV1(x);
  double result = 1.0 / 36.0;
  result *= BV2(1. - y) * (p0[-1] * b2xI + p0[0] * b1xI + p0[1] * b1x + p0[2] * b2x) +
            BV1(1. - y) * (p1[-1] * b2xI + p1[0] * b1xI + p1[1] * b1x + p1[2] * b2x) +
            BV1(y) * (p2[-1] * b2xI + p2[0] * b1xI + p2[1] * b1x + p2[2] * b2x) +
            BV2(y) * (p3[-1] * b2xI + p3[0] * b1xI + p3[1] * b1x + p3[2] * b2x);
  return result;
}

// eval_c in two parts, so that several points' loads can leave together:
// the 4x4 coefficients and the offsets in the cell, then the same sum in the
// same order as eval_c.
struct CStencil {
  double v[16];  // rows Ny-1..Ny+2, columns Nx-1..Nx+2 (v[4 a + b])
  double x, y;
};
__device__ __forceinline__ void eval_c_fetch(const double *d, int64_t st, double xr, double xu,
                                             CStencil &s) {
  int Nx, Ny;
  split(xr, Nx, s.x);
  split(xu, Ny, s.y);
  Nx++;
  Ny++;
  const double *p0 = d + Nx + (int64_t)(Ny - 1) * st;
#pragma unroll
  for (int a = 0; a < 4; a++)
#pragma unroll
    for (int b = 0; b < 4; b++) s.v[4 * a + b] = p0[(int64_t)a * st + b - 1];
}
__device__ __forceinline__ double eval_c_sum(const CStencil &s) {
  const double x = s.x, y = s.y;
  const double *v = s.v;
  const double b2xI = BV2(1. - x);
  const double b1xI = BV1(1. - x);
  const double b2x = BV2(x);
  const double b1x = BV1(x);
  double result = 1.0 / 36.0;
  result *= BV2(1. - y) * (v[0] * b2xI + v[1] * b1xI + v[2] * b1x + v[3] * b2x) +
            BV1(1. - y) * (v[4] * b2xI + v[5] * b1xI + v[6] * b1x + v[7] * b2x) +
            BV1(y) * (v[8] * b2xI + v[9] * b1xI + v[10] * b1x + v[11] * b2x) +
            BV2(y) * (v[12] * b2xI + v[13] * b1xI + v[14] * b1x + v[15] * b2x);
  return result;
}

// the kinds of a point that the foot table holds in place of a foot's xr
constexpr double kFootOut = -1.0, kFootChain = -2.0;

struct ChainTables {
  const int64_t *off;
  const int32_t *len;
  int32_t *head;
  const double *bxr, *bxu;
  const uint8_t *bout;
  double *vals;  // the values of the species being drifted
  int64_t n;
  int roll;      // turn the rings (the last species of the step)
};

}  // namespace vls
