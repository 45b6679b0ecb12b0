// A step in two launches for grids whose padded slice of coefficients fits in
// the LDS of a CU (gfx950, FP64).
//
// Everything of a step but the moment is local to a slice (fixed j), and the
// kick to a column (fixed j, r).  With a kernel per phase a small grid spends
// its step on launches and on the first loads of each kernel, with a few lines
// per CU in flight.  Here
//   k_kick_tile    takes a tile of a slice's columns through the column
//                  splines and the kick in LDS; meanwhile each block sums the
//                  moment partials of all slices for itself (they come from
//                  L2) into the acceleration, so that no launch and no block
//                  waits for the reduction;
//   k_slice_drift  takes a slice through the r- and v-solves in LDS, then
//                  drifts its points and forms the slice's moment partials of
//                  the new f.  Where the slices are fewer than the CUs several
//                  blocks share a slice: each solves it for itself (the CUs
//                  would idle) and drifts a part of its rows.
// What bounds both: the serial chains of the solves (a lane per line: at
// 129x129x64 5.5 us each of three) and the first loads (3 and 5 us); then the
// drift's points (8 evaluations a wave and block, 0.3 us each) and the way of
// the group sums to the partials (4 us).  The operations and their order are
// those of the kernels per phase (vls_kernels.hip): same bits.  Against those,
// a step of 65x65x32 takes 26 us for 32, 91x81x80 36 for 92, 181x81x80 50 for
// 122, 129x129x64 47 for 60 and 69 for 100 without linking, two species of
// 97x97x48 82 for 150.  One launch for the whole step, a block per slice, was
// 29 us at 65x65x32 but 69 at 129x129x64: its evaluations had 64 of the CUs.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <set>

#include "vls_device.hpp"
#include "vls_div.hpp"
#include "vls_internal.hpp"
#include "vls_tile.hpp"

namespace vls {

namespace {

constexpr int kMaxLds = 163840;  // LDS of one, all of which a block may take

// i / d == __umulhi(i, magic(d)) for i d < 2^32
inline unsigned magic(int d) { return (unsigned)(((1ull << 32) + d - 1) / d); }

// The pivots of the natural spline solve, rows 1..kHead and (last) all later
// ones: super-diagonal u, RN(1/d) and its remainder.  They are the same for
// every grid (the first row is c_0 - 2 c_1 + c_2 = 0 whatever the spacing);
// literals cost a row nothing, where an LDS table is read behind the row
// before's write (its address could be the table's): 250 cycles a head row.
// The set-up compares them with the run's table (slice_pivots).
constexpr double kPivU[kHead + 2] = {0.0, 0x0.0p+0, 0x1.0000000000000p-2, 0x1.1111111111111p-2,
    0x1.1249249249249p-2, 0x1.125f8a6956f76p-2, 0x1.1261261261262p-2, 0x1.126143a0aba9dp-2,
    0x1.126145bfe7dedp-2, 0x1.126145e6e884bp-2, 0x1.126145e9b5624p-2, 0x1.126145e9e8da4p-2,
    0x1.126145e9ec8c4p-2, 0x1.126145e9ecd02p-2, 0x1.126145e9ecd50p-2, 0x1.126145e9ecd56p-2,
    0x1.126145e9ecd57p-2, 0x1.126145e9ecd57p-2};
constexpr double kPivRd[kHead + 2] = {0.0, 0x1.0000000000000p+0, 0x1.8000000000000p+0,
    0x1.999999999999ap+0, 0x1.9b6db6db6db6ep+0, 0x1.9b8f4f9e02732p+0, 0x1.9b91b91b91b93p+0,
    0x1.9b91e571017ebp+0, 0x1.9b91e89fdbce4p+0, 0x1.9b91e8da5cc71p+0, 0x1.9b91e8de90137p+0,
    0x1.9b91e8dedd476p+0, 0x1.9b91e8dee2d26p+0, 0x1.9b91e8dee3384p+0, 0x1.9b91e8dee33f8p+0,
    0x1.9b91e8dee3401p+0, 0x1.9b91e8dee3402p+0, 0x1.9b91e8dee3402p+0};
constexpr double kPivRl[kHead + 2] = {0.0, 0x0.0p+0, 0x1.8000000000000p-54,
    -0x1.999999999999ap-54, -0x1.9a1f58d0fac68p-54, 0x1.8d66824e61708p-56, -0x1.2679ca12c88eep-54,
    0x1.e50bd0f2693f2p-54, 0x1.e146a6c0ff79cp-54, -0x1.d42b2b514981bp-54, 0x1.fa760ee70d1c5p-57,
    0x1.85c55fb87d6e8p-55, 0x1.aa34d354ae79bp-57, -0x1.38360a9a30f98p-54, 0x1.80e9a827b6badp-60,
    0x1.ac2a59571744bp-57, 0x1.60e0f4f57eecap-54, 0x1.60e0f4f57eecap-54};
constexpr double kC16 = 1.0 / 6.0;

// The constants of an axis's last row.
struct LineTab {
  double hi2, p, q, rq;
};
__device__ __forceinline__ void line_tab(LineTab *l, const ThomasAxis &ax) {
  l->hi2 = ax.hi2, l->p = ax.p, l->q = ax.q, l->rq = ax.rq;
}
// The natural spline solve of a line in LDS, in place (thomas_forward and
// thomas_backward of the kernels per phase): p[k st] holds the right-hand
// side of row k = 1..L and receives the L + 2 coefficients.  The rows go by
// in chunks of kPF whose reads are issued a chunk ahead.  The forward values
// of the head and of the last rows (whole chunks, kNY rows at most) wait in
// registers for the way down, the others in place.  A row takes about 36
// cycles up and 34 down in registers (a chain of 4 and 2 dependent FP64
// operations of 5 cycles, a DS read of 15 or a write of 20), 60 and 50 in
// place.
constexpr int kPF = 8, kNY = 80;
static_assert(kHead == 2 * kPF, "the head is two chunks");

__device__ __forceinline__ void lds_line(double *p, int st, int L, const LineTab &ax) {
  // uniform, and unknown before this point: what is formed from them would
  // otherwise be kept in scalar registers across the kernel's loops (and
  // spilled to vector lanes)
  st = __builtin_amdgcn_readfirstlane(st);
  L = __builtin_amdgcn_readfirstlane(L);
  asm volatile("" : "+s"(st), "+s"(L));
  const double hi2 = ax.hi2, last1 = ax.p, lastQ = ax.q, lastRq = ax.rq;
  const double rdS = kPivRd[kHead + 1], rlS = kPivRl[kHead + 1], uS = kPivU[kHead + 1];
  double prev = 0.0, prev2 = 0.0;     // y_k, y_{k-1} of the last row done (y_0 = 0)
  double *lp = p + st, *sp = p + st;  // next row to read, next to write
  auto up = [&](double rhs, double rd, double rl) {
    const double y = div_pivot(rhs - kC16 * prev, rd, rl);
    prev2 = prev;
    prev = y;
    return y;
  };
  auto put = [&](double y, int step) {
    *sp = y;
    sp += step;
  };
  auto load = [&](double (&v)[kPF], int step) {  // kPF rows in the direction of step
#pragma unroll
    for (int q = 0; q < kPF; q++) {
      v[q] = *lp;
      lp += step;
    }
  };
  double yh[kHead], y[kNY];
  // chunks in registers, and rows between the head and them
  int nc = L > kHead ? min((L - kHead) / kPF, kNY / kPF) : 0;
  const int nl = L - kHead - nc * kPF;
  if (nc == 0) {
    // short lines: the head's rows that exist, then fewer than kPF others
#pragma unroll
    for (int k = 1; k <= kHead; k++)
      if (k <= L) yh[k - 1] = up(p[k * st], kPivRd[k], kPivRl[k]);
#pragma unroll
    for (int k = 0; k < kPF - 1; k++)
      if (k < nl) y[k] = up(p[(kHead + 1 + k) * st], rdS, rlS);
    sp = p + (L + 1) * st;
  } else {
    double a[kPF], b[kPF];
    load(a, st);
    load(b, st);
#pragma unroll
    for (int q = 0; q < kPF; q++) yh[q] = up(a[q], kPivRd[1 + q], kPivRl[1 + q]);
    load(a, st);
#pragma unroll
    for (int q = 0; q < kPF; q++)
      yh[kPF + q] = up(b[q], kPivRd[1 + kPF + q], kPivRl[1 + kPF + q]);
    // a: the next kPF rows (there are that many: nc >= 1); whole chunks in
    // place, then the rest of them
    sp += kHead * st;
    int k = nl;
#pragma unroll 1
    for (; k >= kPF; k -= kPF) {
#pragma unroll
      for (int q = 0; q < kPF; q++) b[q] = a[q];
      load(a, st);
#pragma unroll
      for (int q = 0; q < kPF; q++) put(up(b[q], rdS, rlS), st);
    }
    if (k > 0) {
#pragma unroll
      for (int q = 0; q < kPF - 1; q++)
        if (q < k) put(up(a[q], rdS, rlS), st);
      lp = sp;
      load(a, st);
    }
#pragma unroll
    for (int c = 0; c < kNY / kPF; c++) {
      if (c < nc) {
        if (c + 1 < nc) load(b, st);
#pragma unroll
        for (int q = 0; q < kPF; q++) y[c * kPF + q] = up(a[q], rdS, rlS);
#pragma unroll
        for (int q = 0; q < kPF; q++) a[q] = b[q];
      }
    }
    sp += nc * kPF * st;
  }
  double tt = 0.0 - hi2 * prev2;
  tt = tt - last1 * prev;
  double cn = div_known(tt, lastQ, lastRq), c2 = cn;
  put(cn, -st);  // row L + 1
  auto down = [&](double yk, double u) {
    const double c = yk - u * cn;
    put(c, -st);
    c2 = cn;
    cn = c;
  };
  if (nc == 0) {
#pragma unroll
    for (int k = kPF - 2; k >= 0; k--)
      if (k < nl) down(y[k], uS);
#pragma unroll
    for (int k = kHead; k >= 1; k--)
      if (k <= L) down(yh[k - 1], kPivU[k]);
  } else {
    asm volatile("" : "+s"(nc));  // compared again on the way down
    double a[kPF], b[kPF];
    // the rows in place after the registers'
    lp = p + (nl + kHead) * st;
    int k = nl;
    const int rest = k % kPF;
#pragma unroll
    for (int q = 0; q < kPF - 1; q++) b[q] = lp[-min(q, rest) * st];
#pragma unroll
    for (int c = kNY / kPF - 1; c >= 0; c--) {
      if (c < nc) {
#pragma unroll
        for (int q = kPF - 1; q >= 0; q--) down(y[c * kPF + q], uS);
      }
    }
    lp -= rest * st;
    load(a, -st);  // (the head's rows if no whole chunk is left: not used)
#pragma unroll
    for (int q = 0; q < kPF - 1; q++)
      if (q < rest) down(b[q], uS);
    k -= rest;
#pragma unroll 1
    for (; k >= kPF; k -= kPF) {
#pragma unroll
      for (int q = 0; q < kPF; q++) b[q] = a[q];
      load(a, -st);
#pragma unroll
      for (int q = 0; q < kPF; q++) down(b[q], uS);
    }
#pragma unroll
    for (int q = kHead - 1; q >= 0; q--) down(yh[q], kPivU[q + 1]);
  }
  // c_0 = (A03 - A01 c_1) - A02 c_2 with A03 = 0, A01 = -2, A02 = 1
  *sp = (0.0 - -2.0 * cn) - 1.0 * c2;
}

// ---------------------------------------------------------------- kick
struct KickArgs {
  const double *src;   // f [nS][nJ][nU][nR]
  double *dst;         // the kicked f (may be src)
  const double *P;     // moment partials [nJ][nR] of f (null: acc holds the acceleration)
  double *dKeep;       // the column splines [j][m][r], slice stride cs (null: not kept)
  const double *gfac, *U_Val;
  double *dM, *Mx, *acc, *mTot;
  int32_t *head;       // the delay lines' heads, advanced by roll (null: none)
  const int32_t *len;
  int64_t nChains, nVal, cs;
  double Ulo, Uhi, start_v, hinv_v;
  ThomasAxis tv;
  int nR, nU, nJ, nS;
  int W, nT;           // columns of a tile, tiles of a slice
  unsigned mulW, mulR;  // i / W == __umulhi(i, mulW), i / nR == __umulhi(i, mulR)
  int roll;
};

// kTK threads: one wave solves, the others sum the moment.  512 where every
// block has a CU for itself (twice the waves in the evaluation), else 256 (two
// blocks on a CU, two solves side by side).

inline size_t kick_lds(int nR, int nU, int nJ, int W, bool sums) {
  const size_t nC = sums ? (nJ + kJC - 1) / kJC : 0;
  return ((size_t)W * (nU + 3) + nU + nR + nC * nR + 1) * sizeof(double) + sizeof(LineTab);
}

// The acceleration in LDS by one wave: dM[r] from the chunk sums Sc [nC][nR],
// the serial prefix, times the factors that accs holds (out: with the global
// outputs).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ void wave_accel(double *Sc, double *accs, int nC, int nR, int lane,
                                           bool out, const KickArgs &a) {
  for (int r = lane; r < nR; r += 64) {
    double m = 0.0;
    for (int c = 0; c < nC; c++) m += Sc[c * nR + r];
    Sc[r] = m;
    if (out) a.dM[r] = m;
  }
  wave_sync();
  if (lane == 0) {
    // 16 entries a batch
    double prev = 0.0;
    int r = 0;
#pragma unroll 1
    for (; r + 16 <= nR; r += 16) {
      double x[16];
#pragma unroll
      for (int k = 0; k < 16; k++) x[k] = Sc[r + k];
#pragma unroll
      for (int k = 0; k < 16; k++) {
        const double y = x[k];
        x[k] = prev;
        prev += y;
      }
#pragma unroll
      for (int k = 0; k < 16; k++) Sc[r + k] = x[k];
    }
#pragma unroll 1
    for (; r < nR; r++) {
      const double y = Sc[r];
      Sc[r] = prev;
      prev += y;
    }
    if (out) *a.mTot = prev;
  }
  wave_sync();
  for (int r = lane; r < nR; r += 64) {
    const double m = Sc[r], x = m * accs[r];
    accs[r] = x;
    if (out) {
      a.Mx[r] = m;
      a.acc[r] = x;
    }
  }
}

template <int kTK>
__global__ void __launch_bounds__(kTK) k_kick_tile(KickArgs a) {
  extern __shared__ double lds[];
  const int nR = a.nR, nU = a.nU, nJ = a.nJ, W = a.W;
  const int nC = a.P ? (nJ + kJC - 1) / kJC : 0;
  double *D = lds, *Us = D + W * (nU + 3), *accs = Us + nU;
  double *Sc = accs + nR;
  LineTab *hv = (LineTab *)(Sc + nC * nR);
  unsigned *ready = (unsigned *)(hv + 1);  // waves whose chunk sums are in Sc
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int j = tile / a.nT, c0 = (tile - j * a.nT) * W;
  const int wid = min(W, nR - c0);  // columns of this tile

  if (a.head)
    for (int64_t k = (int64_t)blockIdx.x * kTK + t; k < a.nChains; k += (int64_t)gridDim.x * kTK) {
      const int h = a.head[k] + a.roll, len = a.len[k];
      a.head[k] = h >= len ? h - len : h;
    }
  if (t == 0) {
    line_tab(hv, a.tv);
    *ready = 0;
  }
  for (int u = t; u < nU; u += kTK) Us[u] = a.U_Val[u];
  for (int r = t; r < nR; r += kTK) accs[r] = a.P ? a.gfac[r] : a.acc[r];
  for (int i = t; i < W; i += kTK) D[(nU + 2) * W + i] = 0.0;  // read with weight 0

  for (int s = 0; s < a.nS; s++) {
    const size_t at = (size_t)s * a.nVal + (size_t)j * nU * nR + c0;
    const double *fj = a.src + at;
    double *fo = a.dst + at;
    // the tile's columns, 16 values of each thread in flight
    constexpr int kB = 16;
    const int n = nU * W;
#pragma unroll 1
    for (int b = t; b < n; b += kB * kTK) {
      double v[kB];
#pragma unroll
      for (int q = 0; q < kB; q++) {
        const int i = min(b + q * kTK, n - 1);
        const int u = __umulhi((unsigned)i, a.mulW), c = i - u * W;
        v[q] = fj[(size_t)u * nR + min(c, wid - 1)];
      }
#pragma unroll
      for (int q = 0; q < kB; q++)
        if (b + q * kTK < n) D[W + b + q * kTK] = v[q];
    }
    __syncthreads();
    if (w == 0) {
      if (lane < W) lds_line(D + lane, W, nU, *hv);
    } else if (a.P && s == 0) {
      // chunk sums of the partials (k_moment_chunks), a thread per (chunk, r)
#pragma unroll 1
      for (int i = t - 64; i < nC * nR; i += kTK - 64) {
        const int c = __umulhi((unsigned)i, a.mulR), r = i - c * nR, jb = c * kJC;
        const int je = min(nJ, jb + kJC);
        double x[kJC];
#pragma unroll
        for (int k = 0; k < kJC; k++) x[k] = a.P[(size_t)min(jb + k, nJ - 1) * nR + r];
        double sum = 0.0;
#pragma unroll
        for (int k = 0; k < kJC; k++)
          if (jb + k < je) sum += x[k];
        Sc[i] = sum;
      }
      // the last wave goes on to the acceleration once the others' chunk sums
      // are in (they run beside it: the wait ends), while wave 0 still solves
      constexpr int kOthers = kTK / 64 - 2;
      if (w < kTK / 64 - 1) {
        wave_sync();
        if (lane == 0)
          __hip_atomic_fetch_add(ready, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
      } else {
        while (__hip_atomic_load(ready, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < kOthers)
          __builtin_amdgcn_s_sleep(1);
        wave_sync();
        wave_accel(Sc, accs, nC, nR, lane, tile == 0, a);
      }
    }
    __syncthreads();
    // the kick's evaluation (k_kick_cols)
    if (a.dKeep) {
      double *dk = a.dKeep + (size_t)j * a.cs + c0;
      const int nk = (nU + 2) * W;
      for (int i = t; i < nk; i += kTK) {
        const int m = __umulhi((unsigned)i, a.mulW), c = i - m * W;
        if (c < wid) dk[(size_t)m * nR + c] = D[i];
      }
    }
    // four points' reads together, then their sums
    constexpr int kE = 4;
#pragma unroll 1
    for (int b = t; b < n; b += kE * kTK) {
      double d[kE][4], yy[kE];
      bool in[kE];
      int o[kE];
#pragma unroll
      for (int q = 0; q < kE; q++) {
        const int i = min(b + q * kTK, n - 1);
        const int u = __umulhi((unsigned)i, a.mulW), c = i - __umul24(u, W);
        const double newU = Us[u] + accs[min(c0 + c, nR - 1)];
        in[q] = !(newU <= a.Ulo) && !(newU >= a.Uhi);
        double y = in[q] ? (newU - a.start_v) * a.hinv_v : 0.0;
        int m;
        split(y, m, y);
        yy[q] = y;
        // row m + 3 is past the column only at y == 0, with weight 0 (zeroed)
        const double *p = D + __umul24(m, W) + c;
#pragma unroll
        for (int k = 0; k < 4; k++) d[q][k] = p[k * W];
        o[q] = c < wid && b + q * kTK < n ? (int)(__umul24(u, nR) + c) : -1;
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < kE; q++) {
        const double x = kick_value(yy[q], d[q][0], d[q][1], d[q][2], d[q][3]);
        if (o[q] >= 0) fo[o[q]] = in[q] ? x : 0.0;
      }
    }
    if (s + 1 < a.nS) __syncthreads();
  }
}

// ---------------------------------------------------------------- drift
struct SliceArgs {
  const double *src;  // the values to drift [nS][nJ][nU][nR]
  double *f;      // the drifted ones (src itself with one block per slice: the blocks of a
                  // slice all read all of it)
  double *P;      // moment partials [nJ][nR] of the new f (null: none)
  double *G;      // [nJ][nG][nR] group sums where several blocks share a slice
  unsigned *cnt;  // [nJ] counters of those blocks (zero between launches)
  double *cOut;   // the drift's coefficients of the last species (null: not kept)
  const double *Ct1, *dU, *dR;
  const double2 *feet;
  ChainTables ch;                       // vals: the first species' plane; roll not used
  const int64_t *chPoint;               // the delay lines' points
  const int32_t *chOrder, *chStart;     // the delay lines by slice: chOrder[chStart[j]..]
  int64_t nVal, nCells, cs;
  ThomasAxis tr, tv;
  int nR, nU, nJ, nS;
  unsigned mulR;   // i / nR == __umulhi(i, mulR) for the slice's point indices
  int hOff;        // ring position of this drift relative to the heads: 0 or -1
  int parts;       // blocks per slice
  int gPart;       // groups of 16 rows of a block
  int maxLines;    // delay lines of a slice, at most
  int loose;       // some delay-line points have no line
};

// Threads: 8 waves, 2 on each SIMD, with 256 VGPRs each, so that a line keeps
// 96 rows in registers.
constexpr int kT = 512;

// LDS of k_slice_drift: the coefficients (rows of odd pitch, one row more than
// the padded slice for stencils on the last knot), dU, the row after the
// block's rows, the axes' constants and the slice's delay lines.
__host__ __device__ inline int slice_pitch(int nR) { return (nR + 2) | 1; }
__host__ __device__ inline int slice_coef(int nR, int nU) { return slice_pitch(nR) * (nU + 3) + 8; }
struct LineRec;
size_t slice_lds(int nR, int nU, int maxLines);

// The thread's index as a value the compiler cannot connect with its other
// uses (each phase then forms its addresses for itself instead of keeping them
// in registers from the phase before).
__device__ __forceinline__ int fresh(int t) {
  asm volatile("" : "+v"(t));
  return t;
}

// Stores and loads between blocks of a launch: through memory (system scope),
// acknowledged before the count that tells of them (as moment_tail).
__device__ __forceinline__ void coherent_store(double *p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ double coherent_load(const double *p) {
  return __hip_atomic_load(const_cast<double *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void wait_stores() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// The moment's group sums of slice j over the groups [g0, g1) of 16 rows, in
// the order of moment_cols_block and k_moment_partial_sp: a wave takes a group
// (its 16 rows and the row after them) of 63 columns.  Row uH comes from halo
// (LDS; the block that owns it may not have written it).  put(g, r, sum).
template <class PUT>
__device__ __forceinline__ void group_sums(const SliceArgs &a, int j, int g0, int g1,
                                           const double *dUs, const double *halo, int uH, PUT put) {
  const int nR = a.nR, nU = a.nU;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nX = (nR + 62) / 63;
  const double ct = a.Ct1[j];
  const double *fj = a.f + (size_t)j * nU * nR;
  for (int task = w; task < (g1 - g0) * nX; task += kT / 64) {
    const int gi = task / nX, g = g0 + gi, x = task - gi * nX;
    const int u0 = 16 * g, r = x * 63 + lane, rc = min(r, nR - 1);
    const bool term = lane < 63 && r < nR - 1;
    const double *col = fj + rc;
    const double dr = term ? a.dR[r] : 0.0;
    double s = 0.0;
    if (a.nS == 1) {
      double row[17];
#pragma unroll
      for (int q = 0; q < 17; q++) row[q] = col[(size_t)min(u0 + q, nU - 1) * nR];
      if (u0 + 16 == uH) row[16] = halo[rc];
      double own = row[0], next = lane_next(own);
#pragma unroll
      for (int q = 0; q < 16; q++) {
        const double b = row[q + 1], bN = lane_next(b);
        if (u0 + q < nU - 1) {
          const double sum4 = ((own + next) + b) + bN;
          s += (((ct * dUs[u0 + q]) * 0.25) * dr) * sum4;
        }
        own = b;
        next = bN;
      }
    } else {
      // a few rows at a time: every species' values of a cell meet in its
      // average (one block per slice: no halo)
      for (int q0 = 0; q0 < 16; q0 += 4) {
        double avg[4] = {0.0, 0.0, 0.0, 0.0};
        for (int k = 0; k < a.nS; k++) {
          double row[5];
#pragma unroll
          for (int q = 0; q < 5; q++)
            row[q] = col[(size_t)k * a.nVal + (size_t)min(u0 + q0 + q, nU - 1) * nR];
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const double own = row[q], b = row[q + 1];
            avg[q] += (((own + lane_next(own)) + b) + lane_next(b)) * 0.25;
          }
        }
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (u0 + q0 + q < nU - 1) s += ((ct * dUs[u0 + q0 + q]) * dr) * avg[q];
      }
    }
    if (lane < 63 && r < nR) put(g, r, s);
  }
}

// P[j][r] from the group sums get(g, r): ((G0 + G1) + G2) + G3 per block of 64
// rows, the blocks left to right.
template <class GET>
__device__ __forceinline__ void group_combine(const SliceArgs &a, int j, GET get) {
  const int nR = a.nR, nU = a.nU, nG = (nU - 1 + 15) / 16, nW = (nU + 63) / 64;
  for (int r = threadIdx.x; r < nR; r += kT) {
    double Pj = 0.0;
    for (int b = 0; b < nW; b++) {
      double v[4];
#pragma unroll
      for (int q = 0; q < 4; q++) v[q] = 4 * b + q < nG ? get(4 * b + q, r) : 0.0;
      const double W = ((v[0] + v[1]) + v[2]) + v[3];
      Pj = b == 0 ? W : Pj + W;
    }
    a.P[(size_t)j * nR + r] = r < nR - 1 ? Pj : 0.0;
  }
}

// The partials alone (before the first step of a call).
__global__ void __launch_bounds__(kT) k_slice_moment(SliceArgs a) {
  extern __shared__ double lds[];
  double *dUs = lds, *G = lds + a.nU;
  const int nR = a.nR;
  for (int u = threadIdx.x; u < a.nU; u += kT) dUs[u] = a.dU[u];
  __syncthreads();
  group_sums(a, blockIdx.x, 0, (a.nU - 1 + 15) / 16, dUs, nullptr, -1,
             [&](int g, int r, double s) { G[g * nR + r] = s; });
  __syncthreads();
  group_combine(a, blockIdx.x, [&](int g, int r) { return G[g * nR + r]; });
}

// The n values of a slice into columns 1..nR of rows 1..nU of the coefficients,
// kB of each thread in flight (n <= kB kT): one round trip to memory.
template <int kB>
__device__ __forceinline__ void load_slice(const double *sj, double *C, int n, int nR, int ps,
                                           unsigned mulR) {
  double v[kB];
  const int i0 = fresh(threadIdx.x);
#pragma unroll
  for (int q = 0; q < kB; q++) v[q] = sj[min(i0 + q * kT, n - 1)];
  __builtin_amdgcn_sched_barrier(0);
  const int i1 = fresh(threadIdx.x);
#pragma unroll
  for (int q = 0; q < kB; q++) {
    const int i = i1 + q * kT;
    if (i < n) C[ps + 1 + i + __umulhi((unsigned)i, mulR) * (unsigned)(ps - nR)] = v[q];
  }
}
static_assert(40 * kT * sizeof(double) >= 163840, "a slice that fits in LDS fits in load_slice<40>");

// A delay line of the slice while its block waits for the solves.
struct LineRec {
  double bxr, bxu, front;  // back foot (kFootOut: outside), value at the front
  int64_t back;            // index of the slot behind the front in vals
  int il;                  // point in the slice (-1: of another block's rows)
  int pad;
};

__global__ void __launch_bounds__(kT) k_slice_drift(SliceArgs a) {
  extern __shared__ double lds[];
  const int nR = a.nR, nU = a.nU;
  const int n = nR * nU, ps = slice_pitch(nR), S = nR + 2, nG = (nU - 1 + 15) / 16;
  double *C = lds, *halo = C + slice_coef(nR, nU), *dUs = halo + nR;
  LineTab *hr = (LineTab *)(dUs + nU), *hv = hr + 1;
  LineRec *rec = (LineRec *)(hv + 1);  // [maxLines]
  int *lastBlock = (int *)(rec + a.maxLines);
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  // the parts of a slice on one XCD (its f in one L2)
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int j = tile / a.parts, part = tile - j * a.parts;
  // this block's groups of 16 rows, and its rows
  const int g0 = part * a.gPart, g1 = min(nG, g0 + a.gPart);
  const int uA = 16 * g0, uB = part == a.parts - 1 ? nU : 16 * g1;

  if (t == 0) {
    line_tab(hr, a.tr);
    line_tab(hv, a.tv);
  }
  for (int u = t; u < nU; u += kT) dUs[u] = a.dU[u];
  // what a stencil on the last knot reads with weight 0: the row after the
  // padded slice, and the column after each row
  for (int i = t; i < ps + 8; i += kT) C[(nU + 2) * ps + i] = 0.0;
  if (ps > S)
    for (int m = t; m < nU + 2; m += kT) C[m * ps + S] = 0.0;

  const bool hasHalo = a.P && uB < nU;
  const int lines0 = a.ch.n ? a.chStart[j] : 0;
  const int nLines = a.ch.n ? a.chStart[j + 1] - lines0 : 0;
#pragma unroll 1
  for (int s = 0; s < a.nS; s++) {
    const size_t at = (size_t)s * a.nVal + (size_t)j * n;
    const double *sj = a.src + at;
    double *fj = a.f + at;
    double *vals = a.ch.vals + (size_t)s * a.nCells;
    // the slice's values, the right-hand sides of the r-solve
    if (n <= 10 * kT)
      load_slice<10>(sj, C, n, nR, ps, a.mulR);
    else if (n <= 20 * kT)
      load_slice<20>(sj, C, n, nR, ps, a.mulR);
    else
      load_slice<40>(sj, C, n, nR, ps, a.mulR);
    __syncthreads();
    // the solves of the rows, then of the padded columns.  One loop, so that
    // the solver, unrolled over its registers, is in the kernel once.
#pragma unroll 1
    for (int ph = 0; ph < 2; ph++) {
      const int lines = ph == 0 ? nU : S, step = ph == 0 ? ps : 1;
      double *first = C + (ph == 0 ? ps : 0);
      const LineTab *ax = ph == 0 ? hr : hv;
#pragma unroll 1
      for (int i = t; i < lines; i += kT)
        lds_line(first + i * step, ph == 0 ? 1 : ps, ph == 0 ? nR : nU, *ax);
      if (ph == 0) {
        // meanwhile the waves without a row bring the first lines of the feet
        // into L2, and the last one collects the delay lines (three dependent
        // loads that the drift would otherwise wait for)
        const int free0 = (lines + 63) / 64 * 64;
        if (t >= free0) {
          const double2 *fp = a.feet + (size_t)j * n;
          double x[4];
#pragma unroll
          for (int q = 0; q < 4; q++)
            x[q] = fp[min(uA * nR + (t - free0 + q * (kT - free0)) * 8, n - 1)].x;
          asm volatile("" ::"v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]));
        }
        if (w == kT / 64 - 1)
          for (int q = lane; q < nLines; q += 64) {
            const int k = a.chOrder[lines0 + q], len = a.ch.len[k];
            const int il = (int)(a.chPoint[k] - (int64_t)j * n);
            const int u = __umulhi((unsigned)il, a.mulR);
            int h = a.ch.head[k] + a.hOff;
            if (h < 0) h += len;
            const int64_t off = a.ch.off[k];
            LineRec l;
            l.bxr = a.ch.bout[k] ? kFootOut : a.ch.bxr[k];
            l.bxu = a.ch.bxu[k];
            l.front = vals[off + h];
            l.back = off + (h == 0 ? len - 1 : h - 1);
            l.il = (u >= uA && u < uB) || (hasHalo && u == uB) ? il : -1;
            rec[q] = l;
          }
      }
      __syncthreads();
    }
    if (a.cOut && part == 0 && s == a.nS - 1) {
      double *co = a.cOut + (size_t)j * a.cs;
      for (int m = w; m < nU + 2; m += kT / 64)
        for (int k = lane; k < S; k += 64) co[m * S + k] = C[m * ps + k];
    }
    // the delay lines (drift_chain), a thread each, from the last one down
    for (int q = kT - 1 - t; q < nLines; q += kT) {
      const LineRec l = rec[q];
      if (l.il < 0) continue;
      if (l.il >= uB * nR) {
        halo[l.il - uB * nR] = l.front;
      } else {
        vals[l.back] = l.bxr > kFootOut ? eval_c(C, ps, l.bxr, l.bxu) : 0.0;
        fj[l.il] = l.front;
      }
    }
    // the drift (k_drift) of this block's rows, the feet of the next kA points
    // loaded ahead; with the row after them for the moment
    const double2 *ft = a.feet + (size_t)j * n;
    const int iB = uB * nR, iE = iB + (hasHalo ? nR : 0);
    constexpr int kA = 4;
    double2 nx[kA];
    const int iW = uA * nR + w * 64;  // the wave's first point
#pragma unroll
    for (int q = 0; q < kA; q++) nx[q] = ft[min(iW + lane + q * kT, n - 1)];
#pragma unroll 1
    for (int b = iW; b < iE; b += kA * kT) {
#pragma unroll
      for (int q = 0; q < kA; q++) {
        if (b + q * kT >= iE) break;
        const int i = b + q * kT + lane;
        const double2 cu = nx[q];
        nx[q] = ft[min(i + kA * kT, n - 1)];
        const bool e = cu.x > kFootOut;
        // the 16 reads together, before the sums
        CStencil st;
        eval_c_fetch(C, ps, e ? cu.x : 0.0, e ? cu.y : 0.0, st);
        __builtin_amdgcn_sched_barrier(0);
        double x = eval_c_sum(st);
        x = e ? x : 0.0;
        if (cu.x >= kFootOut) {  // (delay lines: above)
          if (i < iB)
            fj[i] = x;
          else if (i < iE)
            halo[i - iB] = x;
        }
      }
    }
    if (a.loose) {
      // delay-line points without a line: f keeps its value
      for (int i = uA * nR + t; i < iE; i += kT) {
        const double2 cu = ft[i];
        if (cu.x < kFootOut && cu.y < 0.0) {
          const double x = sj[i];
          if (i < iB)
            fj[i] = x;
          else
            halo[i - iB] = x;
        }
      }
    }
    __syncthreads();
  }
  if (!a.P) return;
  if (a.parts == 1) {
    double *G = C;
    group_sums(a, j, 0, nG, dUs, halo, -1, [&](int g, int r, double s) { G[g * nR + r] = s; });
    __syncthreads();
    group_combine(a, j, [&](int g, int r) { return G[g * nR + r]; });
    return;
  }
  // the block that is the last of its slice to leave its group sums combines
  // them (no block waits for another); it resets the count for the next launch
  double *G = a.G + (size_t)j * nG * nR;
  group_sums(a, j, g0, g1, dUs, halo, uB < nU ? uB : -1,
             [&](int g, int r, double s) { coherent_store(&G[(size_t)g * nR + r], s); });
  wait_stores();
  __syncthreads();
  if (t == 0) {
    const unsigned o =
        __hip_atomic_fetch_add(&a.cnt[j], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *lastBlock = o == (unsigned)(a.parts - 1);
    if (*lastBlock) __hip_atomic_store(&a.cnt[j], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (*lastBlock)
    group_combine(a, j, [&](int g, int r) { return coherent_load(&G[(size_t)g * nR + r]); });
}

size_t slice_lds(int nR, int nU, int maxLines) {
  return (slice_coef(nR, nU) + nR + (size_t)nU + 1) * sizeof(double) + 2 * sizeof(LineTab) +
         maxLines * sizeof(LineRec);
}

// Blocks per slice of the drift: as many as keep the grid within one block per
// CU (of the run's share of them in an ensemble, whose runs execute side by
// side), each with at least one group of 16 rows (several species: the moment
// needs all of a slice's planes in one block).
int slice_parts(const Run &r) {
  const int nG = (r.nU - 1 + 15) / 16;
  return r.nS > 1 ? 1 : std::max(1, std::min(nG, r.cus / r.nJ));
}

SliceArgs slice_args(Run &r) {
  SliceArgs a{};
  a.src = a.f = r.f;
  a.Ct1 = r.Ct1;
  a.dU = r.dU;
  a.dR = r.dR;
  a.feet = (const double2 *)r.feet;
  a.ch = ChainTables{r.ch_off, r.ch_len, r.ch_head, r.ch_xr, r.ch_xu, r.ch_out, r.ch_vals, r.nChains, 0};
  a.chPoint = r.ch_point;
  a.chOrder = r.ch_order;
  a.chStart = r.ch_start;
  a.nVal = r.nVal;
  a.nCells = r.nCells;
  a.cs = r.cs;
  a.tr = r.tr;
  a.tv = r.tv;
  a.nR = r.nR;
  a.nU = r.nU;
  a.nJ = r.nJ;
  a.nS = r.nS;
  a.mulR = magic(r.nR);
  a.G = r.sliceG;
  a.cnt = r.sliceCnt;
  const int nG = (r.nU - 1 + 15) / 16, parts = slice_parts(r);
  a.maxLines = r.maxLines;
  a.loose = r.nLoose > 0;
  a.gPart = (nG + parts - 1) / parts;
  a.parts = (nG + a.gPart - 1) / a.gPart;
  return a;
}

void launch_drift(Run &r, SliceArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(k_slice_drift, dim3(a.nJ * a.parts), dim3(kT), slice_lds(a.nR, a.nU, a.maxLines), s, a);
}

// where the kick leaves f for the drift
double *kicked(Run &r) { return r.sliceF ? r.sliceF : r.f; }

// columns of a tile of the kick: the fewest tiles of at most 64 columns, or
// more of them while they still find idle CUs (down to 16 columns)
int kick_width(const Run &r) {
  int nT = (r.nR + 63) / 64;
  while (r.nJ * (nT + 1) <= r.cus && (r.nR + nT) / (nT + 1) >= 16) nT++;
  return (r.nR + nT - 1) / nT;
}

// ---------------------------------------------------------------- line tiles
struct TileArgs {
  const double *src;
  double *dst;
  ThomasAxis ax;
  int nR, nU, W, nT, pitch;
  unsigned mulIn, mulOut;  // i / (elements of a row in, out) == __umulhi(i, mul)
  int64_t cs;
};

// The r-solves (kRows: lines are rows of f) and v-solves (columns of the
// padded rows, in place allowed) of a tile of a slice's lines in LDS, for the
// drift's spline of grids whose slices don't fit in a CU's LDS and whose lines
// don't fit in registers.  One of the block's two waves solves (222 registers:
// eight waves a CU); the loads and stores of the other blocks on the CU run
// beside it.  Blocks of 128 threads and 52 KB took 16 and 26 us where 256 and
// 80 KB took 15 and 25 at 129x257x96, and 25 and 21 for 23 and 29 at
// 257x129x128.
template <bool kRows>
__global__ void __launch_bounds__(128) k_line_tile(TileArgs a) {
  extern __shared__ double lds[];
  constexpr int kTL = 128, kB = 16;
  const int t = threadIdx.x, W = a.W, nR = a.nR, nU = a.nU, S = nR + 2;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int j = tile / a.nT, l0 = (tile - j * a.nT) * W;
  const int wid = min(W, (kRows ? nU : S) - l0), ps = a.pitch;
  double *D = lds;
  LineTab *tab = (LineTab *)(D + (kRows ? W * ps : (nU + 2) * W));
  if (t == 0) line_tab(tab, a.ax);
  if constexpr (kRows) {
    const double *src = a.src + ((size_t)j * nU + l0) * nR;
    const int n = wid * nR;
#pragma unroll 1
    for (int b = t; b < n; b += kB * kTL) {
      double v[kB];
#pragma unroll
      for (int q = 0; q < kB; q++) v[q] = src[min(b + q * kTL, n - 1)];
#pragma unroll
      for (int q = 0; q < kB; q++) {
        const int e = b + q * kTL;
        if (e < n) D[1 + e + (int)__umulhi((unsigned)e, a.mulIn) * (ps - nR)] = v[q];
      }
    }
  } else {
    const double *src = a.src + (size_t)j * a.cs + S + l0;
    const int n = nU * W;
#pragma unroll 1
    for (int b = t; b < n; b += kB * kTL) {
      double v[kB];
#pragma unroll
      for (int q = 0; q < kB; q++) {
        const int e = min(b + q * kTL, n - 1);
        const int u = __umulhi((unsigned)e, a.mulIn), c = e - u * W;
        v[q] = src[(size_t)u * S + min(c, wid - 1)];
      }
#pragma unroll
      for (int q = 0; q < kB; q++)
        if (b + q * kTL < n) D[W + b + q * kTL] = v[q];
    }
  }
  __syncthreads();
  if (t < wid) lds_line(kRows ? D + t * ps : D + t, kRows ? 1 : W, kRows ? nR : nU, *tab);
  __syncthreads();
  if constexpr (kRows) {
    double *dst = a.dst + (size_t)j * a.cs + (size_t)(l0 + 1) * S;
    const int n = wid * S;
#pragma unroll 4
    for (int e = t; e < n; e += kTL)
      dst[e] = D[e + (int)__umulhi((unsigned)e, a.mulOut) * (ps - S)];
  } else {
    double *dst = a.dst + (size_t)j * a.cs + l0;
    const int n = (nU + 2) * W;
#pragma unroll 4
    for (int e = t; e < n; e += kTL) {
      const int u = __umulhi((unsigned)e, a.mulOut), c = e - u * W;
      if (c < wid) dst[(size_t)u * S + c] = D[e];
    }
  }
}

// ---------------------------------------------------------------- adjoint
// The line adjoints of the drift's spline (the sweeps of k_adj_v and k_adj_r,
// vls_adjoint.hip: c1 -= A01 c0, c2 -= A02 c0, c[t] -= u[t-1] c[t-1] going up,
// then the last row, the scaling by 1/d and the carry c16 c[k] going down) by
// tiles of lines in LDS: the streaming kernels take the line through memory
// twice each way.  Same operations, same order: on grids without register
// line adjoints those of the streaming sweeps (adj_down: the carry c16 c[k]
// rounded, then subtracted), on the others those of the register kernels
// (kFused, k_adj_rows: an fma of c16, after the last row's terms).  A block's
// first wave sweeps (a chain of 1 dependent operation up and 3, fused 2, down,
// a DS read and a write a row).
struct AdjTileArgs {
  double *cb;   // padded coefficients' adjoints; columns: in place
  double *out;  // rows: f's layout
  ThomasAxis ax;
  int nR, nU, W, nT, pitch;
  unsigned mulIn, mulOut;
  int64_t cs;
};

// A line in LDS, in place: p[k st], k = 0..M-1.  Chunks of kQ rows, read a
// chunk ahead.
template <bool kFused>
__device__ __forceinline__ void lds_line_adjoint(double *p, int st, const ThomasAxis &ax) {
  const int M = ax.M;
  constexpr int kQ = 8, kH = kHead + 2;  // rows 0 .. kHead + 1 take the pivots of the head
  st = __builtin_amdgcn_readfirstlane(st);
  asm volatile("" : "+s"(st));
  const double uS = kPivU[kHead + 1], rdS = kPivRd[kHead + 1];
  double h[kH];
#pragma unroll
  for (int t = 0; t < kH; t++) h[t] = p[min(t, M - 1) * st];
  double prev = 0.0;
#pragma unroll
  for (int t = 0; t < kH; t++) {
    if (t < M) {
      if (t == 1) h[t] = fma(-ax.A01, h[0], h[t]);
      if (t == 2) h[t] = fma(-ax.A02, h[0], h[t]);
      if (t >= 2) h[t] = fma(-kPivU[t - 1], prev, h[t]);
      prev = h[t];
      p[t * st] = prev;
    }
  }
  double a[kQ];
  double *sp = p + kH * st;
  int t = kH;
  if (t + kQ <= M) {
#pragma unroll
    for (int q = 0; q < kQ; q++) a[q] = sp[q * st];
#pragma unroll 1
    for (; t + 2 * kQ <= M; t += kQ) {
      double b[kQ];
#pragma unroll
      for (int q = 0; q < kQ; q++) b[q] = a[q];
#pragma unroll
      for (int q = 0; q < kQ; q++) a[q] = sp[(kQ + q) * st];
#pragma unroll
      for (int q = 0; q < kQ; q++) {
        prev = fma(-uS, prev, b[q]);
        *sp = prev;
        sp += st;
      }
    }
#pragma unroll
    for (int q = 0; q < kQ; q++) {
      prev = fma(-uS, prev, a[q]);
      *sp = prev;
      sp += st;
    }
    t += kQ;
  }
  for (; t < M; t++) {
    prev = fma(-uS, prev, *sp);
    *sp = prev;
    sp += st;
  }
  const double tt = prev * ax.rq;  // prev = c[M-1]
  // element k from its value x of the ascending sweep; the carry is c[k + 1],
  // or c16 times that.  last: the last row's coefficient in rows M-2 and M-3.
  double carry = 0.0;
  auto down = [&](double x, double rd) {
    double v = kFused ? fma(-ax.c16, carry, x) : x - carry;
    v *= rd;
    carry = kFused ? v : ax.c16 * v;
    return v;
  };
  auto down_last = [&](double x, double last, double rd) {
    if constexpr (kFused) return down(fma(-last, tt, x), rd);
    double v = fma(-last, tt, x - carry);
    v *= rd;
    carry = ax.c16 * v;
    return v;
  };
  auto put = [&](double v) {
    *sp = v;
    sp -= st;
  };
  sp = p + (M - 2) * st;
  int k = M - 2;
  if (k > kHead) {
    put(down_last(*sp, ax.p, rdS));
    k--;
  }
  if (k > kHead && k == M - 3) {
    put(down_last(*sp, ax.hi2, rdS));
    k--;
  }
  if (k - kQ >= kHead) {
#pragma unroll
    for (int q = 0; q < kQ; q++) a[q] = sp[-q * st];
#pragma unroll 1
    for (; k - 2 * kQ >= kHead; k -= kQ) {
      double b[kQ];
#pragma unroll
      for (int q = 0; q < kQ; q++) b[q] = a[q];
#pragma unroll
      for (int q = 0; q < kQ; q++) a[q] = sp[-(kQ + q) * st];
#pragma unroll
      for (int q = 0; q < kQ; q++) put(down(b[q], rdS));
    }
#pragma unroll
    for (int q = 0; q < kQ; q++) put(down(a[q], rdS));
    k -= kQ;
  }
  for (; k > kHead; k--) put(down(*sp, rdS));
#pragma unroll
  for (int m = kHead; m >= 1; m--) {
    if (m <= M - 2)
      p[m * st] = m >= M - 3 ? down_last(h[m], m == M - 2 ? ax.p : ax.hi2, kPivRd[m])
                             : down(h[m], kPivRd[m]);
  }
}

template <bool kRows, bool kFused>
__global__ void __launch_bounds__(128) k_adj_line_tile(AdjTileArgs a) {
  extern __shared__ double D[];
  constexpr int kTL = 128, kB = 16;
  const int t = threadIdx.x, W = a.W, nR = a.nR, nU = a.nU, S = nR + 2;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int j = tile / a.nT, l0 = (tile - j * a.nT) * W;
  const int wid = min(W, (kRows ? nU : S) - l0), ps = a.pitch;
  double *src = a.cb + (size_t)j * a.cs + (kRows ? (size_t)(l0 + 1) * S : l0);
  const int n = kRows ? wid * S : (nU + 2) * W;
#pragma unroll 1
  for (int b = t; b < n; b += kB * kTL) {
    double v[kB];
#pragma unroll
    for (int q = 0; q < kB; q++) {
      const int e = min(b + q * kTL, n - 1);
      if constexpr (kRows) {
        v[q] = src[e];
      } else {
        const int m = __umulhi((unsigned)e, a.mulIn), c = e - m * W;
        v[q] = src[(size_t)m * S + min(c, wid - 1)];
      }
    }
#pragma unroll
    for (int q = 0; q < kB; q++) {
      const int e = b + q * kTL;
      if (e < n) D[kRows ? e + (int)__umulhi((unsigned)e, a.mulIn) * (ps - S) : e] = v[q];
    }
  }
  __syncthreads();
  if (t < wid) lds_line_adjoint<kFused>(kRows ? D + t * ps : D + t, kRows ? 1 : W, a.ax);
  __syncthreads();
  if constexpr (kRows) {
    double *dst = a.out + ((size_t)j * nU + l0) * nR;
#pragma unroll 4
    for (int e = t; e < wid * nR; e += kTL)
      dst[e] = D[1 + e + (int)__umulhi((unsigned)e, a.mulOut) * (ps - nR)];
  } else {
    // rows 1 .. nU: the r-direction takes no others
#pragma unroll 4
    for (int e = t; e < nU * W; e += kTL) {
      const int u = __umulhi((unsigned)e, a.mulOut), c = e - u * W;
      if (c < wid) src[(size_t)(u + 1) * S + c] = D[W + e];
    }
  }
}

}  // namespace

// Whether the set-up's table holds the pivots that lds_line has as literals.
bool slice_pivots(const ThomasAxis &ax, const double *u, const double *rd, const double *rl) {
  if (ax.c16 != kC16 || ax.A01 != -2.0 || ax.A02 != 1.0 || ax.A03 != 0.0) return false;
  for (int k = 1; k <= ax.M - 2; k++) {
    const int h = k <= kHead ? k : kHead + 1;
    if (u[k] != kPivU[h] || rd[k] != kPivRd[h] || rl[k] != kPivRl[h]) return false;
  }
  return true;
}

bool slice_shape(const Run &r, int maxLdsPerBlock) {
  return maxLdsPerBlock >= kMaxLds && slice_lds(r.nR, r.nU, r.maxLines) <= (size_t)kMaxLds &&
         kick_lds(r.nR, r.nU, r.nJ, kick_width(r), true) <= (size_t)kMaxLds;
}

size_t slice_group_doubles(const Run &r) { return (size_t)r.nJ * ((r.nU + 14) / 16) * r.nR; }
bool slice_shared(const Run &r) { return slice_parts(r) > 1; }

void configure_slice(int maxLdsPerBlock) {
  // once per device: a tenth of a small context's creation otherwise
  static std::mutex mu;
  static std::set<int> done;
  int device = 0;
  VLS_HIP_CHECK(hipGetDevice(&device));
  std::lock_guard<std::mutex> lock(mu);
  if (done.count(device)) return;
  for (const void *fn : {(const void *)k_kick_tile<256>, (const void *)k_kick_tile<512>,
                         (const void *)k_slice_drift, (const void *)k_slice_moment,
                         (const void *)k_line_tile<true>, (const void *)k_line_tile<false>,
                         (const void *)k_adj_line_tile<true, false>,
                         (const void *)k_adj_line_tile<true, true>,
                         (const void *)k_adj_line_tile<false, false>})
    VLS_HIP_CHECK(
        hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, maxLdsPerBlock));
  done.insert(device);
}

bool slice_fits(const Run &r) {
  return r.sliceG && !r.feetPast && !r.backPast &&
         slice_lds(r.nR, r.nU, r.maxLines) <= (size_t)kMaxLds;
}

// Whether a run's steps go by slice unless it is told otherwise.  Every block
// of the kick sums the moment partials of all slices, and past a round of the
// drift (a block fills a CU's registers) or two of the kick (two blocks on a
// CU) the kernels per phase fill the chip as well.  us a step, by slice and
// per phase:
//   slices: 65x65x256 38, 53 and x300 67, 56; x1024 216, 115; 17x17x4096 428,
//     72; 97x97x256 61, 73; 91x81x320 92, 86.  Where a tile of the kick holds
//     all columns a second round pays too, unless the columns are short and
//     have register kernels: 50x50x512 51, 61; 33x65x512 46, 51 and x600 71,
//     56; 49x49x512 50, 54 and x600 77, 59; but 49x33x400 43, 40; 33x33x512
//     40, 38 (two species 63, 75);
//   blocks of the kick: register lines win up to 512 (193x65x128, 512, 59, 65;
//     129x129x160, 480, 76, 80; x192, 576, 94, 87; 193x65x150, 600, 83, 72),
//     others to 640 unless rows are long (150x100x200, 600, 92, 102;
//     181x81x200, 600, 95, 100; 225x60x192, 768, 97, 93; 300x49x100, 500, 69,
//     80 but x128, 640, 94, 88; 257x57x256 149, 123); with a second drift or
//     species to 768 (129x129x256, 768, without linking 146, 159, two
//     species 184, 205).
bool slice_pays(const Run &r) {
  const int W = kick_width(r), nT = (r.nR + W - 1) / W;
  const bool lines = register_lines(r), twice = r.nS > 1 || r.sp.no_linking;
  const bool rounds = nT == 1 && (!lines || r.nU >= 49 || r.nS > 1);
  if (r.nJ > (rounds ? 2 : 1) * kCUs) return false;
  return r.nJ * nT <= (twice ? 3 * kCUs : lines || nT > 3 ? 2 * kCUs : 5 * kCUs / 2);
}

bool slice_on(const Run &r) {
  if (!slice_fits(r)) return false;
  if (r.sliceMode >= 0) return r.sliceMode == 1;
  if (r.lineMode >= 0 || r.kickMode >= 0) return false;
  for (const char *e : {"VLS_NO_SLICE_STEP", "VLS_NO_REGISTER_LINES", "VLS_FUSED_KICK",
                        "VLS_NO_FUSED_KICK", "VLS_KICK_SCRATCH", "VLS_KICK_RSOLVE",
                        "VLS_NO_KICK_MOMENT", "VLS_MOMENT_3K", "VLS_SPLINE_STREAM", "VLS_TILE_R",
                        "VLS_TILE_V"})
    if (getenv(e)) return false;
  return getenv("VLS_SLICE_STEP") || slice_pays(r);
}

size_t partials_lds(const Run &r) {
  return ((size_t)r.nU + (size_t)(r.nU + 14) / 16 * r.nR) * sizeof(double);
}

bool launch_slice_partials(Run &r, const double *f, double *P, hipStream_t s) {
  if (partials_lds(r) > (size_t)kMaxLds) return false;
  SliceArgs a = slice_args(r);
  a.f = const_cast<double *>(f);  // read only
  a.P = P;
  hipLaunchKernelGGL(k_slice_moment, dim3(r.nJ), dim3(kT), partials_lds(r), s, a);
  return true;
}

void launch_slice_start(Run &r, hipStream_t s) {
  SliceArgs a = slice_args(r);
  a.P = r.P;
  if (r.sp.no_linking) {  // the first half step
    a.f = kicked(r);
    launch_drift(r, a, s);
    return;
  }
  launch_slice_partials(r, r.f, r.P, s);
}

static KickArgs kick_args(Run &r, int W) {
  KickArgs k{};
  k.src = k.dst = r.f;
  k.gfac = r.gfac;
  k.U_Val = r.U_Val;
  k.dM = r.dM;
  k.Mx = r.Mx;
  k.acc = r.acc;
  k.mTot = r.mTot;
  k.nVal = r.nVal;
  k.cs = r.cs;
  k.Ulo = r.Ulo;
  k.Uhi = r.Uhi;
  k.start_v = r.start_v;
  k.hinv_v = r.hinv_v;
  k.tv = r.tv;
  k.nR = r.nR;
  k.nU = r.nU;
  k.nJ = r.nJ;
  k.nS = r.nS;
  k.W = W;
  k.nT = (r.nR + W - 1) / W;
  k.mulW = magic(W);
  k.mulR = magic(r.nR);
  return k;
}

void launch_slice_kick(Run &r, hipStream_t s, double *dKeep) {
  KickArgs k = kick_args(r, kick_width(r));
  if (r.sp.no_linking) k.src = kicked(r);
  k.dst = kicked(r);
  k.P = r.P;
  k.dKeep = dKeep;
  k.head = r.nChains ? r.ch_head : nullptr;
  k.len = r.ch_len;
  k.nChains = r.nChains;
  k.roll = r.sp.no_linking ? 2 : 1;
  const bool wide = r.nJ * k.nT <= r.cus;
  hipLaunchKernelGGL(wide ? k_kick_tile<512> : k_kick_tile<256>, dim3(r.nJ * k.nT),
                     dim3(wide ? 512 : 256), kick_lds(r.nR, r.nU, r.nJ, k.W, true), s, k);
}

// Lines per tile of `lines` lines of L rows, in equal tiles of at most kb
// KiB (other: bytes of them not taken by lines), or of 16 lines if two such
// tiles fit on a CU (0: they don't).
static int tile_lines(int L, int lines, size_t other, int kb) {
  const size_t line = (size_t)((L + 3) | 1) * sizeof(double);
  const size_t room = (size_t)kb * 1024 - 512 - other, most = (size_t)kMaxLds / 2 - 512;
  const int W = (int)std::min<size_t>(64, std::max<size_t>(room / line, 16));
  if (W * line + other > most) return 0;
  const int nT = (lines + W - 1) / W;
  return (lines + nT - 1) / nT;
}
constexpr int kLineKB = 52, kKickKB = 80;  // three and two blocks on a CU

static int line_tile_width(const Run &r, bool rows) {
  return tile_lines(rows ? r.nR : r.nU, rows ? r.nU : r.nR + 2, 64, kLineKB);
}
static size_t kick_tile_other(const Run &r) {
  return (r.nU + (size_t)r.nR + 1) * sizeof(double) + sizeof(LineTab);
}

bool line_tile_shape(const Run &r, bool rows) {
  return r.pivots && line_tile_width(r, rows) > 0;
}

// Which of the solves and the kick of a run without register lines go by
// tiles (the axes have the pivots above).  A tile's time is a line's chain and the CU holds 160 KB of lines,
// where the streaming solves have every line in flight but wait for memory
// every segment: tiles win while there are few lines.
//   r: always where 20 rows fit in a tile, else up to four blocks a CU
//      (stream, tile in us: 129x257x96 38, 15; 257x129x128 60, 24;
//      321x321x200 190, 129; 401x401x30 79, 61; but 385x385x128 138, 144 and
//      481x481x40 101, 105)
//   v: the blocks in one round, three a CU (37, 26; 28, 21; but 301x301x64
//      45, 57 and 321x321x100 53, 86: the streaming columns come in rows of
//      512 bytes)
//   kick: always, unless it streams (with the moment, for the column splines
//      and the evaluation: 129x257x96 89, 52; 257x129x128 71, 58; 211x181x64
//      70, 44; 321x321x128 166 streaming, 139; kick_stream_shape)
void choose_line_tiles(Run &r) {
  if (!r.pivots) return;
  for (const char *e : {"VLS_NO_REGISTER_LINES", "VLS_SPLINE_STREAM", "VLS_TILE_R", "VLS_TILE_V"})
    if (getenv(e)) return;
  r.lineTiles = true;
  const int wr = line_tile_width(r, true), wv = line_tile_width(r, false);
  auto blocks = [&](int lines, int w) { return (int64_t)(lines + w - 1) / w * r.nJ; };
  r.tileR = wr > 0 && ((r.nR + 4) * sizeof(double) * 20 <= kLineKB * 1024 ||
                       blocks(r.nU, wr) <= 4 * kCUs);
  r.tileV = wv > 0 && blocks(r.nR + 2, wv) <= 3 * kCUs;
  r.tileK = !r.kept && tile_lines(r.nU, r.nR, kick_tile_other(r), kKickKB) > 0;
}

void launch_line_tile(const Run &r, bool rows, const double *src, double *dst, hipStream_t s) {
  TileArgs a{};
  a.src = src;
  a.dst = dst;
  a.ax = rows ? r.tr : r.tv;
  a.nR = r.nR;
  a.nU = r.nU;
  a.cs = r.cs;
  const int lines = rows ? r.nU : r.nR + 2;
  a.W = line_tile_width(r, rows);
  a.nT = (lines + a.W - 1) / a.W;
  a.pitch = (r.nR + 2) | 1;
  a.mulIn = magic(rows ? r.nR : a.W);
  a.mulOut = magic(rows ? r.nR + 2 : a.W);
  const size_t lds = (rows ? (size_t)a.W * a.pitch : (size_t)a.W * (r.nU + 2)) * sizeof(double) +
                     sizeof(LineTab);
  hipLaunchKernelGGL(rows ? k_line_tile<true> : k_line_tile<false>, dim3(a.nT * r.nJ), dim3(128),
                     lds, s, a);
}

constexpr int kAdjKB = 40;  // four blocks on a CU (of 26 KB: 5% slower)
static int adj_tile_width(const Run &r, bool rows) {
  return tile_lines(rows ? r.nR : r.nU, rows ? r.nU : r.nR + 2, 0, kAdjKB);
}

// The blocks of the tiles in one round: us of the streaming sweeps and of the
// tiles, r: 40 and 16 on average over runs of 151x132x96, 211x181x64,
// 132x258x70 and 97x65x48, v: 31 and 20; at 201x201x200 (1800 blocks) 73 and 47,
// 52 and 51, but the walk after it then takes 27 more.  On register shapes
// the columns are faster there (129x129x64: 9 us against 17), the rows here
// (18 against 14).
bool adj_line_tile(const Run &r, bool rows) {
  const int w = r.lineTiles ? adj_tile_width(r, rows) : 0, lines = rows ? r.nU : r.nR + 2;
  return w > 0 && (int64_t)(lines + w - 1) / w * r.nJ <= 4 * kCUs;
}

void launch_adj_line_tile(const Run &r, bool rows, bool fused, double *cb, double *out,
                          hipStream_t s) {
  AdjTileArgs a{};
  a.cb = cb;
  a.out = out;
  a.ax = rows ? r.tr : r.tv;
  a.nR = r.nR;
  a.nU = r.nU;
  a.cs = r.cs;
  const int lines = rows ? r.nU : r.nR + 2;
  a.W = adj_tile_width(r, rows);
  a.nT = (lines + a.W - 1) / a.W;
  a.pitch = (r.nR + 2) | 1;
  a.mulIn = magic(rows ? r.nR + 2 : a.W);
  a.mulOut = magic(rows ? r.nR : a.W);
  const size_t lds = (size_t)a.W * (rows ? a.pitch : r.nU + 2) * sizeof(double);
  void (*fn)(AdjTileArgs) = k_adj_line_tile<false, false>;
  if (rows) fn = k_adj_line_tile<true, false>;
  if (rows && fused) fn = k_adj_line_tile<true, true>;
  hipLaunchKernelGGL(fn, dim3(a.nT * r.nJ), dim3(128), lds, s, a);
}

void launch_kick_tile(Run &r, hipStream_t s, double *dKeep) {
  KickArgs k = kick_args(r, tile_lines(r.nU, r.nR, kick_tile_other(r), kKickKB));
  k.nS = 1;  // the plane r.f
  k.dKeep = dKeep;
  hipLaunchKernelGGL(k_kick_tile<256>, dim3(r.nJ * k.nT), dim3(256),
                     kick_lds(r.nR, r.nU, r.nJ, k.W, false), s, k);
}

void launch_slice_drift(Run &r, hipStream_t s, bool last) {
  SliceArgs a = slice_args(r);
  // the kick has advanced the heads by the step's drifts: this is its last
  a.src = kicked(r);
  a.hOff = -1;
  if (r.sp.no_linking && !last) {
    launch_drift(r, a, s);  // and the first half of the next step
    a.src = r.f;
    a.f = kicked(r);
    a.hOff = 0;
  }
  a.P = last ? nullptr : r.P;
  a.cOut = last ? r.c : nullptr;
  launch_drift(r, a, s);
}

}  // namespace vls
