// Line solves and kick of lines too long for a tile in LDS or registers
// (gfx950, FP64): streaming, with the elimination taken twice.
//
// A line's forward values y_k are needed again, last first, by the back
// substitution.  Written over the line and read back they make four passes
// over memory of a solve that reads and writes its line once.  Here the
// elimination keeps only every kSeg-th y; the back substitution takes the
// line a segment of kSeg rows at a time from its end, repeats the segment's
// elimination from the kept y before it in registers and substitutes back:
// two reads and one write.  The repeated operations are the same, so are the
// bits.  At 513x513x256, whose planes of 0.54 GB come from HBM, the v-solves
// take 342 to 374 us for 477 and the r-solves 496 to 516 for 646 (637 with
// segments of 16 columns: rows start off the 128-byte lines, and a segment's
// first and last line are fetched twice).  Columns take
// segments of 16 rows: of 32, the two copies of a segment do not fit in the
// 168 registers that leave three waves a SIMD.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include "vls_device.hpp"
#include "vls_div.hpp"
#include "vls_internal.hpp"
#include "vls_tile.hpp"

namespace vls {
namespace {

// rows of a segment
constexpr int kSegR = 32, kSegV = 16, kSegK = kSegRows;

// the loop constants of an axis
struct Steady {
  double c16, rd, rl, u;
};
__device__ __forceinline__ Steady steady(const ThomasAxis &ax, int lz) {
  // per-lane values (x + lz == x), so that no loop waits for a scalar load
  return {ax.c16 + (double)lz, ax.rdS + (double)lz, ax.rlS + (double)lz, ax.uS + (double)lz};
}

// y of row k from its right-hand side and the y before it
__device__ __forceinline__ double eliminate(const ThomasAxis &ax, const Steady &st, int k, bool edge,
                                            double rhs, double before) {
  double rd = st.rd, rl = st.rl;
  if (edge && k <= kHead) {
    rd = ax.rd[k];
    rl = ax.rl[k];
  }
  return div_pivot(rhs - st.c16 * before, rd, rl);
}

// c of the last row of a line whose last elimination values are y2, y1
__device__ __forceinline__ double last_row(const ThomasAxis &ax, double y2, double y1) {
  double t = 0.0 - ax.hi2 * y2;
  t = t - ax.p * y1;
  return div_known(t, ax.q, ax.rq);
}

// A row of a wave's columns: a wave-uniform address (scalar registers) and the
// lane's byte offset in it.  step() moves by whole rows; opaque, or the
// compiler would keep the offset of every row of a segment in registers.
struct RowPtr {
  char *p;
  int64_t bytes;  // from a row to the next
  __device__ __forceinline__ RowPtr(const double *a, int64_t row, int64_t stride)
      : p((char *)(a + row * stride)), bytes(stride * (int64_t)sizeof(double)) {}
  __device__ __forceinline__ void step(int n) {
    p += n * bytes;
    uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)p);
    uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uintptr_t)p >> 32));
    asm volatile("" : "+s"(lo), "+s"(hi));
    p = (char *)((uintptr_t)lo | (uintptr_t)hi << 32);
  }
  __device__ __forceinline__ double &at(uint32_t off) const { return *(double *)(p + off); }
};

// The elimination of a column, the right-hand side of row k in row k of a
// (stride doubles apart), kAhead rows ahead; KEEP(k, y) sees the y of every
// kSeg-th row but the last.
template <int kSeg, int kAhead, class KEEP>
__device__ __forceinline__ void down_sweep(const ThomasAxis &ax, const Steady &st, const double *a,
                                           int64_t stride, uint32_t off, KEEP keep) {
  static_assert(kSeg % kAhead == 0 && kAhead >= kHead, "");
  const int n = ax.M - 2;
  double b[kAhead];
  RowPtr in(a, 1, stride);
#pragma unroll
  for (int q = 0; q < kAhead; q++) {
    b[q] = in.at(off);
    in.step(1 + q < n ? 1 : 0);
  }
  double y = ax.A03;
  auto rows = [&](int k0, bool edge) {
#pragma unroll
    for (int q = 0; q < kAhead; q++) {
      const int k = k0 + q;
      if (!edge || k <= n) y = eliminate(ax, st, k, edge, b[q], y);
      b[q] = in.at(off);
      in.step(k + kAhead < n ? 1 : 0);
    }
  };
  rows(1, true);
  int k0 = 1 + kAhead;
  for (; k0 + kAhead - 1 < n; k0 += kAhead) {
    if (k0 % kSeg == 1) keep(k0 - 1, y);
    rows(k0, false);
  }
  if (k0 <= n && k0 % kSeg == 1) keep(k0 - 1, y);
}

// Back substitution of a column with its elimination repeated: KEPT(k) the y
// kept of row k, OUT(k, c) takes the coefficients k = M-1 .. 0.  The next
// segment's right-hand sides are on their way during a segment.
template <int kSeg, class KEPT, class OUT>
__device__ __forceinline__ void up_sweep(const ThomasAxis &ax, const Steady &st, const double *a,
                                         int64_t stride, uint32_t off, KEPT kept, OUT out) {
  const int n = ax.M - 2, sTop = (n - 1) / kSeg;
  double b[kSeg], y[kSeg];
  RowPtr in(a, sTop * kSeg + 1, stride);
#pragma unroll
  for (int i = 0; i < kSeg; i++) {
    b[i] = in.at(off);
    in.step(sTop * kSeg + 1 + i < n ? 1 : 0);
  }
  double before = sTop > 0 ? kept(sTop * kSeg) : ax.A03;
  double end = 0.0;  // y of the segment's last row, below the top one
  double cn = 0.0, c2 = 0.0;
  auto down = [&](int k0, bool edge, bool top) {
    double ym = before, y2 = 0.0;
#pragma unroll
    for (int i = 0; i < kSeg; i++) {
      if (!edge || k0 + i <= n) {
        y2 = ym;
        ym = eliminate(ax, st, k0 + i, edge, b[i], ym);
        if (i == kSeg - 1 && !top) ym = end;
        y[i] = ym;
      }
    }
    if (edge && top) {
      cn = last_row(ax, y2, ym);
      out(ax.M - 1, cn);
    }
  };
  auto up = [&](int k0, bool edge) {
#pragma unroll
    for (int i = kSeg - 1; i >= 0; i--) {
      const int k = k0 + i;
      if (!edge || k <= n) {
        double u = st.u;
        if (edge && k <= kHead) u = ax.u[k];
        const double c = y[i] - u * cn;
        out(k, c);
        c2 = cn;
        cn = c;
      }
    }
  };
  for (int s = sTop; s >= 0; s--) {
    const int k0 = s * kSeg + 1;
    const bool edge = s == sTop || s == 0;
    if (edge)
      down(k0, true, s == sTop);
    else
      down(k0, false, false);
    end = before;
    if (s > 0) {
      // rows k0 - kSeg .. k0 - 2 (the segment's last y is the kept one)
      in = RowPtr(a, k0 - kSeg, stride);
#pragma unroll
      for (int i = 0; i < kSeg - 1; i++) {
        b[i] = in.at(off);
        in.step(1);
      }
      before = s > 1 ? kept((s - 1) * kSeg) : ax.A03;
    }
    if (edge)
      up(k0, true);
    else
      up(k0, false);
  }
  out(0, (ax.A03 - ax.A01 * cn) - ax.A02 * c2);
}

}  // namespace

// v-solves: lane = padded column, every access a coalesced row segment.  src
// may be c itself; the kept y go to their rows of c, which hold no
// right-hand side that is still needed (a segment's last row is known).
__global__ void __launch_bounds__(64, 3)
k_spline_v_stream(const double *src, double *c, int nR, int64_t cs, int lzmask, ThomasAxis ax) {
  const int lane = threadIdx.x;
  const int S = nR + 2;
  const Tile2 t = xcd_tile2((S + 63) / 64);
  const int col = t.x * 64 + lane;
  if (col >= S) return;  // no barriers below
  const Steady st = steady(ax, lane & lzmask);
  const double *in = src + (size_t)t.j * cs + t.x * 64;
  double *tab = c + (size_t)t.j * cs + t.x * 64;
  const uint32_t off = lane * sizeof(double);
  down_sweep<kSegV, 16>(ax, st, in, S, off, [&](int k, double y) { RowPtr(tab, k, S).at(off) = y; });
  RowPtr o(tab, ax.M - 1, S);
  up_sweep<kSegV>(
      ax, st, in, S, off, [&](int k) { return RowPtr(tab, k, S).at(off); },
      [&](int, double v) {
        o.at(off) = v;
        o.step(-1);
      });
}

// r-solves: lane = row, 64 consecutive rows of a slice per wave; segments of
// kSeg columns through a transpose in LDS, so that the global accesses are
// row segments.  The kept y of segment s waits in column 1 + s of the row's
// coefficients: that column is in a segment before s + 1, which takes the y.
__global__ void __launch_bounds__(64)
k_spline_r_stream(const double *__restrict__ f, double *__restrict__ c, int nR, int nU, int64_t cs,
                  int lzmask, ThomasAxis ax) {
  constexpr int kSeg = kSegR, kRowP = kSeg + 1;
  __shared__ double chunk[64 * kRowP];
  const int M = nR + 2;
  const int lane = threadIdx.x;
  const Steady st = steady(ax, lane & lzmask);
  const Tile2 tl = xcd_tile2((nU + 63) / 64);
  const int u0 = tl.x * 64;
  const int rows = min(64, nU - u0);
  const int rsub = lane / kSeg, ksub = lane % kSeg;
  constexpr int kR = 64 / kSeg;  // rows of a pass
  const double *src = f + ((size_t)tl.j * nU + u0) * nR;
  double *dst = c + (size_t)tl.j * cs + (size_t)(u0 + 1) * M;
  double *own = dst + (size_t)min(lane, rows - 1) * M;  // the lane's row
  const bool live = lane < rows;
  double t[kSeg], v[kSeg];
  // pass q takes rows row0(q) .. row0(q) + kR - 1 (the last ones of a short
  // tile again where it has no further); opaque, so that the passes' offsets
  // are formed where they are used instead of held in registers
  const int sub = min(rsub, rows - 1);
  auto row0 = [&](int q) {
    int m = max(rows - kR, 0);
    asm volatile("" : "+s"(m));
    return min(q * kR, m);
  };
  auto load = [&](int e0) {  // columns e0 .. of the rows
    const double *p = src + min(e0 + ksub, nR - 1) + sub * nR;
#pragma unroll
    for (int q = 0; q < kSeg; q++) t[q] = p[row0(q) * nR];
  };
  auto turn = [&] {  // t[] to the lane's row v[]
#pragma unroll
    for (int q = 0; q < kSeg; q++) chunk[(row0(q) + sub) * kRowP + ksub] = t[q];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSeg; i++) v[i] = chunk[lane * kRowP + i];
    __syncthreads();
  };
  const int n = nR, sTop = (n - 1) / kSeg;
  double ym = ax.A03, y2 = 0.0;
  auto down = [&](int s, bool edge) {  // v[]: right-hand sides to y
    const int k0 = s * kSeg + 1;
#pragma unroll
    for (int i = 0; i < kSeg; i++) {
      if (!edge || k0 + i <= n) {
        y2 = ym;
        ym = eliminate(ax, st, k0 + i, edge, v[i], ym);
        v[i] = ym;
      }
    }
  };
  load(0);
  for (int s = 0; s <= sTop; s++) {
    turn();
    if (s < sTop) load((s + 1) * kSeg);
    if (s == 0 || s == sTop)
      down(s, true);
    else
      down(s, false);
    if (s < sTop && live) own[1 + s] = ym;
  }
  double cn = last_row(ax, y2, ym), c2 = cn;
  if (live) own[M - 1] = cn;
  for (int s = sTop; s >= 0; s--) {
    const int k0 = s * kSeg + 1;
    const bool edge = s == 0 || s == sTop;
    if (s < sTop) {
      turn();
      ym = s > 0 ? own[s] : ax.A03;
      if (edge)
        down(s, true);
      else
        down(s, false);
    }
    if (s > 0) load((s - 1) * kSeg);
    auto up = [&](bool edge) {
#pragma unroll
      for (int i = kSeg - 1; i >= 0; i--) {
        const int k = k0 + i;
        if (!edge || k <= n) {
          double u = st.u;
          if (edge && k <= kHead) u = ax.u[k];
          const double x = v[i] - u * cn;
          v[i] = x;
          c2 = cn;
          cn = x;
        }
      }
    };
    if (edge)
      up(true);
    else
      up(false);
#pragma unroll
    for (int i = 0; i < kSeg; i++) chunk[lane * kRowP + i] = v[i];
    __syncthreads();
    const int k = k0 + ksub;
#pragma unroll
    for (int q = 0; q < kSeg; q++) {
      const int row = row0(q) + sub;
      if (k <= n) dst[row * M + k] = chunk[row * kRowP + ksub];
    }
    __syncthreads();
  }
  if (live) own[0] = (ax.A03 - ax.A01 * cn) - ax.A02 * c2;
}

// The kick of the columns of f into out (f's layout), from the y kept by the
// elimination (k_kick_down: [j][k / kSeg - 1][r]) and the acceleration.  The
// back substitution goes through a column's coefficients from the last, and
// the points' targets, U + acc, rise with U: a lane evaluates each of its
// points as the four rows of its cell are there, last point first, so that
// the coefficients never leave the registers (dKeep: unless they are to be
// kept).  513x513x256: 261 us, 4.1 TB/s of read, kept and written columns.
// Dynamic LDS: U_Val.
template <bool kKeep>
__global__ void __launch_bounds__(64, 3)
k_kick_up(const double *__restrict__ f, double *__restrict__ out, double *__restrict__ dKeep,
          const double *__restrict__ kept, const double *__restrict__ U_Val,
          const double *__restrict__ acc, int nR, int nU, int nJ, int64_t ds, double Ulo, double Uhi,
          double start_v, double hinv_v, int lzmask, ThomasAxis ax) {
  extern __shared__ double Us[];
  const int lane = threadIdx.x;
  for (int u = lane; u < nU; u += 64) Us[u] = U_Val[u];
  __syncthreads();
  const int i0 = xcd_tile(blockIdx.x, gridDim.x) * 64, i = i0 + lane;
  if (i >= nR * nJ) return;  // no barriers below
  // the wave's columns may be of several slices: offsets from the first one's
  const int j0 = __builtin_amdgcn_readfirstlane(i0 / nR), K = (nU - 1) / kSegK;
  const int j = i / nR, r = i - j * nR;
  const Steady st = steady(ax, lane & lzmask);
  const uint32_t off = ((uint32_t)(j - j0) * nU * nR + r) * sizeof(double);
  const uint32_t offK = ((uint32_t)(j - j0) * K * nR + r) * sizeof(double);
  const uint32_t offD = ((uint32_t)(j - j0) * ds + r) * sizeof(double);
  char *fo = (char *)(out + (size_t)j0 * nU * nR);
  const uint32_t row = nR * sizeof(double);
  const double a = acc[r];
  // the next point to evaluate: row u, at byte at, cell pn (-1: none left),
  // offset py; uv: U of the point below it
  int u = nU - 1, pn;
  uint32_t at = off + u * row;
  double py = 0.0;
  for (; u >= 0 && Us[u] + a >= Uhi; u--, at -= row) *(double *)(fo + at) = 0.0;
  double uv = Us[max(u, 0)];
  auto next = [&] {
    const double newU = uv + a;
    pn = -1;
    if (u >= 0 && !(newU <= Ulo)) {
      split((newU - start_v) * hinv_v, pn, py);
      uv = Us[max(u - 1, 0)];
    }
  };
  next();
  double w0 = 0.0, w1 = 0.0, w2 = 0.0, w3 = 0.0;
  RowPtr dr(dKeep + (size_t)j0 * ds, ax.M - 1, nR);
  up_sweep<kSegK>(
      ax, st, f + (size_t)j0 * nU * nR - nR, nR, off,
      [&](int k) { return RowPtr(kept + (size_t)j0 * K * nR, k / kSegK - 1, nR).at(offK); },
      [&](int k, double c) {
        if constexpr (kKeep) {
          dr.at(offD) = c;
          dr.step(-1);
        }
        w3 = w2;
        w2 = w1;
        w1 = w0;
        w0 = c;
        if (k == ax.M - 1) w1 = w2 = c;  // row M of the last cell: weight 0, any finite row
        while (pn >= k) {
          *(double *)(fo + at) = kick_value(py, w0, w1, w2, w3);
          u--;
          at -= row;
          next();
        }
      });
  for (; u >= 0; u--, at -= row) *(double *)(fo + at) = 0.0;
}

void launch_stream_r(const Run &r, const double *src, double *dst, hipStream_t s) {
  hipLaunchKernelGGL(k_spline_r_stream, dim3((r.nU + 63) / 64 * r.nJ), dim3(64), 0, s, src, dst,
                     r.nR, r.nU, r.cs, 0, r.tr);
}

void launch_stream_v(const Run &r, const double *src, double *dst, hipStream_t s) {
  hipLaunchKernelGGL(k_spline_v_stream, dim3((r.nR + 2 + 63) / 64 * r.nJ), dim3(64), 0, s, src, dst,
                     r.nR, r.cs, 0, r.tv);
}

void launch_kick_up(const Run &r, double *out, double *dKeep, hipStream_t s) {
  hipLaunchKernelGGL(dKeep ? k_kick_up<true> : k_kick_up<false>, dim3((r.nR * r.nJ + 63) / 64), dim3(64), r.nU * sizeof(double), s,
                     r.f, out, dKeep, r.kept, r.U_Val, r.acc, r.nR, r.nU, r.nJ, r.cs, r.Ulo, r.Uhi,
                     r.start_v, r.hinv_v, 0, r.tv);
}

size_t kept_doubles(const Run &r) { return (size_t)r.nJ * ((r.nU - 1) / kSegK) * r.nR; }

}  // namespace vls
