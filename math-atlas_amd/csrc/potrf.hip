// Cholesky factorization and solve.
//
// Replaces ATL_dpotrf (AtlasBase/Clint/atlas-lp.base:332-360), the recursive
// ATL_dpotrfL (:909-968) / ATL_dpotrfU (:675-733) with their small closed
// forms (:809-908), and ATL_dpotrs (:969-1050).
//
// Same recursion as ATLAS: factor the leading half, TRSM the off-diagonal
// block, SYRK the trailing block, factor it.  The recursion stops at
// diagonal blocks of order <= DB, factored by one workgroup in registers,
// which also writes the inverse of its factor; the TRSMs of the recursion
// apply those inverses as GEMMs instead of inverting again.  The
// first non-positive pivot writes info to device memory; every later launch
// of the factorization reads that word and returns at once, which gives
// ATLAS's "stop at the first failure" without a host round trip.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "atlg_internal.hpp"
#include "tri_inv.hpp"

namespace atlg {
namespace {

constexpr int DB = kTrsmNB;    // diagonal block order

#ifndef ATLG_POTRF_RB
#define ATLG_POTRF_RB 384
#endif
constexpr long RB = ATLG_POTRF_RB;  // block width of the right-looking outer steps

// Factors the n x n (n <= DB) diagonal block at A and writes inv(L) of the
// block to Dinv (DB x DB, column-major, zeros above the diagonal).
// lower: A = L L^T from the lower triangle; else A = U^T U from the upper
// triangle, handled as L = U^T, so one algorithm serves both.  The other
// triangle of A is never read or written; order beyond n is padded with the
// identity.
//
// What bounds it: the chain of 128 pivots on one compute unit.  Everything is
// kept in the layout of the matrix core's accumulator: lane (n, k) =
// (l & 15, l >> 4) holds, of a 16x16 tile, row n and the columns 4 b + k in
// register b.  A register is then at once the 16x4 and the 4x16 operand of a
// 16x16x4 MFMA, so a block of four columns needs no data movement: its rows
// below are X' = X inv(L11)^T (one MFMA per tile, with the 4x4 inverse), and
// its share of the tile's other columns is one MFMA of X' with X'.
// Left-looking by 16-column steps d over the tiles in LDS; wave 0 runs the
// chain, eight waves have one tile each:
//   1. wave 0 factors tile (d, d) four columns at a time: the 4x4 block
//      through v_readlane, its factor by every lane alike, X' and
//      the tile's own update by MFMA, an identity tile carried along to the
//      tile's inverse.  Beside it the other waves subtract the earlier
//      columns' products from their tile of column d, and the one whose tile
//      is that inverse from the next diagonal tile;
//   2. they multiply their tile by the diagonal tile's inverse.
// The identity rides along below the block: its rows become L^-T, so the
// inverse costs MFMAs beside the factorization instead of a chain of its own,
// and column d always has eight tiles: block rows d + 1 .. 7 and identity
// rows 0 .. d.  A step is 5400 cycles of factor and 1500 of solve and next
// diagonal; the block with its inverse takes 28 us (80 us as 32-wide panels
// factored column by column through LDS, the inverse by doubling after it).
constexpr int PT = 16;              // tile order
constexpr int PTN = DB / PT;        // tiles per side
// Waves are dealt to the four SIMDs in turn: 0 is the chain's, waves 4 and 8
// only keep its SIMD free, and the tiles go to the others.
constexpr int PW_WAVES = 11, PW_THREADS = 64 * PW_WAVES;
// LDS pitches: lane (n, k) reads row n, column k of four: 4 n + k covers the
// bank pairs evenly
constexpr int PLD = DB + 4, YLD = PT + 4;

// 1/sqrt(d), d > 0: the hardware estimate (about 2^-23) and one third-order
// step; the products stay in range for subnormal d.
__device__ __forceinline__ double rsqrt3(double d) {
  const double y = __builtin_amdgcn_rsq(d);
  const double e = __builtin_fma(-(d * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}

__global__ void __launch_bounds__(PW_THREADS)
potf2_inv_kernel(int n, double* __restrict__ A, long lda, int lower, int* __restrict__ dinfo,
                 int info_off, double* __restrict__ Dinv) {
  typedef TriMfma<double> TM;
  typedef TM::acc_t acc_t;
  const int failed = *dinfo;  // an earlier block's failure: looked at once the loads are issued
  __shared__ double S[DB * PLD];        // A, then L below and on the diagonal, L^-T above it
  __shared__ double Y[PTN][PT * YLD];   // diagonal tiles of L^-T
  // the next diagonal tile, products of the columns before d taken off
  // (alternating: wave 0 reads one while the next is written)
  __shared__ double N[2][4][64];
  __shared__ int fail_sh;
  const int t = threadIdx.x, lane = t & 63, hw = __builtin_amdgcn_readfirstlane(t >> 6);
  const int w = hw % 4 == 0 ? (hw == 0 ? 0 : -1) : hw - hw / 4;  // 0: the chain, 1..8: tiles
  const int ln = lane & 15, lk = lane >> 4;
  const acc_t zero = {0, 0, 0, 0};
  // element (i, c), i >= c, of the block
  auto store = [&](int i, int c, double x) {
    if (i < n && c <= i) {
      if (lower) A[i + (size_t)c * lda] = x;
      else A[c + (size_t)i * lda] = x;
    }
  };
  // fill: the tiles on and below the diagonal, 36 of them, four per working
  // wave, all loads in flight
  if (w >= 0) {
    double v[4][4];
    int ti[4], tc[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      int u = w + (1 + PTN) * q, i = 0;
      while (u > i) u -= ++i;
      ti[q] = i;
      tc[q] = u;
      const int gi = PT * i + ln;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const int c = PT * u + 4 * b + lk;
        v[q][b] = gi == c ? 1.0 : 0.0;
        if (gi < n && c <= gi) v[q][b] = lower ? A[gi + (size_t)c * lda] : A[c + (size_t)gi * lda];
      }
    }
    // the inverse's tiles above the diagonal
    if (failed == 0)
    for (int u = w; u < PTN * (PTN - 1) / 2; u += 1 + PTN) {
      int c = 1, i = u;
      while (i >= c) i -= c++;
      double* z = Dinv + PT * i + ln + (size_t)(PT * c + lk) * DB;
#pragma unroll
      for (int b = 0; b < 4; b++) z[4 * b * DB] = 0.0;
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int b = 0; b < 4; b++)
        S[(PT * ti[q] + ln) * PLD + PT * tc[q] + 4 * b + lk] = v[q][b];
  }
  if (failed != 0) return;
  if (t == 0) fail_sh = -1;
  __syncthreads();

  acc_t T = zero;  // wave 0: the diagonal tile, the others: their tile
  double keep[4] = {0, 0, 0, 0};  // a finished tile on its way to memory
  if (w == 0) {
#pragma unroll
    for (int b = 0; b < 4; b++) T[b] = S[ln * PLD + 4 * b + lk];
  }
  for (int d = 0; d < PTN; d++) {
    const int c0 = PT * d;
    const double* row_d = S + (c0 + ln) * PLD + lk;  // tile row d, this lane's entries
    // this wave's tile: block row `rt` (L) or identity row `rt` (L^-T)
    const bool inv = w >= PTN - d;  // w = 1 .. 7 - d: block rows, then identity rows 0 .. d
    const int rt = inv ? w - (PTN - d) : d + w;
    if (w == 0) {
      int bad = -1;  // first non-positive pivot of the tile
      acc_t Z;       // the identity on its way to the transposed inverse
#pragma unroll
      for (int b = 0; b < 4; b++) Z[b] = ln == 4 * b + lk ? 1.0 : 0.0;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        double a[4][4], r[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int i = j; i < 4; i++) a[i][j] = tri_lane(T[b], 16 * j + 4 * b + i);
        bool pos = true;
#pragma unroll
        for (int j = 0; j < 4; j++) {
          if (!(a[j][j] > 0.0) && pos) {
            pos = false;
            bad = 4 * b + j;
          }
          r[j] = rsqrt3(a[j][j]);
          a[j][j] *= r[j];
#pragma unroll
          for (int i = j + 1; i < 4; i++) a[i][j] *= r[j];
#pragma unroll
          for (int c = j + 1; c < 4; c++)
#pragma unroll
            for (int i = c; i < 4; i++) a[i][c] -= a[i][j] * a[c][j];
        }
        bad = __builtin_amdgcn_readfirstlane(bad);
        if (bad >= 0) {  // the block's columns before it are part of the leading factor
          if (lane == 0) {
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
              for (int c = 0; c < i; c++)
                if (4 * b + c < bad) S[(c0 + 4 * b + i) * PLD + c0 + 4 * b + c] = a[i][c];
#pragma unroll
            for (int c = 0; c < 3; c++)
              if (4 * b + c < bad) S[(c0 + 4 * b + c) * PLD + c0 + 4 * b + c] = a[c][c];
          }
          break;
        }
        // inv(L11): every lane solves for the column lk, and keeps row ln of it
        double wc[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          double sum = lk == i ? 1.0 : 0.0;
#pragma unroll
          for (int c = 0; c < i; c++) sum -= a[i][c] * wc[c];
          wc[i] = sum * r[i];
        }
        double wo = ln < 4 ? wc[0] : 0.0;
#pragma unroll
        for (int i = 1; i < 4; i++) wo = ln == i ? wc[i] : wo;
        const acc_t x = TM::op(wo, T[b], zero);
        const acc_t z = TM::op(wo, Z[b], zero);
        __builtin_amdgcn_sched_barrier(0);  // stores in the shadow of the MFMAs
        if (lane == 0) {
#pragma unroll
          for (int i = 0; i < 4; i++)
#pragma unroll
            for (int c = 0; c <= i; c++) S[(c0 + 4 * b + i) * PLD + c0 + 4 * b + c] = a[i][c];
        }
        __builtin_amdgcn_sched_barrier(0);
        const double xm = ln >= 4 * b + 4 ? x[0] : 0.0;
        if (b < 3) {
          T = TM::op(-xm, xm, T);
          Z = TM::op(-xm, z[0], Z);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (ln >= 4 * b + 4) S[(c0 + ln) * PLD + c0 + 4 * b + lk] = xm;
        Y[d][ln * YLD + 4 * b + lk] = z[0];
      }
      if (lane == 0 && bad >= 0) fail_sh = c0 + bad;
    } else if (w > 0) {
      // T = A(rt, d) - sum over e < d of X(rt, e) X(d, e)^T; identity rows
      // start at their own column
      const double* row = S + (PT * rt + ln) * PLD + lk;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const double x = row[c0 + 4 * b];
        T[b] = inv ? (rt == d && ln == 4 * b + lk ? 1.0 : 0.0) : x;
      }
      acc_t T2 = zero;
      for (int e = inv ? rt : 0; e < d; e++) {
        const double* x2 = inv && e == rt ? &Y[rt][ln * YLD + lk] : row + PT * e;
        double p[4], q[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
          p[b] = -row_d[PT * e + 4 * b];
          q[b] = x2[4 * b];
        }
        T = TM::op(p[0], q[0], T);
        T2 = TM::op(p[1], q[1], T2);
        T = TM::op(p[2], q[2], T);
        T2 = TM::op(p[3], q[3], T2);
      }
#pragma unroll
      for (int b = 0; b < 4; b++) T[b] += T2[b];
      if (w == PTN && d + 1 < PTN) {
        // identity row d has no products yet: this wave does the next
        // diagonal tile's
        const double* row_n = row_d + PT * PLD;
        acc_t U = zero, U2 = zero;
#pragma unroll
        for (int b = 0; b < 4; b++) U[b] = row_n[c0 + PT + 4 * b];
        for (int e = 0; e < d; e++) {
          double p[4];
#pragma unroll
          for (int b = 0; b < 4; b++) p[b] = row_n[PT * e + 4 * b];
          U = TM::op(-p[0], p[0], U);
          U2 = TM::op(-p[1], p[1], U2);
          U = TM::op(-p[2], p[2], U);
          U2 = TM::op(-p[3], p[3], U2);
        }
#pragma unroll
        for (int b = 0; b < 4; b++) N[d & 1][b][lane] = U[b] + U2[b];
      }
    }
    lds_barrier();
    const int fail = fail_sh;
    if (fail >= 0) {
      // the factor of the leading minor (all rows and columns before the
      // failing one) is complete in memory; of the rows from there on, this
      // tile's earlier columns as far as they got, the rest as it was
      if (w == 0) {
#pragma unroll
        for (int b = 0; b < 4; b++)
          if (c0 + 4 * b + lk < fail) store(c0 + ln, c0 + 4 * b + lk, row_d[c0 + 4 * b]);
        if (t == 0) *dinfo = info_off + fail + 1;
      }
      return;
    }
    if (w > 0 && w < PTN) {  // (the last wave's tile is the inverse itself)
      const double* y = &Y[d][lk * YLD + ln];
      double p[4];
#pragma unroll
      for (int b = 0; b < 4; b++) p[b] = y[4 * b * YLD];
      acc_t X = TM::op(p[0], T[0], zero), X2 = TM::op(p[1], T[1], zero);
      X = TM::op(p[2], T[2], X);
      X2 = TM::op(p[3], T[3], X2);
#pragma unroll
      for (int b = 0; b < 4; b++) {
        keep[b] = X[b] + X2[b];
        S[(PT * rt + ln) * PLD + c0 + 4 * b + lk] = keep[b];
      }
    }
    lds_barrier();
    // results to memory, off the chain
    if (w == PTN) {
#pragma unroll
      for (int b = 0; b < 4; b++) {
        store(c0 + ln, c0 + 4 * b + lk, row_d[c0 + 4 * b]);
        keep[b] = Y[d][ln * YLD + 4 * b + lk];
      }
    }
    if (w > 0) {
      if (!inv) {
#pragma unroll
        for (int b = 0; b < 4; b++) store(PT * rt + ln, c0 + 4 * b + lk, keep[b]);
      } else {  // inv(L)(i, c) = L^-T(c, i)
        double* z = Dinv + c0 + lk + (size_t)(PT * rt + ln) * DB;
#pragma unroll
        for (int b = 0; b < 4; b++) z[4 * b] = keep[b];
      }
    }
    if (w == 0 && d + 1 < PTN) {  // column d's product from the next diagonal tile
      const double* row_n = row_d + PT * PLD + c0;
      double p[4];
      acc_t T2 = zero;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        p[b] = row_n[4 * b];
        T[b] = N[d & 1][b][lane];
      }
      T = TM::op(-p[0], p[0], T);
      T2 = TM::op(-p[1], p[1], T2);
      T = TM::op(-p[2], p[2], T);
      T2 = TM::op(-p[3], p[3], T2);
#pragma unroll
      for (int b = 0; b < 4; b++) T[b] += T2[b];
    }
  }
}

void potrf_rec(hipStream_t s, bool lower, long N, double* A, long lda, int* dinfo, int off,
               double* W, int* status) {
  if (N <= 0) return;
  if (N <= DB) {
    hipLaunchKernelGGL(potf2_inv_kernel, dim3(1), dim3(PW_THREADS), 0, s, (int)N, A, lda,
                       lower ? 1 : 0, dinfo, off, W + (size_t)(off / DB) * DB * DB);
    ATLG_LAUNCHED();
    return;
  }
  // Right-looking by RB-column blocks (then ATLAS's halving inside a block):
  // each step's update is one large SYRK instead of the many small GEMMs of
  // a halving recursion over the whole order.
  long nl = (N > 2 * RB) ? RB : ((N / 2) / DB) * DB;
  if (nl < DB) nl = DB;
  const long nr = N - nl;
  potrf_rec(s, lower, nl, A, lda, dinfo, off, W, status);
  double* A22 = A + nl + nl * lda;
  const double* Winv = W + (size_t)(off / DB) * DB * DB;  // inverses of this node's A11
  if (lower) {
    // A21 <- A21 L11^-T: op(A) = L11^T, whose diagonal-block inverses are
    // the transposes of the stored inv(L_bb)
    double* A21 = A + nl;
    trsm(s, kRight, kLower, kTrans, kNonUnit, nr, nl, 1.0, A, lda, A21, lda, dinfo, Winv, 1,
         {status, dinfo});
    gemm(s, kNoTrans, kTrans, nr, nr, nl, -1.0, A21, lda, A21, lda, 1.0, A22, lda, 1, dinfo);
  } else {
    // A12 <- U11^-T A12: op(A) = U11^T = L11, inverses stored as is
    double* A12 = A + nl * lda;
    trsm(s, kLeft, kUpper, kTrans, kNonUnit, nl, nr, 1.0, A, lda, A12, lda, dinfo, Winv, 0,
         {status, dinfo});
    gemm(s, kTrans, kNoTrans, nr, nr, nl, -1.0, A12, lda, A12, lda, 1.0, A22, lda, 2, dinfo);
  }
  potrf_rec(s, lower, nr, A22, lda, dinfo, off + (int)nl, W, status);
}

// Look-ahead (1) or plain right-looking steps (0).  At N = 16384 the
// look-ahead with the panels on 32 compute units and the SYRKs on the rest
// takes 55 ms against 65 ms for plain steps; on a shared device (no masked
// streams) both took 65 ms: the 128-block leaves, which need 156 KB of LDS,
// wait for a compute unit free of SYRK workgroups.
// Without masked streams: grid cap of the look-ahead's trailing SYRK
// (workgroups).
#ifndef ATLG_CHOL_LOOKAHEAD
#define ATLG_CHOL_LOOKAHEAD 1
#endif
#ifndef ATLG_CHOL_CAP
#define ATLG_CHOL_CAP 384
#endif
// Compute units of the panel stream when the look-ahead runs panels and
// updates on a CU-masked stream pair (0: both share the device).
#ifndef ATLG_CHOL_PANEL_CUS
#define ATLG_CHOL_PANEL_CUS 32
#endif
constexpr long kCholLaMin = 2048;

// Look-ahead step width where `rem` columns are left (ATLG_CHOL_STEP when
// set; multiples of 128): the chain of diagonal blocks is the longer path at
// the end, the trailing SYRK, more efficient the deeper it is, before.
// Measured on MI355X with one width throughout (ms, 28 us leaves): N=2048
// 128: 1.07, 256: 1.06, 384: 1.11; N=4096 128: 2.38, 256: 2.18, 384: 2.21,
// 512: 2.48; N=8192 128: 8.03, 256: 6.82, 384: 6.50, 512: 6.57; N=16384
// 256: 33.6, 384: 30.8, 512: 30.4; 16 panel units instead of 32 the same, 64
// 4-12% slower.
#ifndef ATLG_CHOL_STEP
#define ATLG_CHOL_STEP 0
#endif
inline long chol_step(long rem) {
  if (ATLG_CHOL_STEP > 0) return ATLG_CHOL_STEP;
  return rem < 4608 ? 256 : (rem < 12288 ? 384 : 512);
}

// Whether step k's panel solve (rest x nb1, after the diagonal block of nb1
// columns) goes to the update side.  Per step, the update side runs the
// trailing SYRK (U, at ATLG_CHOL_UPD_TFLOPS), the panel side the leaves
// (ATLG_CHOL_LEAF_US per 128 columns, with the small solves and updates
// between them) and, when narrow, the solve on its ATLG_CHOL_PANEL_CUS units;
// wide, it runs after U on the update side, whose units would else wait.
// (N = 2048 .. 16384 within 2% for 30 to 100 us and 40 to 60 TFLOP/s.)
#ifndef ATLG_CHOL_UPD_TFLOPS
#define ATLG_CHOL_UPD_TFLOPS 50.0
#endif
#ifndef ATLG_CHOL_LEAF_US
#define ATLG_CHOL_LEAF_US 35.0
#endif
inline bool chol_solve_wide(long rest, long nb1) {
  if (rest <= 0) return false;
  const double upd_rate = ATLG_CHOL_UPD_TFLOPS * 1e12,
               panel_rate = upd_rate * ATLG_CHOL_PANEL_CUS / (256.0 - ATLG_CHOL_PANEL_CUS);
  const double r = (double)rest, b = (double)nb1;
  return r * r * b / upd_rate <
         b / 128.0 * ATLG_CHOL_LEAF_US * 1e-6 + 2.0 * r * b * b / panel_rate;
}

// Right-looking Cholesky by chol_step()-column blocks with one step of
// look-ahead:
// while the caller's stream applies step k's SYRK to the columns right of
// block k+1, the auxiliary stream factors block k+1 (updated first) and
// solves its panel.  lower: A = L L^T, panel L21 = A21 L11^-T, update
// A22 -= L21 L21^T; upper: A = U^T U, U12 = U11^-T A12, A22 -= U12^T U12.
// `status`: the failure word of the caller's stream.
void potrf_lookahead(hipStream_t s0, bool lower, long N, double* A, long lda, int* dinfo,
                     double* W, int* status) {
  const auto lock = aux_lock();
  hipStream_t s1 = aux_stream();
  hipEvent_t e_upd = aux_event(0), e_panel = aux_event(1);
  // with a CU-masked pair the 128-block leaves (156 KB of LDS) never wait
  // for a compute unit free of SYRK workgroups
  hipStream_t caller = s0, sp = nullptr, sg = nullptr;
  const bool split =
      ATLG_CHOL_PANEL_CUS > 0 && split_streams(ATLG_CHOL_PANEL_CUS, caller, &sp, &sg);
  if (split) {
    ATLG_HIP(hipEventRecord(aux_event(2), caller));
    ATLG_HIP(hipStreamWaitEvent(sg, aux_event(2), 0));
    ATLG_HIP(hipStreamWaitEvent(sp, aux_event(2), 0));
    s0 = sg;
    s1 = sp;
  }
  auto at = [&](long i, long j) { return A + i + j * lda; };
  // the panel of the block at k (kb columns) below/right of it, rows/cols r
  auto panel_ptr = [&](long k, long kb) { return lower ? at(k + kb, k) : at(k, k + kb); };
  auto solve_panel = [&](hipStream_t s, long k, long kb, long r) {
    if (r <= 0) return;
    const double* Winv = W + (size_t)(k / DB) * DB * DB;
    if (lower)
      trsm(s, kRight, kLower, kTrans, kNonUnit, r, kb, 1.0, at(k, k), lda, panel_ptr(k, kb), lda,
           dinfo, Winv, 1, {status, dinfo});
    else
      trsm(s, kLeft, kUpper, kTrans, kNonUnit, kb, r, 1.0, at(k, k), lda, panel_ptr(k, kb), lda,
           dinfo, Winv, 0, {status, dinfo});
  };
  // A(c0.., c0..c0+nc) -= P_c P_c^T restricted to the stored triangle, P the
  // panel of block k (kb wide) from its row/column c0 on; m rows/cols in all
  auto update = [&](hipStream_t s, long k, long kb, long c0, long m, long nc, int cap) {
    if (m <= 0 || nc <= 0) return;
    if (lower) {
      const double* P = at(c0, k);
      gemm(s, kNoTrans, kTrans, m, nc, kb, -1.0, P, lda, P, lda, 1.0, at(c0, c0), lda, 1, dinfo,
           cap);
    } else {
      const double* P = at(k, c0);
      gemm(s, kTrans, kNoTrans, nc, m, kb, -1.0, P, lda, P, lda, 1.0, at(c0, c0), lda, 2, dinfo,
           cap);
    }
  };
  // the off-diagonal part of block column c0 (nc wide, r rows/columns past
  // it) minus the product of block k's panel rows
  auto update_col = [&](hipStream_t s, long k, long kb, long c0, long nc, long r) {
    if (r <= 0) return;
    if (lower)
      gemm(s, kNoTrans, kTrans, r, nc, kb, -1.0, at(c0 + nc, k), lda, at(c0, k), lda, 1.0,
           at(c0 + nc, c0), lda, 0, dinfo);
    else
      gemm(s, kTrans, kNoTrans, nc, r, kb, -1.0, at(k, c0), lda, at(k, c0 + nc), lda, 1.0,
           at(c0, c0 + nc), lda, 0, dinfo);
  };
  hipEvent_t e_col = aux_event(4);
  auto width = [&](long k) { return std::min(chol_step(N - k), N - k); };
  const long kb0 = width(0);
  potrf_rec(s0, lower, kb0, A, lda, dinfo, 0, W, status);
  solve_panel(s0, 0, kb0, N - kb0);
  for (long k0 = 0; k0 + width(k0) < N; k0 += width(k0)) {
    const long kb = width(k0), k1 = k0 + kb, nb1 = width(k1);
    const long rest = N - k1 - nb1;
    // block k+1 first, then the rest of step k's update, beside which the
    // auxiliary stream factors block k+1 and solves its panel: its diagonal
    // block alone (all the leaf needs; N=4096 2.26 -> 2.18 ms, 8192 the same),
    // then the rest of its block column (what the panel solve needs)
    update(s0, k0, kb, k1, nb1, nb1, 0);
    ATLG_HIP(hipEventRecord(e_upd, s0));
    update_col(s0, k0, kb, k1, nb1, rest);
    ATLG_HIP(hipEventRecord(e_col, s0));
    update(s0, k0, kb, k1 + nb1, rest, rest, split ? 0 : ATLG_CHOL_CAP);
    ATLG_HIP(hipStreamWaitEvent(s1, e_upd, 0));
    potrf_rec(s1, lower, nb1, at(k1, k1), lda, dinfo, (int)k1, W, status);
    // The panel solve is a GEMM-shaped TRSM of rest x nb1: on the panel
    // units while the trailing update keeps the others busy, on the update
    // side once that update is the shorter path (its units would wait).
    const bool solve_wide = split && chol_solve_wide(rest, nb1);
    if (!solve_wide) {
      ATLG_HIP(hipStreamWaitEvent(s1, e_col, 0));
      solve_panel(s1, k1, nb1, rest);
    }
    ATLG_HIP(hipEventRecord(e_panel, s1));
    ATLG_HIP(hipStreamWaitEvent(s0, e_panel, 0));
    if (solve_wide) solve_panel(s0, k1, nb1, rest);
  }
  if (split) {  // every panel was joined into s0 above
    ATLG_HIP(hipEventRecord(aux_event(3), s0));
    ATLG_HIP(hipStreamWaitEvent(caller, aux_event(3), 0));
  }
}

}  // namespace

void potrf(hipStream_t s, int uplo, long N, double* A, long lda, int* dinfo) {
  const bool lookahead = ATLG_CHOL_LOOKAHEAD && N >= kCholLaMin;
  if (lookahead) refuse_capture(s, "potrf");
  set_int(s, dinfo, 0);
  if (N <= 0) return;
  const long nblk = (N + DB - 1) / DB;
  double* W = static_cast<double*>(scratch(s, kSlotFactInv, sizeof(double) * nblk * DB * DB));
  int* status = status_word(s);
  if (lookahead)
    potrf_lookahead(s, uplo == kLower, N, A, lda, dinfo, W, status);
  else
    potrf_rec(s, uplo == kLower, N, A, lda, dinfo, 0, W, status);
}

void potrs(hipStream_t s, int uplo, long N, long NRHS, const double* A, long lda, double* B,
           long ldb) {
  if (N == 0 || NRHS == 0) return;
  if (uplo == kUpper) {
    trsm(s, kLeft, kUpper, kTrans, kNonUnit, N, NRHS, 1.0, A, lda, B, ldb);
    trsm(s, kLeft, kUpper, kNoTrans, kNonUnit, N, NRHS, 1.0, A, lda, B, ldb);
  } else {
    trsm(s, kLeft, kLower, kNoTrans, kNonUnit, N, NRHS, 1.0, A, lda, B, ldb);
    trsm(s, kLeft, kLower, kTrans, kNonUnit, N, NRHS, 1.0, A, lda, B, ldb);
  }
}

}  // namespace atlg
