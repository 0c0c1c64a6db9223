// Triangular solve with many right-hand sides on the matrix cores (FP64, and
// FP32 for the single-precision factorization of the mixed solver).
//
// Replaces ATL_dtrsm (AtlasBase/Clint/trsm-micro.base:200-420: recursive
// halving trsm_recL/R, then iptrsm/trsmL_LNUT/utrsm with reciprocal
// diagonals, :550-1700, and the nano-kernels of
// AtlasBase/Students/trsm-nano.base:297-344).  ATLAS keeps reciprocal
// diagonals and runs everything off the diagonal as amm GEMM; this version
// goes one step further:
//   1. one launch inverts every NB x NB diagonal block of op(A) in LDS
//      (one workgroup per block, by 16x16 tiles), writing full NB x NB
//      inverses;
//   2. a recursive halving driver (the same split as trsm_recL/R) updates
//      with large GEMMs down to an order that one launch solves with these
//      inverses (trsv_xcd.hpp), or, for very many right-hand sides, to single
//      blocks, whose inverses apply as in-place GEMMs.
// All flops but the small inversions run on the 16x16x4 MFMA GEMM.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <map>
#include <mutex>
#include <type_traits>

#include "atlg_internal.hpp"
#include "tri_inv.hpp"

namespace atlg {
namespace {

constexpr int NB = kTrsmNB;    // diagonal block order (<= GEMM tile edge)

// Element (i, j) of op(A).
template <class S>
__device__ inline S opa(const S* A, long lda, bool trans, long i, long j) {
  return trans ? A[j + i * lda] : A[i + j * lda];
}

// Inverts the diagonal blocks of op(A) (order na).  Block b covers rows and
// columns [b*NB, b*NB + nbb).  An upper-triangular op(A) block U is handled
// as the lower-triangular J U J (J = order reversal), so one lower inversion
// serves all cases.  Output: Dinv + b*NB*NB, column-major, ld NB, zeros
// outside the triangle; Unit diagonals are never read.  NT is the order held
// in LDS: NB for the general case; 32 or 64 when na <= NT (one block), which
// then writes only the leading NT x NT part of the block (the solves read the
// leading na x na part) and needs a fraction of the LDS, so the launch fits
// beside GEMM workgroups on a busy device.
//
// Latency-bound: one workgroup per block, a wave per row of 16x16 tiles.
// Tiles are kept in the accumulator's layout (lane (n, k) = (l & 15, l >> 4)
// holds row n, columns 4 b + k in register b), in which a register is also an
// operand of the 16x16x4 MFMA.  The waves first invert the diagonal tiles,
// four columns at a time, each its own, by carrying the identity to L^-T;
// then each computes its row of L^-T tile by tile from its own results, the
// tiles of L in LDS and the diagonal inverses, with no barrier between the
// waves.  The 64 blocks of an order-8192 triangle take 20 us; a solve of
// order 128 went from 38 to 28 us (8x8 register inverses and five doubling
// levels with four barriers each before).
template <class R, int NT>
__global__ void __launch_bounds__(4 * NT)
trtri_diag_kernel(int na, const R* __restrict__ A, long lda, int trans, int lower, int unit,
                  R* __restrict__ Dinv, const int* __restrict__ skip) {
  typedef TriMfma<R> M;
  typedef typename M::acc_t acc_t;
  constexpr int TS = 16, TN = NT / TS, LD = NT + 4, YLD = TS + 4;
  constexpr int TILES = TN * (TN + 1) / 2, PER = (TILES + TN - 1) / TN;
  __shared__ R S[NT * LD];        // L below and on the diagonal, L^-T above it
  __shared__ R Y[TN][TS * YLD];   // diagonal tiles of L^-T
  const int bk = blockIdx.x, t = threadIdx.x;
  const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int ln = lane & 15, lk = lane >> 4;
  // as an operand's row (a result's column), lane ln stands for column pm
  const int pm = std::is_same<R, double>::value ? ln : 4 * (ln & 3) + (ln >> 2);
  const acc_t zero = {0, 0, 0, 0};
  const long o = (long)bk * NB;
  const int n = (int)min((long)NT, na - o);
  const bool tr = trans != 0;
  const bool skipped = skip && *skip;
  {
    R v[PER][4];
#pragma unroll
    for (int q = 0; q < PER; q++) {
      int u = w + TN * q, ti = 0;
      while (u > ti) u -= ++ti;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const int i = TS * ti + ln, j = TS * u + 4 * b + lk;
        R x = i == j ? R(1) : R(0);
        if (i >= j && i < n && !(i == j && unit))
          x = lower ? opa(A, lda, tr, o + i, o + j) : opa(A, lda, tr, o + n - 1 - i, o + n - 1 - j);
        v[q][b] = x;
      }
    }
    if (skipped) return;
#pragma unroll
    for (int q = 0; q < PER; q++) {
      int u = w + TN * q, ti = 0;
      const bool in = u < TILES;
      while (u > ti) u -= ++ti;
      if (in) {
#pragma unroll
        for (int b = 0; b < 4; b++) S[(TS * ti + ln) * LD + TS * u + 4 * b + lk] = v[q][b];
      }
    }
  }
  R* D = Dinv + (size_t)bk * NB * NB;
  for (int idx = t; idx < NT * NT; idx += 4 * NT) {
    const int i = idx % NT, j = idx / NT;
    if (!(lower ? (i >= j && i < n) : (i <= j && j < n))) D[i + (size_t)j * NB] = R(0);
  }
  // inv(L)(i, j) to its place
  auto put = [&](int i, int j, R x) {
    if (i >= j && i < n) D[lower ? i + (size_t)j * NB : n - 1 - i + (size_t)(n - 1 - j) * NB] = x;
  };
  lds_barrier();
  {  // the diagonal tile of this wave's row
    const R* row = S + (TS * w + ln) * LD + TS * w + lk;
    const R* rop = S + (TS * w + pm) * LD + TS * w + lk;
    acc_t Z;
#pragma unroll
    for (int b = 0; b < 4; b++) Z[b] = ln == 4 * b + lk ? R(1) : R(0);
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const double x = (double)row[4 * b];
      R a[4][4], wc[4];
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = j; i < 4; i++) a[i][j] = (R)tri_lane(x, 16 * j + 4 * b + i);
      // the 4x4 block's inverse: every lane solves for column lk and keeps
      // the row its operand lane stands for
#pragma unroll
      for (int i = 0; i < 4; i++) {
        R sum = lk == i ? R(1) : R(0);
#pragma unroll
        for (int c = 0; c < i; c++) sum -= a[i][c] * wc[c];
        wc[i] = sum * (R(1) / a[i][i]);
      }
      R wo = pm == 0 ? wc[0] : R(0);
#pragma unroll
      for (int i = 1; i < 4; i++) wo = pm == i ? wc[i] : wo;
      const R z = M::op(wo, Z[b], zero)[0];
      if (b < 3) Z = M::op(pm >= 4 * b + 4 ? -rop[4 * b] : R(0), z, Z);
      Z[b] = z;
      Y[w][ln * YLD + 4 * b + lk] = z;
      put(TS * w + 4 * b + lk, TS * w + ln, z);
    }
  }
  lds_barrier();
  // row w of L^-T: tile d = -(sum over e < d of its tile e times L(d, e)^T)
  // times the inverse of diagonal tile d
  R* mine = S + (TS * w + ln) * LD + lk;
  for (int d = w + 1; d < TN; d++) {
    const R* ld = S + (TS * d + pm) * LD + lk;
    acc_t T = zero, T2 = zero;
    for (int e = w; e < d; e++) {
      const R* x2 = e == w ? &Y[w][ln * YLD + lk] : mine + TS * e;
      R p[4], q[4];
#pragma unroll
      for (int b = 0; b < 4; b++) {
        p[b] = -ld[TS * e + 4 * b];
        q[b] = x2[4 * b];
      }
      T = M::op(p[0], q[0], T);
      T2 = M::op(p[1], q[1], T2);
      T = M::op(p[2], q[2], T);
      T2 = M::op(p[3], q[3], T2);
    }
    const R* y = &Y[d][lk * YLD + pm];
    acc_t X = zero, X2 = zero;
#pragma unroll
    for (int b = 0; b < 4; b += 2) {
      X = M::op(y[4 * b * YLD], T[b] + T2[b], X);
      X2 = M::op(y[4 * (b + 1) * YLD], T[b + 1] + T2[b + 1], X2);
    }
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const R x = X[b] + X2[b];
      mine[TS * d + 4 * b] = x;
      put(TS * d + 4 * b + lk, TS * w + ln, x);
    }
  }
}

constexpr long kSvSpin = 1L << 22;         // default polls (round trips) before giving up

__device__ inline int ld_flag(const int* p) {
  return __hip_atomic_load(const_cast<int*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_flag(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

#include "trsv_xcd.hpp"

template <class S>
struct Ctx {
  hipStream_t s;
  bool left, lower_eff, trans;
  const S* A;
  long lda;
  S* B;
  long ldb;
  long M, N;   // B is M x N
  const S* Dinv;
  int dtrans;  // kTrans when Dinv holds the transposes of inv(op(A)_bb)
  const int* skip;
  WaitReport rep;
  unsigned char* fixed;  // exchange memory of the one-launch solves, or nullptr: the stream's own
};

// op(A)[i0:, j0:] as a GEMM operand: pointer and transpose flag.
template <class S>
inline void opa_block(const Ctx<S>& c, long i0, long j0, const S** p, int* t) {
  if (!c.trans) {
    *p = c.A + i0 + j0 * c.lda;
    *t = kNoTrans;
  } else {
    *p = c.A + j0 + i0 * c.lda;
    *t = kTrans;
  }
}

long split(long n) {
  long n1 = ((n / 2) / NB) * NB;
  return n1 > 0 ? n1 : NB;
}

// Solves on rows/cols [r0, r0+n) of op(A) with scale alpha.
template <class S>
void solve(const Ctx<S>& c, long r0, long n, S alpha) {
  const S one = S(1), mone = S(-1), zero = S(0);
  if (n <= NB) {
    const S* D = c.Dinv + (size_t)(r0 / NB) * NB * NB;
    if (c.left) {
      S* Bb = c.B + r0;
      gemm<S>(c.s, c.dtrans, kNoTrans, n, c.N, n, alpha, D, NB, Bb, c.ldb, zero, Bb, c.ldb, 0,
              c.skip);
    } else {
      S* Bb = c.B + r0 * c.ldb;
      gemm<S>(c.s, kNoTrans, c.dtrans, c.M, n, n, alpha, Bb, c.ldb, D, NB, zero, Bb, c.ldb, 0,
              c.skip);
    }
    return;
  }
  // X op(A) = B is op(A)^T X^T = B^T
  const long rhs = c.left ? c.N : c.M;
  if (n <= tx_order(rhs) &&
      trsv_one_launch<S>(c.s, c.lower_eff == c.left, c.trans == c.left, n, rhs, alpha,
                         c.A + r0 + r0 * c.lda, c.lda, c.Dinv + (size_t)(r0 / NB) * NB * NB,
                         (c.dtrans == kTrans) == c.left, c.B + (c.left ? r0 : r0 * c.ldb),
                         c.left ? 1 : c.ldb, c.left ? c.ldb : 1, c.skip, c.rep, c.fixed))
    return;
  const long n1 = split(n), n2 = n - n1;
  const S* Ap;
  int ta;
  if (c.left) {
    S* B1 = c.B + r0;
    S* B2 = c.B + r0 + n1;
    if (c.lower_eff) {
      // [L11 0; L21 L22]: X1 first, then B2 <- alpha*B2 - L21*X1
      solve(c, r0, n1, alpha);
      opa_block(c, r0 + n1, r0, &Ap, &ta);
      gemm<S>(c.s, ta, kNoTrans, n2, c.N, n1, mone, Ap, c.lda, B1, c.ldb, alpha, B2, c.ldb, 0,
           c.skip);
      solve(c, r0 + n1, n2, one);
    } else {
      // [U11 U12; 0 U22]: X2 first, then B1 <- alpha*B1 - U12*X2
      solve(c, r0 + n1, n2, alpha);
      opa_block(c, r0, r0 + n1, &Ap, &ta);
      gemm<S>(c.s, ta, kNoTrans, n1, c.N, n2, mone, Ap, c.lda, B2, c.ldb, alpha, B1, c.ldb, 0,
           c.skip);
      solve(c, r0, n1, one);
    }
  } else {
    S* B1 = c.B + r0 * c.ldb;
    S* B2 = c.B + (r0 + n1) * c.ldb;
    if (c.lower_eff) {
      // X [L11 0; L21 L22] = B: X2 first, then B1 <- alpha*B1 - X2*L21
      solve(c, r0 + n1, n2, alpha);
      opa_block(c, r0 + n1, r0, &Ap, &ta);
      gemm<S>(c.s, kNoTrans, ta, c.M, n1, n2, mone, B2, c.ldb, Ap, c.lda, alpha, B1, c.ldb, 0,
           c.skip);
      solve(c, r0, n1, one);
    } else {
      // X [U11 U12; 0 U22] = B: X1 first, then B2 <- alpha*B2 - X1*U12
      solve(c, r0, n1, alpha);
      opa_block(c, r0, r0 + n1, &Ap, &ta);
      gemm<S>(c.s, kNoTrans, ta, c.M, n2, n1, mone, B1, c.ldb, Ap, c.lda, alpha, B2, c.ldb, 0,
           c.skip);
      solve(c, r0 + n1, n2, one);
    }
  }
}

// ---- one right-hand side, long triangle: one sync-free cooperative launch ---
//
// op(A) = A (Left, NoTrans).  The rows are cut
// into 128-row blocks; workgroup w solves the blocks w, w+G, w+2G, ... in
// solve order (top down for lower, bottom up for upper).  For its block it
// accumulates A(block, q) x_q over the earlier blocks q as soon as each x_q
// is published (a ready flag per block), then applies the block's inverse
// from tri_inverse_blocks and publishes x.  The smallest unfinished block
// always has all its inputs, so the launch cannot deadlock while every
// workgroup is resident (cooperative launch); the waits are bounded anyway:
// an overrun sets the launch's error word, which makes every workgroup
// leave, and ORs ATLG_FAIL_TRSV into the stream's failure word.  Published x and the flags go through
// agent-scope (coherence point) atomic loads and stores, as in getrf's
// cooperative panel.
constexpr int SV_T = 256;                  // threads: 2 per block row
// Shortest triangle that takes this path.  Against halving down to
// trsv_xcd.hpp's launches, one right-hand side, op(A) = A: order 4096 178
// against 168 us, 6000 238 against 268, 16384 734 against 830; with two
// right-hand sides or op(A) = A^T the halving is the faster at every order
// (8192: 378 against 406 and 390 against 648 us).  FP32, by whole mixed
// solves with six such solves each (the cooperative launch costs its 40 us
// there): order 6000 21.46 against 21.02 ms, 8192 30.0 against 29.7, 12288
// 64.8 against 64.9, 20000 123.0 against 124.9.
template <class S>
constexpr long kTrsvMin = sizeof(S) == 8 ? 4097 : 10240;

template <class S>
__device__ inline S ld_co(const S* p);
template <>
__device__ inline double ld_co<double>(const double* p) {
  const unsigned long long u = __hip_atomic_load(
      reinterpret_cast<unsigned long long*>(const_cast<double*>(p)), __ATOMIC_RELAXED,
      __HIP_MEMORY_SCOPE_AGENT);
  return __longlong_as_double(static_cast<long long>(u));
}
template <>
__device__ inline float ld_co<float>(const float* p) {
  return __uint_as_float(__hip_atomic_load(reinterpret_cast<unsigned*>(const_cast<float*>(p)),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ inline void st_co(double* p, double x) {
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p),
                     static_cast<unsigned long long>(__double_as_longlong(x)), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_co(float* p, float x) {
  __hip_atomic_store(reinterpret_cast<unsigned*>(p), __float_as_uint(x), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
// Publication of a solved block.  Everything that crosses workgroups (the
// solved x values and the flags) is accessed only with agent-scope atomic
// loads and stores, which gfx950 performs coherently at the device level
// (the sc1 form: stores write through, loads do not take a stale per-XCD L2
// copy).  What the protocol needs is order: every thread waits until its
// own x stores are acknowledged (s_waitcnt 0) before the workgroup barrier,
// the flag is stored after the barrier, and a reader issues its x loads
// only after its flag load has returned 1 (and a barrier).  Agent-scope
// release/acquire fences would give the same order but also write back and
// invalidate the whole L2 of the XCD at every block (buffer_wbl2 /
// buffer_inv), which made each solve several times slower.

__global__ void sv_reset(int* flags, int n) {
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x)
    flags[e] = 0;
}

template <class S>
__global__ void __launch_bounds__(SV_T)
trsv_sf_kernel(int n, int nb, int upper, S alpha, const S* __restrict__ A, long lda,
               const S* __restrict__ Dinv, S* __restrict__ B, int* __restrict__ flags,
               int* __restrict__ err, int* __restrict__ status, int* __restrict__ info,
               long limit) {
  __shared__ S part[2][NB];
  __shared__ S xs[NB];
  __shared__ int ok;
  const int t = threadIdx.x, r = t & (NB - 1), h = t >> 7;
  for (int li = blockIdx.x; li < nb; li += gridDim.x) {
    const int p = upper ? nb - 1 - li : li;
    const long r0 = (long)p * NB;
    const int rows = (int)min((long)NB, n - r0);
    S acc = S(0);
    for (int lj = 0; lj < li; lj++) {
      const int q = upper ? nb - 1 - lj : lj;
      const long c0 = (long)q * NB;
      const int cols = (int)min((long)NB, n - c0);
      // this thread's 64 entries of op(A)(block p, block q): issued before
      // the wait, they do not depend on x_q
      S va[64];
      const int cend = (r < rows) ? min(64, cols - h * 64) : 0;
      const S* a = A + (r0 + r) + (size_t)(c0 + h * 64) * lda;
#pragma unroll
      for (int c = 0; c < 64; c++) va[c] = (c < cend) ? a[(size_t)c * lda] : S(0);
      if (t == 0) {
        // one round trip per poll; the error word only every 256 polls
        bool good = true;
        long spins = 0;
        while (ld_flag(&flags[q]) == 0) {
          if (++spins >= limit || ((spins & 255) == 0 && ld_flag(err))) {
            st_flag(err, 1);
            atomicOr(status, ATLG_FAIL_TRSV);
            if (info) *info = INT_MIN;
            good = false;
            break;
          }
        }
        ok = good;
      }
      __syncthreads();  // x_q is read (ld_co) only after the flag was seen
      if (!ok) return;  // same value in every thread
      if (t < NB) xs[t] = (t < cols) ? ld_co(&B[c0 + t]) : S(0);
      __syncthreads();
#pragma unroll
      for (int c = 0; c < 64; c++) acc += va[c] * xs[h * 64 + c];
      __syncthreads();
    }
    part[h][r] = acc;
    __syncthreads();
    if (t < NB) xs[t] = (t < rows) ? alpha * B[r0 + t] - part[0][t] - part[1][t] : S(0);
    __syncthreads();
    // x = inv(A_pp) (alpha b - acc): thread (r, h) sums 64 of the 128 columns
    const S* D = Dinv + (size_t)p * NB * NB + r + (size_t)h * 64 * NB;
    S y = S(0);
#pragma unroll
    for (int c0 = 0; c0 < 64; c0 += 16) {
      S d[16];
#pragma unroll
      for (int c = 0; c < 16; c++) d[c] = D[(size_t)(c0 + c) * NB];
#pragma unroll
      for (int c = 0; c < 16; c++) y += d[c] * xs[h * 64 + c0 + c];
    }
    part[h][r] = y;
    __syncthreads();
    if (t < rows) st_co(&B[r0 + t], part[0][t] + part[1][t]);
    // every thread's x stores are acknowledged before the barrier, and the
    // flag is stored after it
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t == 0) st_flag(&flags[p], 1);
  }
}

// Left solve with op(A) = A and one right-hand side, `lower` saying whether A
// is lower triangular, and Dinv holding the inverses of A's diagonal blocks.
template <class S>
void trsv_long(hipStream_t s, bool lower, long n, S alpha, const S* A, long lda, const S* Dinv,
               S* B, const WaitReport& rep) {
  const int nb = (int)((n + NB - 1) / NB);
  int* flags = static_cast<int*>(scratch(s, kSlotTrsv, sizeof(int) * (nb + 64)));
  int* err = flags + nb;
  hipLaunchKernelGGL(sv_reset, dim3((unsigned)std::min(64, (nb + 64 + 255) / 256)), dim3(256), 0,
                     s, flags, nb + 1);
  ATLG_LAUNCHED();
  int dev = 0, cus = 0;
  ATLG_HIP(hipGetDevice(&dev));
  ATLG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  int nn = (int)n, nbk = nb, up = lower ? 0 : 1;
  int G = std::max(1, std::min(nb, cus));
  int *status = rep.status ? rep.status : status_word(s), *info = rep.info;
  long limit = wait_limit(kSvSpin);
  void* args[] = {&nn, &nbk, &up,  &alpha,  &A,    &lda,  &Dinv,
                  &B,  &flags, &err, &status, &info, &limit};
  ATLG_HIP(hipLaunchCooperativeKernel(reinterpret_cast<const void*>(&trsv_sf_kernel<S>), dim3(G),
                                      dim3(SV_T), args, 0, s));
}

}  // namespace

template <class S>
void tri_inverse_blocks(hipStream_t s, long na, const S* A, long lda, int ta, int uplo, int diag,
                        S* Dinv, const int* skip) {
  if (na <= 0) return;
  const bool tr = is_trans(ta);
  const long nblk = (na + NB - 1) / NB;
  const int trn = tr ? 1 : 0, low = (uplo == kLower) != tr ? 1 : 0, un = diag == kUnit ? 1 : 0;
  if (na <= 32)
    hipLaunchKernelGGL((trtri_diag_kernel<S, 32>), dim3(1), dim3(4 * 32), 0, s, (int)na, A,
                       lda, trn, low, un, Dinv, skip);
  else if (na <= 64)
    hipLaunchKernelGGL((trtri_diag_kernel<S, 64>), dim3(1), dim3(4 * 64), 0, s, (int)na, A,
                       lda, trn, low, un, Dinv, skip);
  else
    hipLaunchKernelGGL((trtri_diag_kernel<S, NB>), dim3((unsigned)nblk), dim3(4 * NB), 0, s,
                       (int)na, A, lda, trn, low, un, Dinv, skip);
  ATLG_LAUNCHED();
}

template <class S>
void trsm(hipStream_t s, int side, int uplo, int ta, int diag, long M, long N, S alpha,
          const S* A, long lda, S* B, long ldb, const int* skip, const S* dinv, int dinv_trans,
          WaitReport rep) {
  if (M <= 0 || N <= 0) return;
  if (alpha == S(0)) {
    scale<S>(s, M, N, S(0), B, ldb, 0, skip);
    return;
  }
  Ctx<S> c;
  c.s = s;
  c.left = (side == kLeft);
  c.trans = is_trans(ta);
  c.lower_eff = ((uplo == kLower) != c.trans);
  c.A = A;
  c.lda = lda;
  c.B = B;
  c.ldb = ldb;
  c.M = M;
  c.N = N;
  c.skip = skip;
  c.rep = rep;
  c.fixed = nullptr;
  const long na = c.left ? M : N;
  c.dtrans = dinv ? (dinv_trans ? kTrans : kNoTrans) : kNoTrans;
  if (dinv) {
    c.Dinv = dinv;
  } else {
    const long nblk = (na + NB - 1) / NB;
    S* D = static_cast<S*>(scratch(s, kSlotTrsmInv, sizeof(S) * nblk * NB * NB));
    tri_inverse_blocks<S>(s, na, A, lda, ta, uplo, diag, D, skip);
    c.Dinv = D;
  }
  if (c.left && !c.trans && c.dtrans == kNoTrans && !skip && N == 1 && na >= kTrsvMin<S>) {
    trsv_long<S>(s, c.lower_eff, na, alpha, A, lda, c.Dinv, B, rep);
    return;
  }
  solve(c, 0, na, alpha);
}

// The allocation-free form: the diagonal-block inverses go to the file-scope
// device array (at most kNoAllocMaxOrder / kTrsmNB blocks), and so does the
// exchange area of the one-launch solves and their failure words; the solve is
// otherwise trsm()'s without its sync-free launch for one right-hand side.
template <class S>
void trsm_noalloc(hipStream_t s, int side, int uplo, int ta, int diag, long M, long N, S alpha,
                  const S* A, long lda, S* B, long ldb) {
  if (M <= 0 || N <= 0) return;
  if (alpha == S(0)) {
    scale<S>(s, M, N, S(0), B, ldb, 0, nullptr);
    return;
  }
  const long na = side == kLeft ? M : N;
  if (na > kNoAllocMaxOrder) throw HipFailure{"trsm_noalloc: order above the allocation-free maximum"};
  S* D = static_cast<S*>(noalloc_scratch());
  tri_inverse_blocks<S>(s, na, A, lda, ta, uplo, diag, D, nullptr);
  Ctx<S> c;
  c.s = s;
  c.left = (side == kLeft);
  c.trans = is_trans(ta);
  c.lower_eff = ((uplo == kLower) != c.trans);
  c.A = A;
  c.lda = lda;
  c.B = B;
  c.ldb = ldb;
  c.M = M;
  c.N = N;
  c.skip = nullptr;
  c.fixed = static_cast<unsigned char*>(noalloc_scratch()) + kNoAllocInvBytes;
  c.rep.status = noalloc_word(s, true);
  c.Dinv = D;
  c.dtrans = kNoTrans;
  solve(c, 0, na, alpha);
}

template void trsm_noalloc<double>(hipStream_t, int, int, int, int, long, long, double,
                                   const double*, long, double*, long);

template void tri_inverse_blocks<double>(hipStream_t, long, const double*, long, int, int, int,
                                         double*, const int*);
template void tri_inverse_blocks<float>(hipStream_t, long, const float*, long, int, int, int,
                                        float*, const int*);
template void trsm<double>(hipStream_t, int, int, int, int, long, long, double, const double*,
                           long, double*, long, const int*, const double*, int, WaitReport);
template void trsm<float>(hipStream_t, int, int, int, int, long, long, float, const float*, long,
                          float*, long, const int*, const float*, int, WaitReport);

}  // namespace atlg

// ---- the device array behind atlg_dtrsm_noalloc ---------------------------
// kNoAllocMaxOrder / kTrsmNB inverses of 128 x 128 doubles (8 MiB), the
// exchange area of the one-launch solves (24 MiB) and their failure words, one
// copy per device, zero at first, held until the process ends.  Its name is only a host-side
// stand-in for the symbol: host code uses the address that
// hipGetSymbolAddress returns for the current device, never the name itself.
static __device__ __align__(256) unsigned char scratch[atlg::kNoAllocBytes];

namespace atlg {
namespace {
constexpr int kMaxDevices = 64;
std::mutex g_noalloc_mu;
void* g_noalloc_ptr[kMaxDevices] = {};
std::map<hipStream_t, int> g_noalloc_words[kMaxDevices];  // stream -> its word's index
}  // namespace

// Address of the array on the current device, resolved once per device
// (with that device current) and kept.
void* noalloc_scratch() {
  int dev = 0;
  ATLG_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) throw HipFailure{"trsm_noalloc: device index out of range"};
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  if (!g_noalloc_ptr[dev]) {
    void* p = nullptr;
    ATLG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(::scratch)));
    g_noalloc_ptr[dev] = p;
  }
  return g_noalloc_ptr[dev];
}

int* noalloc_word(hipStream_t s, bool make) {
  int dev = 0;
  ATLG_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return nullptr;  // (noalloc_scratch() refuses the solve)
  int index = 0;
  {
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    auto& words = g_noalloc_words[dev];
    const auto it = words.find(s);
    if (it != words.end()) {
      index = it->second;
    } else {
      if (!make) return nullptr;
      index = (int)std::min(words.size(), kNoAllocWords - 1);
      words[s] = index;
    }
  }
  unsigned char* end = static_cast<unsigned char*>(noalloc_scratch()) + kNoAllocBytes;
  return reinterpret_cast<int*>(end) - kNoAllocWords + index;
}

}  // namespace atlg
