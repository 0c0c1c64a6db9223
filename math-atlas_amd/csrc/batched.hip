// Batched Cholesky factor/solve of many independent SPD systems of uneven
// order in one persistent launch.  ATLAS factors one matrix per call
// (ATL_dpotrf / ATL_dpotrs, AtlasBase/Clint/atlas-lp.base:332-360, 969-1050);
// the per-system arithmetic here is the same lower Cholesky A = L L^T and the
// same pair of triangular solves, and the mixed-precision driver follows
// LAPACK's dsposv refinement (single-precision factor, double-precision
// residual, stop when ||r||_inf < ||x||_inf * ||A||_inf * eps * sqrt(n) for
// every right-hand side, at most 30 iterations).
//
// Work distribution: the host orders the systems longest first (n^3 is the
// work) and every workgroup pulls the next system from an atomic counter
// until the queue is drained, so every workgroup exits after the last system.
// One workgroup (kBW waves) owns a system from start to finish.
//
// Per system (batched_chol.hpp): a left-looking factorization by block columns
// of 64 on the matrix cores, each wave taking 16 or 32 rows at a time (chosen
// per system on the host by the decision tree the empirical search
// generates), and sweeps over the factor for four right-hand sides at a time
// in LDS; the forward sweep of the first four runs beside the factorization.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <mutex>
#include <numeric>
#include <vector>

#include "atlg_internal.hpp"
#include "atlg_batched_tune.h"
#include "tri_inv.hpp"

namespace atlg {
namespace {

constexpr int kBW = 4;          // waves per workgroup
constexpr int kBT = 64 * kBW;   // threads per workgroup

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// The 16x16x4 MFMA for each scalar type.  D = X1 * X2 with lane l supplying
// X1[l&15][l>>4] and X2[l>>4][l&15]; lane l, register r holds row
// (l>>4) + 4 r (FP64) or 4 (l>>4) + r (FP32) of column l & 15.
template <class S>
struct Mfma;
template <>
struct Mfma<double> {
  typedef d4 acc_t;
  static __device__ __forceinline__ acc_t op(double x1, double x2, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(x1, x2, c, 0, 0, 0);
  }
};
template <>
struct Mfma<float> {
  typedef f4 acc_t;
  static __device__ __forceinline__ acc_t op(float x1, float x2, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x1, x2, c, 0, 0, 0);
  }
};

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS of one workgroup, typed per scalar at use: the tiles of the diagonal
// block (a factorization) and the sweeps' partial sums take turns in LT; Y
// holds up to four right-hand sides ([row][4]) of a system of order <=
// kYmax / 4, or the mixed solver's FP32 ones and X for its residual.
constexpr int kYmax = 6144;
constexpr int kMixN = kYmax / 6;  // 4 floats and 4 doubles a row
struct alignas(16) Smem {
  double LT[11 * 16 * 17];
  double red[kBW * 8];  // reductions
  double Y[kYmax];
  int flag;             // failure index + 1, 0 = fine
  int cur;              // system taken from the queue
};

#include "batched_chol.hpp"

// Whether four right-hand sides of a system fit in LDS.
__device__ __forceinline__ bool rhs_fit(int n) { return 4 * n <= kYmax; }
// Y ([row][NQ] in LDS, zero to the end of the last tile) = B, and B = Y
template <class S, int NQ = 4, class T>
__device__ __forceinline__ void rhs_in(int n, int nrhs, const T* B, int ldb, S* Y) {
  for (int r = 0; r < NQ; r++)
    for (int i = threadIdx.x; i < ((n + kTile - 1) & -kTile); i += kBT)
      Y[i * NQ + r] = r < nrhs && i < n ? (S)B[i + (size_t)r * ldb] : S(0);
  __syncthreads();
}
template <class S, int NQ = 4>
__device__ __forceinline__ void rhs_out(int n, int nrhs, S* B, int ldb, const S* Y) {
  for (int r = 0; r < nrhs; r++)
    for (int i = threadIdx.x; i < n; i += kBT) B[i + (size_t)r * ldb] = Y[i * NQ + r];
}

// acc[q] += sum_{c < w} p[c*st] * b[c + (r0+q)*ldb] for the right-hand sides
// r0 + q < nrhs, in order of c, four loads of p in flight at a time (the
// mixed solver's FP64 residual).
template <class S>
__device__ __forceinline__ void row_dot4(const S* p, size_t st, int w, const S* b, int sc, int sq,
                                         int r0, int nrhs, S (&acc)[4]) {
  int c = 0;
#pragma unroll 1
  for (; c + 4 <= w; c += 4) {
    S lv[4];
#pragma unroll
    for (int u = 0; u < 4; u++) lv[u] = p[(size_t)(c + u) * st];
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (r0 + q < nrhs) acc[q] += lv[u] * b[(size_t)(c + u) * sc + (size_t)q * sq];
  }
  for (; c < w; c++) {
    const S lv = p[(size_t)c * st];
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (r0 + q < nrhs) acc[q] += lv * b[(size_t)c * sc + (size_t)q * sq];
  }
}

// Solves L L^T X = B in place (B: n x nrhs, column-major, ldb), eight
// right-hand sides at a time in LDS where they fit, else four: a sweep is
// latency, so more of them cost little (1000 systems of order 200 with 16:
// 570 us against 730 by fours; 256 of order 600 with 8: 391 against 599).
template <class S, int NG>
__device__ __forceinline__ void solve_group(int n, const S* __restrict__ L, int lda, S* __restrict__ b,
                                            int ldb, int nr, Smem& sm) {
  S* Y = reinterpret_cast<S*>(sm.Y);
  __syncthreads();  // the last group is in memory
  rhs_in<S, 4 * NG>(n, nr, b, ldb, Y);
  sweep<S, false, false, NG>(n, L, lda, sm, Y);
  sweep<S, true, false, NG>(n, L, lda, sm, Y);
  rhs_out<S, 4 * NG>(n, nr, b, ldb, Y);
}
template <class S>
__device__ __attribute__((noinline)) void solve_sys(int n, const S* __restrict__ L, int lda,
                                                    S* __restrict__ B, int ldb, int nrhs, Smem& sm) {
  for (int r0 = 0; r0 < nrhs;) {
    S* b = B + (size_t)r0 * ldb;
    if (nrhs - r0 > 4 && 8 * n <= kYmax) {
      solve_group<S, 2>(n, L, lda, b, ldb, min(8, nrhs - r0), sm);
      r0 += 8;
      continue;
    }
    const int nr = min(4, nrhs - r0);
    if (rhs_fit(n)) {
      solve_group<S, 1>(n, L, lda, b, ldb, nr, sm);
    } else {
      sweep<S, false, true>(n, L, lda, sm, b, ldb, nr);
      sweep<S, true, true>(n, L, lda, sm, b, ldb, nr);
    }
    r0 += 4;
  }
}

// Takes the next queue entry (or -1 when drained); every thread gets it.
__device__ int next_system(unsigned* counter, int nsys, Smem& sm) {
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned q = atomicAdd(counter, 1u);
    sm.cur = (q < (unsigned)nsys) ? (int)q : -1;
  }
  __syncthreads();
  return sm.cur;
}

template <class S>
struct SysDesc {
  S* A;
  S* B;
  const S* Bsrc;  // copied into B first when not null
  int n, lda, ldb, idx, width;
};

// mode: 0 factor, 1 factor + solve, 2 solve with a given factor.
// What bounds it: 2000 uneven systems (n 16..512, 4 right-hand sides) take
// 1.9 ms, 3.3 ms by 32-wide block columns with the diagonal block factored
// column by column in LDS; a system of 512 alone 0.53 against 1.26 ms.  Of 860
// us that one of 512 takes beside another on its compute unit, 540 are row
// tiles' products (half of it matrix core time), 170 pivots, 140 sweeps.
// Two workgroups per compute unit: a third leaves 168 registers, and the
// spills cost more than the latency it hides (2.2 ms).
template <class S>
__global__ void __launch_bounds__(kBT) __attribute__((amdgpu_waves_per_eu(2)))
posv_batched_kernel(int nsys, const SysDesc<S>* __restrict__ desc, int nrhs, int mode,
                    int* __restrict__ info, unsigned* __restrict__ counter) {
  __shared__ Smem sm;
  for (;;) {
    const int q = next_system(counter, nsys, sm);
    if (q < 0) return;
    const SysDesc<S> d = desc[q];
    if (d.Bsrc) {
      for (int r = 0; r < nrhs; r++)
        for (int i = threadIdx.x; i < d.n; i += kBT)
          d.B[i + (size_t)r * d.ldb] = d.Bsrc[i + (size_t)r * d.ldb];
      __syncthreads();
    }
    // the first four right-hand sides' forward substitution runs beside the
    // factorization in LDS; B is left as it was when that fails
    const bool fuse = mode == 1 && nrhs > 0 && rhs_fit(d.n);
    const int nf = fuse ? min(nrhs, 4) : 0;
    S* Y = reinterpret_cast<S*>(sm.Y);
    if (fuse) rhs_in<S>(d.n, nf, d.B, d.ldb, Y);
    const int f = mode != 2 ? chol_sys<S>(d.n, d.A, d.lda, d.width, sm, fuse ? Y : nullptr) : 0;
    if (f == 0 && mode != 0) {
      if (fuse) {
        sweep<S, true, false>(d.n, d.A, d.lda, sm, Y);
        rhs_out<S>(d.n, nf, d.B, d.ldb, Y);
      }
      if (nrhs > nf)
        solve_sys<S>(d.n, d.A, d.lda, d.B + (size_t)nf * d.ldb, d.ldb, nrhs - nf, sm);
    }
    if (threadIdx.x == 0 && mode != 2) info[d.idx] = f;
  }
}

// ---- mixed precision: FP32 factor, FP64 residual and update ---------------
struct MixDesc {
  const double* A;  // FP64 matrix (lower triangle read)
  const double* B;  // FP64 right-hand sides
  double* X;        // FP64 solution
  float* A32;       // workspace n x n (ld n)
  float* W32;       // workspace n x nrhs (ld n)
  int n, lda, ldb, ldx, idx, width;
};

__device__ double block_max(double v, Smem& sm) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sm.red[threadIdx.x >> 6] = v;
  __syncthreads();
  double m = sm.red[0];
  for (int k = 1; k < kBW; k++) m = fmax(m, sm.red[k]);
  return m;
}

// r = B - A X for the rows this thread owns; returns max |x| and max |r| of
// right-hand side r0..r0+3 across the workgroup, writing float(r) to W32.
__device__ void residual(const MixDesc& d, int nrhs, Smem& sm, bool* conv, double cte) {
  const int n = d.n;
  // X staged in LDS when it fits: the rows' dot products then read it there
  // instead of from global memory
  const bool stage = rhs_fit(n);
  for (int r0 = 0; r0 < nrhs; r0 += 4) {
    double xm[4] = {0, 0, 0, 0}, rm[4] = {0, 0, 0, 0};
    if (stage) {
      for (int e = threadIdx.x; e < 4 * n; e += kBT) {
        const int j = e >> 2, q = e & 3;
        sm.Y[e] = (r0 + q < nrhs) ? d.X[j + (size_t)(r0 + q) * d.ldx] : 0.0;
      }
      __syncthreads();
    }
    for (int i = threadIdx.x; i < n; i += kBT) {
      double acc[4] = {0, 0, 0, 0};
      // row i of the lower triangle, then column i below the diagonal
      if (stage) {
        row_dot4<double>(d.A + i, (size_t)d.lda, i + 1, sm.Y, 4, 1, r0, nrhs, acc);
        row_dot4<double>(d.A + (size_t)i * d.lda + i + 1, 1, n - i - 1, sm.Y + 4 * (i + 1), 4,
                         1, r0, nrhs, acc);
      } else {
        const double* xr = d.X + (size_t)r0 * d.ldx;
        row_dot4<double>(d.A + i, (size_t)d.lda, i + 1, xr, 1, d.ldx, r0, nrhs, acc);
        row_dot4<double>(d.A + (size_t)i * d.lda + i + 1, 1, n - i - 1, xr + i + 1, 1, d.ldx, r0,
                         nrhs, acc);
      }
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (r0 + q < nrhs) {
          const double rv = d.B[i + (size_t)(r0 + q) * d.ldb] - acc[q];
          xm[q] = fmax(xm[q], fabs(d.X[i + (size_t)(r0 + q) * d.ldx]));
          rm[q] = fmax(rm[q], fabs(rv));
          d.W32[i + (size_t)(r0 + q) * n] = (float)rv;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (r0 + q >= nrhs) break;
      const double xn = block_max(xm[q], sm), rn = block_max(rm[q], sm);
      if (!(rn < xn * cte)) *conv = false;
    }
  }
}

// The same with X, the residual and the right-hand sides' maxima by tiles on
// the matrix cores (n <= kMixN, at most four right-hand
// sides): float(r) goes to Y.
__device__ bool residual_lds(const MixDesc& d, int nrhs, Smem& sm, float* Y, double cte) {
  typedef Mfma<double> M;
  const int n = d.n;
  const int lane = threadIdx.x & 63, ln = lane & 15, lk = lane >> 4, wave = threadIdx.x >> 6;
  double* XS = sm.Y + 2 * kMixN;
  rhs_in<double>(n, nrhs, d.X, d.ldx, XS);
  double xm = 0.0, rm = 0.0;  // of right-hand side lk
  for (int t = wave; kTile * t < n; t += kBW) {
    const int i = kTile * t + ln;
    d4 acc = {0, 0, 0, 0};
    sym_row_tile(n, d.A, (size_t)d.lda, t, [&](int k, double v) {
      const double x = XS[4 * k + (ln & 3)];
      acc = M::op(ln < 4 ? x : 0.0, v, acc);
    });
    if (i < n && lk < nrhs) {
      const double r = d.B[i + (size_t)lk * d.ldb] - acc[0];
      xm = fmax(xm, fabs(XS[4 * i + lk]));
      rm = fmax(rm, fabs(r));
      Y[4 * i + lk] = (float)r;
      // (a NaN is no maximum: fmax drops it, here as in residual())
    }
  }
  for (int o = 8; o > 0; o >>= 1) {
    xm = fmax(xm, __shfl_xor(xm, o, 64));
    rm = fmax(rm, __shfl_xor(rm, o, 64));
  }
  __syncthreads();
  if (ln == 0) {
    sm.red[wave * 8 + 2 * lk] = xm;
    sm.red[wave * 8 + 2 * lk + 1] = rm;
  }
  __syncthreads();
  bool conv = true;
  for (int q = 0; q < nrhs; q++) {
    double x = 0.0, r = 0.0;
    for (int w = 0; w < kBW; w++) {
      x = fmax(x, sm.red[w * 8 + 2 * q]);
      r = fmax(r, sm.red[w * 8 + 2 * q + 1]);
    }
    if (!(r < x * cte)) conv = false;
  }
  return conv;
}

// The same workgroups; the 2000 systems above take 3.9 ms (5.8 ms before).  A third workgroup
// per compute unit gains 1% there and costs 20% on 800 systems up to order 256.  Beside the
// factorization, what bounds it is reading the FP64 triangle: once for the norm and the FP32
// copy, once per residual (each tile read along its rows, then along its columns).
__global__ void __launch_bounds__(kBT) __attribute__((amdgpu_waves_per_eu(2)))
mixed_posv_kernel(int nsys, const MixDesc* __restrict__ desc, int nrhs, int itermax,
                  int* __restrict__ info, int* __restrict__ iter, unsigned* __restrict__ counter) {
  __shared__ Smem sm;
  for (;;) {
    const int q = next_system(counter, nsys, sm);
    if (q < 0) return;
    const MixDesc d = desc[q];
    const int n = d.n;
    // ||A||_inf of the symmetric matrix, A32 = float(lower(A)), overflow check
    double rs = 0.0;
    bool over = false;
    const int ln = threadIdx.x & 15;
    for (int t = threadIdx.x >> 6; kTile * t < n; t += kBW) {
      const int i = kTile * t + ln;
      double s = 0.0;
      sym_row_tile(n, d.A, (size_t)d.lda, t, [&](int k, double v) {
        if (k >= n) return;
        s += fabs(v);
        if (k <= i && i < n) {
          if (fabs(v) > (double)FLT_MAX) over = true;
          d.A32[i + (size_t)k * n] = (float)v;
        }
      });
      s += __shfl_xor(s, 16, 64);
      s += __shfl_xor(s, 32, 64);
      if (i < n) rs = fmax(rs, s);
    }
    const double anrm = block_max(rs, sm);
    const double ov = block_max(over ? 1.0 : 0.0, sm);
    const bool fuse = nrhs > 0 && nrhs <= 4 && n <= kMixN;
    float* Y = reinterpret_cast<float*>(sm.Y);
    int it = 0;
    if (n == 0) {
      it = 0;
    } else if (ov != 0.0) {
      it = -2;
    } else {
      // W32 = float(B), or Y when the right-hand sides fit in LDS
      if (fuse)
        rhs_in<float>(n, nrhs, d.B, d.ldb, Y);
      else
        for (int r = 0; r < nrhs; r++)
          for (int i = threadIdx.x; i < n; i += kBT)
            d.W32[i + (size_t)r * n] = (float)d.B[i + (size_t)r * d.ldb];
      __syncthreads();
      it = chol_sys<float>(n, d.A32, n, d.width, sm, fuse ? Y : nullptr) != 0 ? -3 : 0;
    }
    if (it == 0 && n > 0) {
      // X = float solve of B
      if (fuse) sweep<float, true, false>(n, d.A32, n, sm, Y);
      else solve_sys<float>(n, d.A32, n, d.W32, n, nrhs, sm);
      __syncthreads();
      for (int r = 0; r < nrhs; r++)
        for (int i = threadIdx.x; i < n; i += kBT)
          d.X[i + (size_t)r * d.ldx] = (double)(fuse ? Y[i * 4 + r] : d.W32[i + (size_t)r * n]);
      __syncthreads();
      const double cte = anrm * (DBL_EPSILON * 0.5) * sqrt((double)n);
      it = -(itermax + 1);
      for (int k = 0; k <= itermax; k++) {
        bool conv = true;
        if (fuse) conv = residual_lds(d, nrhs, sm, Y, cte);
        else residual(d, nrhs, sm, &conv, cte);  // ends with a barrier (block_max)
        if (conv) {
          it = k;
          break;
        }
        if (k == itermax) break;
        if (fuse) {
          sweep<float, false, false>(n, d.A32, n, sm, Y);
          sweep<float, true, false>(n, d.A32, n, sm, Y);
        } else {
          solve_sys<float>(n, d.A32, n, d.W32, n, nrhs, sm);
          __syncthreads();
        }
        for (int r = 0; r < nrhs; r++)
          for (int i = threadIdx.x; i < n; i += kBT)
            d.X[i + (size_t)r * d.ldx] += (double)(fuse ? Y[i * 4 + r] : d.W32[i + (size_t)r * n]);
        __syncthreads();
      }
    }
    if (threadIdx.x == 0) {
      iter[d.idx] = it;
      info[d.idx] = 0;
    }
  }
}

__global__ void zero_counter(unsigned* c) { *c = 0u; }

// ---- host side -------------------------------------------------------------

// Pinned staging for the descriptor upload, reused once the previous copy
// from it has completed.
struct Staging {
  void* host = nullptr;
  size_t cap = 0;
  hipEvent_t done = nullptr;
};
std::mutex g_stage_mu;
Staging g_stage;

void* stage_upload(hipStream_t s, const void* src, size_t bytes, Slot slot) {
  void* dev = scratch(s, slot, bytes);
  std::lock_guard<std::mutex> lk(g_stage_mu);
  if (g_stage.done) ATLG_HIP(hipEventSynchronize(g_stage.done));
  if (bytes > g_stage.cap) {
    if (g_stage.host) ATLG_HIP(hipHostFree(g_stage.host));
    g_stage.host = nullptr;
    g_stage.cap = 0;
    ATLG_HIP(hipHostMalloc(&g_stage.host, bytes, hipHostMallocDefault));
    g_stage.cap = bytes;
  }
  if (!g_stage.done) ATLG_HIP(hipEventCreateWithFlags(&g_stage.done, hipEventDisableTiming));
  std::memcpy(g_stage.host, src, bytes);
  ATLG_HIP(hipMemcpyAsync(dev, g_stage.host, bytes, hipMemcpyHostToDevice, s));
  ATLG_HIP(hipEventRecord(g_stage.done, s));
  return dev;
}

// Longest-first order of the systems (n^3 decides; ties by index).
std::vector<int> lpt_order(int nsys, const int* n) {
  std::vector<int> ord(nsys);
  std::iota(ord.begin(), ord.end(), 0);
  std::stable_sort(ord.begin(), ord.end(), [n](int a, int b) { return n[a] > n[b]; });
  return ord;
}

int grid_for(hipStream_t s, const BatchTune& tune, int nsys) {
  (void)s;
  int dev = 0, cus = 256;
  ATLG_HIP(hipGetDevice(&dev));
  ATLG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  return std::max(1, std::min(nsys, cus * std::max(1, tune.wg_per_cu)));
}

unsigned* reset_counter(hipStream_t s) {
  unsigned* counter = static_cast<unsigned*>(scratch(s, kSlotBatchCtr, 256));
  hipLaunchKernelGGL(zero_counter, dim3(1), dim3(1), 0, s, counter);
  ATLG_LAUNCHED();
  return counter;
}

BatchTune g_tune[2] = {{-1, ATLG_BATCH_WPC_D}, {-1, ATLG_BATCH_WPC_S}};
std::mutex g_tune_mu;

// Rows that a wave takes at a time below a system's diagonal blocks (16 or
// 32): by the override threshold when set, else by the generated decision
// tree of the empirical search.
int width_for(const BatchTune& tune, bool single, int n) {
  if (tune.t16_max >= 0) return n <= tune.t16_max ? 16 : 32;
  return single ? atlg_batched_width_s(n) : atlg_batched_width_d(n);
}

}  // namespace

BatchTune batch_tune(bool single) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  return g_tune[single ? 1 : 0];
}
void set_batch_tune(bool single, const BatchTune& t) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tune[single ? 1 : 0] = t;
}

template <class S>
void posv_batched(hipStream_t s, int mode, int nsys, const int* n, S* const* A, const int* lda,
                  S* const* B, const int* ldb, const S* const* Bsrc, int nrhs, int* info,
                  const BatchTune& tune, const int* orig) {
  if (nsys <= 0) return;
  const std::vector<int> ord = lpt_order(nsys, n);
  std::vector<SysDesc<S>> desc(nsys);
  for (int q = 0; q < nsys; q++) {
    const int k = ord[q];
    desc[q] = SysDesc<S>{A[k], B ? B[k] : nullptr, Bsrc ? Bsrc[k] : nullptr, n[k], lda[k],
                         ldb ? ldb[k] : 1, orig ? orig[k] : k,
                         width_for(tune, std::is_same<S, float>::value, n[k])};
  }
  auto* dd = static_cast<const SysDesc<S>*>(
      stage_upload(s, desc.data(), sizeof(SysDesc<S>) * nsys, kSlotBatchDesc));
  unsigned* counter = reset_counter(s);
  hipLaunchKernelGGL(posv_batched_kernel<S>, dim3(grid_for(s, tune, nsys)), dim3(kBT), 0, s, nsys,
                     dd, nrhs, mode, info, counter);
  ATLG_LAUNCHED();
}

template void posv_batched<double>(hipStream_t, int, int, const int*, double* const*, const int*,
                                   double* const*, const int*, const double* const*, int, int*,
                                   const BatchTune&, const int*);
template void posv_batched<float>(hipStream_t, int, int, const int*, float* const*, const int*,
                                  float* const*, const int*, const float* const*, int, int*,
                                  const BatchTune&, const int*);

void dsposv_batched(hipStream_t s, int nsys, const int* n, double* const* A, const int* lda,
                    const double* const* B, const int* ldb, double* const* X, const int* ldx,
                    int nrhs, int* info, int* iter, int itermax, const BatchTune& tune) {
  if (nsys <= 0) return;
  const std::vector<int> ord = lpt_order(nsys, n);
  size_t ws = 0;
  std::vector<size_t> off(nsys);
  for (int q = 0; q < nsys; q++) {
    off[q] = ws;
    const size_t nn = (size_t)n[ord[q]];
    ws += (nn * nn + nn * (size_t)nrhs + 63) & ~(size_t)63;  // floats, 256-byte aligned
  }
  float* W = static_cast<float*>(scratch(s, kSlotBatchWork, std::max<size_t>(ws, 64) * 4));
  std::vector<MixDesc> desc(nsys);
  for (int q = 0; q < nsys; q++) {
    const int k = ord[q];
    const size_t nn = (size_t)n[k];
    desc[q] = MixDesc{A[k], B[k], X[k], W + off[q], W + off[q] + nn * nn, n[k], lda[k], ldb[k],
                      ldx[k], k, width_for(tune, true, n[k])};
  }
  auto* dd = static_cast<const MixDesc*>(
      stage_upload(s, desc.data(), sizeof(MixDesc) * nsys, kSlotBatchDesc));
  unsigned* counter = reset_counter(s);
  hipLaunchKernelGGL(mixed_posv_kernel, dim3(grid_for(s, tune, nsys)), dim3(kBT), 0, s, nsys, dd,
                     nrhs, itermax, info, iter, counter);
  ATLG_LAUNCHED();
  // Systems whose refinement did not converge (or whose FP32 factor failed)
  // get the FP64 factor and solve, as LAPACK's dsposv does; A then holds the
  // FP64 factor and X the FP64 solution.
  std::vector<int> it(nsys);
  ATLG_HIP(hipMemcpyAsync(it.data(), iter, sizeof(int) * nsys, hipMemcpyDeviceToHost, s));
  ATLG_HIP(hipStreamSynchronize(s));
  std::vector<int> fn, flda, fldx, forig;
  std::vector<double*> fA, fX;
  std::vector<const double*> fB;
  for (int k = 0; k < nsys; k++) {
    if (it[k] >= 0) continue;
    fn.push_back(n[k]);
    flda.push_back(lda[k]);
    fldx.push_back(ldx[k]);
    forig.push_back(k);
    fA.push_back(A[k]);
    fX.push_back(X[k]);
    if (ldb[k] == ldx[k]) {
      fB.push_back(B[k]);  // copied into X inside the launch
    } else {
      ATLG_HIP(hipMemcpy2DAsync(X[k], sizeof(double) * ldx[k], B[k], sizeof(double) * ldb[k],
                                sizeof(double) * n[k], nrhs, hipMemcpyDeviceToDevice, s));
      fB.push_back(nullptr);
    }
  }
  if (fn.empty()) return;
  posv_batched<double>(s, 1, (int)fn.size(), fn.data(), fA.data(), flda.data(), fX.data(),
                       fldx.data(), fB.data(), nrhs, info, batch_tune(false), forig.data());
  ATLG_HIP(hipStreamSynchronize(s));
}

}  // namespace atlg
