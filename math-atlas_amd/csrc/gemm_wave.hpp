// GEMM by independent waves of 32x32, for products whose 128x128 tiles would
// leave the device idle; included by gemm.hip.
//
// What bounds such a product: a 128x128 tile per workgroup gives an order-1000
// product 64 workgroups for 256 compute units, and each of them a serial chain
// of K steps with a barrier.  Here a wave owns a 32x32 tile of C (2x2 MFMA
// tiles, 16 accumulators per lane) and a slice of K, and loads both operands
// straight into the MFMA registers, two 16-deep chunks ahead: no LDS, no
// barrier in the K loop.  Per 16-deep chunk a wave moves 8 KB against 1024
// cycles of MFMA, so the four SIMDs of a compute unit ask its 64 B/clk vector
// cache for half its rate.  A workgroup is WM x WN waves of C times WS slices
// of K; the slices' sums meet in LDS at the end, in slice order, so results do
// not depend on timing.
//
// Lane (fx, fk) = (l & 15, l >> 4) supplies, at step ks of a chunk, row
// (column) 16 i + fx of tile i at k = 4 fk + ks.  An operand contiguous along
// its tile side (A, B^T) is loaded element by element, 16 lanes to a 128-byte
// line; one contiguous along k (A^T, B) four k per lane with 16-byte loads
// (8-byte aligned, which global loads allow).  Rows past the edge are clamped
// on load and masked on store; the last chunk of K, when ragged, loads
// element by element with zeros past K.
#pragma once

constexpr int GW_T = 32;   // wave tile
constexpr int GW_K = 16;   // k per chunk

template <class S, bool XC>
struct GwOperand {
  typedef S vec2 __attribute__((ext_vector_type(2)));
  static constexpr int E = sizeof(S);
  const S* base;     // tile origin at k = 0
  long ld;
  unsigned off[2];   // byte offset of this lane's element (tile i, k = 4 fk)
  int x[2], fk;      // clamped rows, relative to the tile
  __device__ __forceinline__ void init(const S* P, long ld_, int x0, int X, int fx, int fk_) {
    ld = ld_;
    fk = fk_;
    base = XC ? P + x0 : P + (size_t)x0 * ld;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      x[i] = min(16 * i + fx, X - 1 - x0);
      off[i] = XC ? (unsigned)((x[i] + 4L * fk * ld) * E) : (unsigned)((4L * fk + x[i] * ld) * E);
    }
  }
  // v[ks][i]: row 16 i + fx of the tile at k = k0 + 4 fk + ks
  __device__ __forceinline__ void load(int k0, S (&v)[4][2]) const {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<S*>(XC ? base + (size_t)k0 * ld : base + k0), 0, 0x7fffffff, kBufDword3);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      if constexpr (XC) {
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
          if constexpr (E == 8)
            v[ks][i] = __builtin_bit_cast(
                S, __builtin_amdgcn_raw_buffer_load_b64(r, off[i], ks * (int)ld * E, 0));
          else
            v[ks][i] = bit32(__builtin_amdgcn_raw_buffer_load_b32(r, off[i], ks * (int)ld * E, 0));
        }
      } else if constexpr (E == 8) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const vec2 w = __builtin_bit_cast(
              vec2, __builtin_amdgcn_raw_buffer_load_b128(r, off[i] + 16 * h, 0, 0));
          v[2 * h][i] = w[0];
          v[2 * h + 1][i] = w[1];
        }
      } else {
        const auto w = __builtin_amdgcn_raw_buffer_load_b128(r, off[i], 0, 0);
#pragma unroll
        for (int ks = 0; ks < 4; ks++) v[ks][i] = bit32(w[ks]);
      }
    }
  }
  __device__ __forceinline__ static S bit32(unsigned u) {
    return (S)__builtin_bit_cast(float, u);
  }
  __device__ __forceinline__ void load_tail(int k0, int K, S (&v)[4][2]) const {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int ks = 0; ks < 4; ks++) {
        const int k = k0 + 4 * fk + ks;
        v[ks][i] = S(0);
        if (k < K) v[ks][i] = XC ? base[x[i] + (size_t)k * ld] : base[k + (size_t)x[i] * ld];
      }
  }
};

// XT: batch members blockIdx.y at strides sa, sb, sc, K ranges trimmed by
// ktrim, K a multiple of GW_K; the tiles in gemm_rega_f64's order.
template <class S, bool AT, bool BT, int WM, int WN, int WS, bool XT = false>
__global__ void __launch_bounds__(64 * WM * WN * WS)
gemm_wave(int M, int N, int K, S alpha, const S* A, long lda, const S* B, long ldb, S beta,
          S* C, long ldc, int mode, const int* __restrict__ skip, long sa, long sb, long sc,
          int ktrim) {
  typedef Mfma<S> MF;
  constexpr int TM_ = GW_T * WM, TN_ = GW_T * WN, NW = WM * WN;
  if (skip && *skip) return;
  __shared__ S part[WS > 1 ? WS * NW * 16 * 64 : 1];
  const int tilesM = (M + TM_ - 1) / TM_, tilesN = (N + TN_ - 1) / TN_;
  int tm, tn;
  if (XT) {
    const unsigned id = blockIdx.y * gridDim.x + blockIdx.x, member = id % gridDim.y;
    trim_tile_of(id / gridDim.y, mode, ktrim, tilesM, tilesN, tm, tn);
    A += (size_t)member * sa;
    B += (size_t)member * sb;
    C += (size_t)member * sc;
  } else
  // (the triangle's enumeration needs square tiles; others drop what lies
  // outside it wave by wave)
  if (WM != WN || mode == 0) tile_of(blockIdx.x, gridDim.x, tilesM, tilesN, tm, tn);
  else tri_tile_of(blockIdx.x, mode, tilesM, tilesN, tm, tn);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sl = wave / NW, wt = wave % NW;
  const int m0 = tm * TM_ + GW_T * (wt % WM), n0 = tn * TN_ + GW_T * (wt / WM);
  const int fx = lane & 15, fk = lane >> 4;
  typename MF::acc_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = typename MF::acc_t{0, 0, 0, 0};
  // a wave whose tile lies outside C (or the triangle) has nothing to add
  bool live = m0 < M && n0 < N;
  if (mode == 1 && m0 + GW_T - 1 < n0) live = false;
  if (mode == 2 && n0 + GW_T - 1 < m0) live = false;
  if (live) {
    GwOperand<S, !AT> oa;
    GwOperand<S, BT> ob;
    oa.init(A, lda, m0, M, fx, fk);
    ob.init(B, ldb, n0, N, fx, fk);
    const int full = K / GW_K;
    int nch = (K + GW_K - 1) / GW_K, cb = 0;  // chunks, and the first
    if (XT) {
      if (ktrim & 1) cb = n0 / GW_K;
      if (ktrim & 2) cb = max(cb, m0 / GW_K);
      if (ktrim & 4) nch = min(nch, (m0 + GW_T) / GW_K);
      nch = max(0, nch - cb);
    }
    const int c0 = cb + (int)((long)nch * sl / WS), c1 = cb + (int)((long)nch * (sl + 1) / WS);
    const int ce = min(c1, full);  // whole chunks [c0, ce)
    S a[2][4][2], b[2][4][2];
    auto mma = [&](int d) {
#pragma unroll
      for (int ks = 0; ks < 4; ks++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) acc[i][j] = MF::op(b[d][ks][j], a[d][ks][i], acc[i][j]);
    };
    if (c0 < ce) {
      // loads past the slice repeat its last chunk and are never used
      oa.load(c0 * GW_K, a[0]);
      ob.load(c0 * GW_K, b[0]);
      oa.load(min(c0 + 1, ce - 1) * GW_K, a[1]);
      ob.load(min(c0 + 1, ce - 1) * GW_K, b[1]);
      int c = c0;
      for (; c + 1 < ce; c += 2) {
#pragma unroll
        for (int d = 0; d < 2; d++) {
          mma(d);
          __builtin_amdgcn_sched_barrier(0);
          oa.load(min(c + 2 + d, ce - 1) * GW_K, a[d]);
          ob.load(min(c + 2 + d, ce - 1) * GW_K, b[d]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (c < ce) mma(0);
    }
    if (ce < c1) {  // the ragged end of K
      oa.load_tail(full * GW_K, K, a[0]);
      ob.load_tail(full * GW_K, K, b[0]);
      mma(0);
    }
  }
  if (WS > 1) {
    // slice sums in slice order: wave (sl, wt) finishes the accumulators
    // e = sl, sl + WS, ... of tile wt
    S* mine = part + (size_t)(wt * WS + sl) * 16 * 64 + lane;
#pragma unroll
    for (int e = 0; e < 16; e++) mine[64 * e] = acc[e >> 3][(e >> 2) & 1][e & 3];
    __syncthreads();
  } else if (WM != WN) {
    __syncthreads();  // C may be B (WM x 1) or A (1 x WN): reads precede writes
  }
  if (!live) return;
#pragma unroll
  for (int e0 = 0; e0 < 16; e0 += WS) {
    // WS == 1: the accumulators themselves; else one sum per round
    const int e = WS > 1 ? e0 + sl : e0;
    S v;
    if (WS > 1) {
      const S* p = part + (size_t)wt * WS * 16 * 64 + 64 * e + lane;
      v = p[0];
#pragma unroll
      for (int s = 1; s < WS; s++) v += p[(size_t)s * 16 * 64];
    } else {
      v = acc[e0 >> 3][(e0 >> 2) & 1][e0 & 3];
    }
    const int i = e >> 3, j = (e >> 2) & 1, r = e & 3;
    const int gi = m0 + 16 * i + c_m(lane), gj = n0 + 16 * j + MF::c_n(lane, r);
    if (gi >= M || gj >= N || (mode == 1 && gi < gj) || (mode == 2 && gi > gj)) continue;
    S* c = C + (size_t)gi + (size_t)gj * ldc;
    const S w = alpha * v;
    *c = (beta == S(0)) ? w : w + beta * (*c);
  }
}
