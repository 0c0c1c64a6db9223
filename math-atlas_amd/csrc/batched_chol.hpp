// One workgroup's Cholesky factorization of one system, and its triangular
// sweeps with right-hand sides in LDS; included by batched.hip.
//
// Left-looking by block columns of 64: four column tiles of 16.  All tiles
// are kept in one layout, lane (n, k) = (l & 15, l >> 4) holding row n and
// the columns 4 b + k in register b, which makes a register the 4x16 operand
// of a 16x16x4 MFMA as it is: a row tile goes through
//   acc = sum over earlier columns (operands straight from memory),
//   X_c = (acc_c - A_c) (-inv(L_cc)^T), acc_e += X_c L_ec^T for e > c
// without leaving its registers.  Wave i starts with row tile i of the
// diagonal block: wave c factors tile (c, c) and inverts it, the waves below
// solve and subtract, then every wave takes row tiles of its own until the
// block column is done.
//
// What bounds it: alone, the chain of pivots and the latency of the operand
// loads; with every compute unit full, the reads of earlier columns (n^3/384
// elements a system, from memory once the systems outgrow the caches) and the
// matrix cores.  64 columns rather than 32 halve those reads.
#pragma once

constexpr int kTile = 16;
constexpr int kColT = 4;                 // column tiles of a block column, one per wave
constexpr int kWide = kTile * kColT;
constexpr int kTP = kTile + 1;           // LDS pitch of a tile
constexpr int kTileLds = kTile * kTP;
static_assert(kColT == kBW, "wave i starts with row tile i of the diagonal block");

// The lane's index, computed where it is used: the compiler otherwise hoists
// every phase's lane-dependent addresses out of the loop over the systems and
// spills them (536 bytes a lane).
__device__ __forceinline__ int lane_here() {
  int l = threadIdx.x & 63;
  asm volatile("" : "+v"(l));
  return l;
}

// Row (or column) of a tile that lane ln supplies as the 16x4 operand, for
// the accumulators to be in the layout above.
template <class S>
__device__ __forceinline__ int tile_row(int ln) {
  return sizeof(S) == 8 ? ln : 4 * (ln & 3) + (ln >> 2);
}
// LDS tile (i, c), i > c, of the diagonal block; tiles 6 .. 9 are the
// negated inverses of the diagonal tiles, tile 10 the latest diagonal tile.
__device__ __forceinline__ int low_tile(int i, int c) { return i * (i - 1) / 2 + c; }

// 1/sqrt(d), d > 0: the hardware estimate (about 2^-23) and one third-order
// step; the products stay in range for subnormal d.
__device__ __forceinline__ double rsqrt3(double d) {
  const double y = __builtin_amdgcn_rsq(d);
  const double e = __builtin_fma(-(d * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}

// Factors a tile held in the layout above, in FP64 for both types (so the
// accumulators serve as both operands), four columns at a time as the
// Cholesky leaf of potrf does: the 4x4 block by every lane alike, the rows
// below by its inverse, an identity tile carried along to the inverse.
// Stores L to F and -inv(L) to V (pitch kTP); returns the first non-positive
// pivot's index, or -1.
template <class S>
__device__ __forceinline__ int factor_tile(d4 T, S* F, S* V) {
  typedef Mfma<double> M;
  const int lane = lane_here(), ln = lane & 15, lk = lane >> 4;
  const d4 zero = {0, 0, 0, 0};
  d4 Z;
#pragma unroll
  for (int b = 0; b < 4; b++) Z[b] = ln == 4 * b + lk ? 1.0 : 0.0;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    double a[4][4], r[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = j; i < 4; i++) a[i][j] = tri_lane(T[b], 16 * j + 4 * b + i);
    int bad = -1;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (!(a[j][j] > 0.0) && bad < 0) bad = 4 * b + j;
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
    if (bad >= 0) return bad;
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
    const d4 x = M::op(wo, T[b], zero);
    const d4 z = M::op(wo, Z[b], zero);
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int c = 0; c <= i; c++) F[(4 * b + i) * kTP + 4 * b + c] = (S)a[i][c];
    }
    const double xm = ln >= 4 * b + 4 ? x[0] : 0.0;
    if (b < 3) {
      T = M::op(-xm, xm, T);
      Z = M::op(-xm, z[0], Z);
    }
    if (ln >= 4 * b + 4) F[ln * kTP + 4 * b + lk] = (S)xm;
    V[(4 * b + lk) * kTP + ln] = (S)-z[0];
  }
  return -1;
}

// acc += (tile at P, pitch kTP, as the columns) times X
template <class S>
__device__ __forceinline__ typename Mfma<S>::acc_t tile_mul(const S* P, const typename Mfma<S>::acc_t& X,
                                                            typename Mfma<S>::acc_t acc) {
  const int lane = lane_here();
  const S* p = P + tile_row<S>(lane & 15) * kTP + (lane >> 4);
#pragma unroll
  for (int s = 0; s < 4; s++) acc = Mfma<S>::op(p[4 * s], X[s], acc);
  return acc;
}
// Lane (n, k) of the result: row n of X times right-hand side k of the 16
// rows of y (LDS, [row][4])
template <class S>
__device__ __forceinline__ S tile_rhs(const S* y, const typename Mfma<S>::acc_t& X) {
  const int lane = lane_here(), q = tile_row<S>(lane & 15), lk = lane >> 4;
  typename Mfma<S>::acc_t D = {0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const S v = y[(4 * s + lk) * 4 + (q & 3)];
    D = Mfma<S>::op(q < 4 ? v : S(0), X[s], D);
  }
  return D[0];
}

// R row tiles from row0 on, their first NC column tiles of block column J:
// acc = L[rows, 0:J] L[J:J+64, 0:J]^T.  A's tile is subtracted when its column
// tile is due: sums of products alone round less.  Rows past the end are
// clamped (their results are not used).
template <class S, int R, int NC>
__device__ __forceinline__ void row_tiles(int n, const S* __restrict__ A, size_t lda, int J, int row0,
                                          typename Mfma<S>::acc_t (&acc)[R][kColT]) {
  typedef Mfma<S> M;
  const int lane = lane_here(), ln = lane & 15, lk = lane >> 4;
  const S *pr[R], *pc[NC];
#pragma unroll
  for (int h = 0; h < R; h++) pr[h] = A + min(row0 + kTile * h + ln, n - 1) + lk * lda;
#pragma unroll
  for (int c = 0; c < NC; c++)
    pc[c] = A + min(J + kTile * c + tile_row<S>(ln), n - 1) + lk * lda;
  // G steps of four columns multiply while the next G load: 1024 cycles of
  // FP64 MFMAs ahead
  constexpr int G = R == 1 ? 4 : 2;
  S xr[2][G][R], xc[2][G][NC];
  auto load = [&](int u) {
#pragma unroll
    for (int g = 0; g < G; g++) {
#pragma unroll
      for (int h = 0; h < R; h++) {
        xr[u][g][h] = *pr[h];
        pr[h] += 4 * lda;
      }
#pragma unroll
      for (int c = 0; c < NC; c++) {
        xc[u][g][c] = *pc[c];
        pc[c] += 4 * lda;
      }
    }
  };
  auto mul = [&](int u) {
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int h = 0; h < R; h++) acc[h][c] = M::op(xc[u][g][c], xr[u][g][h], acc[h][c]);
  };
  if (J > 0) load(0);
#pragma unroll
  for (int h = 0; h < R; h++)
#pragma unroll
    for (int c = 0; c < NC; c++) acc[h][c] = typename M::acc_t{0, 0, 0, 0};
  for (int k = 0; k < J; k += 8 * G) {  // J is a multiple of kWide
    load(1);
    mul(0);
    if (k + 8 * G < J) load(0);
    mul(1);
  }
}
// The tile of A at row (clamped to the matrix) and column col0, columns right
// of the diagonal clamped.
template <class S>
__device__ __forceinline__ typename Mfma<S>::acc_t a_tile(int n, const S* A, size_t lda, int row,
                                                          int col0, int lk) {
  typename Mfma<S>::acc_t a;
  row = min(row, n - 1);
#pragma unroll
  for (int b = 0; b < 4; b++) a[b] = A[row + min(col0 + 4 * b + lk, row) * lda];
  return a;
}

// Row tiles below the diagonal block: accumulate, solve, store, and take the
// block column's share off their right-hand sides.
template <class S, int R>
__device__ __forceinline__ void lower_tiles(int n, S* __restrict__ A, size_t lda, int J, int row0,
                                            const S* lt, S* Y) {
  typedef typename Mfma<S>::acc_t acc_t;
  const int lane = lane_here(), ln = lane & 15, lk = lane >> 4;
  acc_t acc[R][kColT], a0[R];
#pragma unroll
  for (int h = 0; h < R; h++) a0[h] = a_tile<S>(n, A, lda, row0 + kTile * h + ln, J, lk);
  row_tiles<S, R, kColT>(n, A, lda, J, row0, acc);
#pragma unroll
  for (int h = 0; h < R; h++) {
    const int row = row0 + kTile * h + ln;
    S* a = A + row + (size_t)(J + lk) * lda;
    S ys = S(0);
#pragma unroll
    for (int c = 0; c < kColT; c++) {
      const acc_t d = acc[h][c] - a0[h];
      if (c + 1 < kColT) a0[h] = a_tile<S>(n, A, lda, row, J + kTile * (c + 1), lk);
      const acc_t X = tile_mul<S>(lt + (6 + c) * kTileLds, d, acc_t{0, 0, 0, 0});
#pragma unroll
      for (int e = c + 1; e < kColT; e++)
        acc[h][e] = tile_mul<S>(lt + low_tile(e, c) * kTileLds, X, acc[h][e]);
      if (Y) ys += tile_rhs<S>(Y + (J + kTile * c) * 4, X);
      if (row < n) {
#pragma unroll
        for (int b = 0; b < 4; b++) a[(size_t)(kTile * c + 4 * b) * lda] = X[b];
      }
    }
    if (Y && row < n) Y[row * 4 + lk] -= ys;
  }
}

// Factors one system; returns 0 or the LAPACK info (first failing minor).
// Y, when not null: L Y = B is solved in place beside the factorization
// ([row][4] in LDS, n <= kYmax / 4).
// rows: a wave takes 16 or 32 of them at a time below the diagonal block.
template <class S>
__device__ __forceinline__ int chol_sys(int n, S* __restrict__ A, int lda_, int rows, Smem& sm, S* Y) {
  typedef typename Mfma<S>::acc_t acc_t;
  const size_t lda = (size_t)lda_;
  S* lt = reinterpret_cast<S*>(sm.LT);
  const int lane = lane_here(), ln = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int J = 0; J < n; J += kWide) {
    const int nt = min(kColT, (n - J + kTile - 1) / kTile);  // column tiles
    // the diagonal block, row tile `wave`
    const int row0 = J + kTile * wave, row = row0 + ln;
    acc_t acc[1][kColT], X = {0, 0, 0, 0};
    acc_t a0 = a_tile<S>(n, A, lda, row, J, lk);
    if (wave < nt) {
      if (wave == 0) row_tiles<S, 1, 1>(n, A, lda, J, row0, acc);
      else if (wave == 1) row_tiles<S, 1, 2>(n, A, lda, J, row0, acc);
      else if (wave == 2) row_tiles<S, 1, 3>(n, A, lda, J, row0, acc);
      else row_tiles<S, 1, 4>(n, A, lda, J, row0, acc);
    }
    if (threadIdx.x == 0) sm.flag = 0;
    for (int c = 0; c < nt; c++) {
      S* vt = lt + (6 + c) * kTileLds;
      if (wave == c) {
        d4 T;
#pragma unroll
        for (int b = 0; b < 4; b++) {
          S x = acc[0][0][b];
#pragma unroll
          for (int e = 1; e < kColT; e++) x = c == e ? acc[0][e][b] : x;
          T[b] = row < n ? (double)(a0[b] - x) : (ln == 4 * b + lk ? 1.0 : 0.0);
        }
        // the chain goes before the other waves' products
        __builtin_amdgcn_s_setprio(3);
        const int f = factor_tile<S>(T, lt + 10 * kTileLds, vt);
        __builtin_amdgcn_s_setprio(0);
        if (f >= 0 && lane == 0) sm.flag = row0 + f + 1;
      }
      lds_barrier();
      if (sm.flag) return sm.flag;
      if (wave == c) {
        const S* p = lt + 10 * kTileLds + ln * kTP + lk;
        S* g = A + row + (size_t)(row0 + lk) * lda;
#pragma unroll
        for (int b = 0; b < 4; b++)
          if (row < n && 4 * b + lk <= ln) g[(size_t)(4 * b) * lda] = p[4 * b];
        if (Y) {  // y_c = inv(L_cc) y_c, the last step's share first
          if (c > 0) {
            const S ys = tile_rhs<S>(Y + (row0 - kTile) * 4, X);
            if (row < n) Y[row * 4 + lk] -= ys;
            wave_sync();
          }
          acc_t V;
#pragma unroll
          for (int s = 0; s < 4; s++) V[s] = vt[ln * kTP + 4 * s + lk];
          const S y = -tile_rhs<S>(Y + row0 * 4, V);
          if (row < n) Y[row * 4 + lk] = y;
        }
      } else if (wave > c && wave < nt) {
        acc_t a = acc[0][0];
#pragma unroll
        for (int e = 1; e < kColT - 1; e++) a = c == e ? acc[0][e] : a;
        a -= a0;
        a0 = a_tile<S>(n, A, lda, row, J + kTile * (c + 1), lk);  // for the next step
        X = tile_mul<S>(vt, a, acc_t{0, 0, 0, 0});
        S* p = lt + low_tile(wave, c) * kTileLds + ln * kTP + lk;
        S* g = A + row + (size_t)(J + kTile * c + lk) * lda;
#pragma unroll
        for (int b = 0; b < 4; b++) {
          p[4 * b] = X[b];
          if (row < n) g[(size_t)(4 * b) * lda] = X[b];
        }
      }
      lds_barrier();
      if (wave > c && wave < nt) {
#pragma unroll
        for (int e = 1; e < kColT; e++)
          if (e > c && e <= wave)
            acc[0][e] = tile_mul<S>(lt + low_tile(e, c) * kTileLds, X, acc[0][e]);
        if (Y && wave > c + 1) {
          const S ys = tile_rhs<S>(Y + (J + kTile * c) * 4, X);
          if (row < n) Y[row * 4 + lk] -= ys;
        }
      }
    }
    // the rows below
    const int RT = (n - J + kTile - 1) / kTile;
    int rt = kColT;
    for (; rows == 2 * kTile && RT - rt >= 2 * kBW; rt += 2 * kBW)
      lower_tiles<S, 2>(n, A, lda, J, J + kTile * (rt + 2 * wave), lt, Y);
    for (rt += wave; rt < RT; rt += kBW) lower_tiles<S, 1>(n, A, lda, J, J + kTile * rt, lt, Y);
    __syncthreads();  // the columns are in memory, the tiles and Y free
  }
  return 0;
}

// lane j of each 16 lanes to all of them
template <int J>
__device__ __forceinline__ float row_lane(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + J, 0xf, 0xf, false));
}
template <int J>
__device__ __forceinline__ double row_lane(double v) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)u, 0x150 + J, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), 0x150 + J, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// Solves the 16 unknowns of a diagonal tile, lane (i, k): row i, right-hand
// sides k, 4 + k, ...  x[j]: the row's entries of already solved unknowns,
// else zero.
template <class S, bool TR, int NG, int STEP = 0>
__device__ __forceinline__ void tile_solve(S (&y)[NG], const S (&x)[kTile], S rinv) {
  if constexpr (STEP < kTile) {
    constexpr int j = TR ? kTile - 1 - STEP : STEP;
#pragma unroll
    for (int g = 0; g < NG; g++) y[g] -= x[j] * row_lane<j>(y[g] * rinv);
    tile_solve<S, TR, NG, STEP + 1>(y, x, rinv);
  } else {
#pragma unroll
    for (int g = 0; g < NG; g++) y[g] *= rinv;
  }
}

// L Y = B or (TR) L^T Y = B in place for up to 4 NG right-hand sides, Y in LDS
// as [row][4 NG] or (GLB) in memory, nr columns of leading dimension ldy.
// By blocks of 64 unknowns: every wave sums a share of the solved ones'
// products on the matrix cores, then wave t has tile t of the block and the
// tiles are solved in turn.
template <class S, bool TR, bool GLB, int NG = 1>
__device__ __forceinline__ void sweep(int n, const S* __restrict__ L, int lda_, Smem& sm, S* Y,
                                      size_t ldy = 0, int nr = 4 * NG) {
  constexpr int NQ = 4 * NG;
  static_assert(sizeof(S) * kBW * kWide * NQ <= sizeof(sm.LT), "partial sums");
  typedef Mfma<S> M;
  typedef typename M::acc_t acc_t;
  const size_t lda = (size_t)lda_;
  S* P = reinterpret_cast<S*>(sm.LT);  // [wave][tile][row][NQ]
  const int lane = lane_here(), ln = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = tile_row<S>(ln);
  auto at = [&](int i, int q) -> S& { return GLB ? Y[i + min(q, nr - 1) * ldy] : Y[i * NQ + q]; };
  auto barrier = [&] {
    if (GLB) __syncthreads();
    else lds_barrier();
  };
  const int nb = (n + kWide - 1) / kWide;
  for (int s = 0; s < nb; s++) {
    const int J = kWide * (TR ? nb - 1 - s : s);
    const int nt = min(kColT, (n - J + kTile - 1) / kTile);
    const int t = TR ? nt - 1 - wave : wave;  // this wave's tile, solved wave-th
    const int row = J + kTile * t + ln;
    const bool in = wave < nt && row < n;
    // the solved unknowns' products, 16 at a time
    const int k0 = TR ? J + kWide : 0, kn = TR ? n : J;
    acc_t acc[kColT];
#pragma unroll
    for (int c = 0; c < kColT; c++) acc[c] = acc_t{0, 0, 0, 0};
    // (half a chunk multiplies while the next half loads)
    S v[2][kColT][2], yv[2][2];
    auto load = [&](int b, int k) {
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const int kk = TR ? k + 4 * lk + 2 * b + u : k + 8 * b + 4 * u + lk;
        const int kc = min(kk, n - 1);
#pragma unroll
        for (int c = 0; c < kColT; c++) {
          const int i = min(J + kTile * c + ln, n - 1);
          v[b][c][u] = TR ? L[kc + i * lda] : L[i + kc * lda];
        }
        const S y = at(kc, q & (NQ - 1));
        yv[b][u] = q < NQ && kk < kn ? y : S(0);
      }
    };
    auto mul = [&](int b) {
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int c = 0; c < kColT; c++) acc[c] = M::op(yv[b][u], v[b][c][u], acc[c]);
    };
    int k = k0 + kTile * wave;
    if (k < kn) {
      load(0, k);
      load(1, k);
    }
    for (; k < kn; k += kWide) {
      mul(0);
      if (k + kWide < kn) load(0, k + kWide);
      mul(1);
      if (k + kWide < kn) load(1, k + kWide);
    }
    // this wave's diagonal tile
    S x[kTile], rinv = S(0);
#pragma unroll
    for (int j = 0; j < kTile; j++) {
      const int c = J + kTile * t + j, r = in ? row : 0;
      const S v = TR ? L[max(min(c, n - 1), r) + r * lda] : L[r + max(min(c, r), 0) * lda];
      x[j] = in && c < n && (TR ? j > ln : j < ln) ? v : S(0);
    }
    if (in) rinv = L[row + row * lda];
    if (kn > k0) {
#pragma unroll
      for (int c = 0; c < kColT; c++)
#pragma unroll
        for (int g = 0; g < NG; g++)
          P[((wave * kColT + c) * kTile + ln) * NQ + 4 * g + lk] = acc[c][g];
      barrier();
    }
    S y[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) y[g] = S(0);
    if (in) {
      rinv = S(1) / rinv;
#pragma unroll
      for (int g = 0; g < NG; g++) {
        y[g] = at(row, 4 * g + lk);
        if (kn > k0) {
#pragma unroll
          for (int u = 0; u < kBW; u++)
            y[g] -= P[((u * kColT + t) * kTile + ln) * NQ + 4 * g + lk];
        }
      }
    }
    for (int d = 0; d < nt; d++) {  // tiles in solve order
      const int td = J + kTile * (TR ? nt - 1 - d : d);
      S o[kTile];
      if (wave > d && wave < nt) {
#pragma unroll
        for (int j = 0; j < kTile; j++) {
          const int c = min(td + j, n - 1), r = in ? row : n - 1;
          o[j] = TR ? L[max(c, r) + r * lda] : L[r + min(c, r) * lda];
        }
      }
      if (wave == d) {
        tile_solve<S, TR, NG>(y, x, rinv);
#pragma unroll
        for (int g = 0; g < NG; g++)
          if (in && 4 * g + lk < nr) at(row, 4 * g + lk) = y[g];
      }
      barrier();
      if (wave > d && wave < nt) {
#pragma unroll
        for (int j = 0; j < kTile; j++)
          if (td + j < n) {
#pragma unroll
            for (int g = 0; g < NG; g++) y[g] -= o[j] * at(td + j, 4 * g + lk);
          }
      }
    }
  }
}

// The symmetric FP64 matrix of the mixed solver, by tiles of 16 of its rows:
// f(kk, v) sees row 16 t + ln against each index kk < n of its 16-index chunk
// u times, lane quarter lk at kk = 4 u + lk of the chunk (left of the diagonal
// tile and in it) or 4 lk + u (below, read by columns), so that 16 lanes
// read 128 contiguous bytes either way.
template <class F>
__device__ __forceinline__ void sym_row_tile(int n, const double* __restrict__ A, size_t lda, int t,
                                             F f) {
  const int lane = lane_here(), ln = lane & 15, lk = lane >> 4;
  const int nt = (n + kTile - 1) / kTile, i = min(kTile * t + ln, n - 1);
  double v[2][4];
  auto index = [&](int kt, int u) { return kTile * kt + (kt > t ? 4 * lk + u : 4 * u + lk); };
  auto load = [&](int b, int kt) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int kk = min(index(kt, u), n - 1);
      v[b][u] = A[max(i, kk) + min(i, kk) * lda];
    }
  };
  auto use = [&](int b, int kt) {
#pragma unroll
    for (int u = 0; u < 4; u++) f(index(kt, u), v[b][u]);
  };
  load(0, 0);
  for (int kt = 0; kt < nt; kt += 2) {
    if (kt + 1 < nt) load(1, kt + 1);
    use(0, kt);
    if (kt + 1 >= nt) break;
    if (kt + 2 < nt) load(0, kt + 2);
    use(1, kt + 1);
  }
}
