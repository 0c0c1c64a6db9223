// Triangular solve with few right-hand sides in one launch; included by
// trsm.hip.
//
// What bounds such a solve: a chain over the diagonal blocks.  The blocked
// recursion pays two launches per 128-row block (order 1000: 16 launches,
// about 70 us more than this launch).  Here workgroup li of a group owns 64
// rows and the group's 16 right-hand sides; it folds in each earlier block as
// it appears, applies its block's inverse and publishes its rows.  Four waves
// multiply (16 rows each, one wave per SIMD, 16 MFMAs per block), four others
// fetch the solved blocks: with both in one wave the in-order load counter
// makes every poll wait for the next block of op(A) as well (order 2048,
// transposed: 112 us against 88).  The block solved right before this one is
// multiplied by -inv(A_pp) A_pq, formed ahead, so that its product does not
// wait for a pass through the inverse.  A step of the chain is one exchange,
// two LDS passes and two products of 1024 cycles (inv(A_pp) times what the
// earlier blocks left starts at the barrier that the last one's arrival opens):
// 1.8 us measured.
// 128-row blocks double the product and spill.  Orders 500 / 1000 / 2048
// with 3 right-hand sides take 40 / 55 / 85 us (27 of each: the inverses),
// by blocked launches 148 / 341 and, four right-hand sides at most, 141 us.
//
// The exchange area starts out filled with a sentinel, a signalling NaN that
// no result can equal (results pass through canonicalize); each word is
// stored once and polled, without flags, with agent-scope accesses.  The
// workgroups of a group are 8 apart, which puts them on one XCD: faster, not
// needed for correctness (stores that stop at that XCD's L2 would save a
// tenth, but rely on it).  A workgroup waits only for workgroups of smaller
// index, which were dispatched before it, so the launch needs no
// co-residency; the waits are bounded as the other kernels'.
#pragma once

constexpr int kTxB = 64;                    // rows per workgroup
constexpr int kTxCols = 16;                 // right-hand sides per group
constexpr int kTxGroups = 8;                // groups side by side, an XCD each
constexpr int kTxWaves = kTxB / 16;           // multiplying waves; as many fetch
constexpr int kTxThreads = 2 * 64 * kTxWaves;
constexpr int kTxLd = kTxCols + 1;          // LDS pitch of a block of right-hand sides
constexpr long kTxBlock = kTxB * kTxCols;   // words of one block in the exchange area
typedef unsigned long long tx_word;
constexpr tx_word kTxSent = 0x7FF4A5A5A5A5A5A5ull;
static_assert(NB % kTxB == 0, "an inverted block holds whole row blocks");

__global__ void tx_reset(tx_word* x, long n, int* err) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n;
       e += (long)gridDim.x * blockDim.x)
    __hip_atomic_store(x + e, kTxSent, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (blockIdx.x == 0 && threadIdx.x == 0) st_flag(err, 0);
}

// A 16 x 64 operand of 16 MFMA steps: lane (n, k) holds row n at columns
// 16 c + 4 k + s (any order of the columns serves while both operands agree;
// this one gives a lane four adjacent columns).
template <class S>
struct TxRows {
  S v[kTxB / 16][4];
  // element (row n, column k) at p[k * step] (STEP1: step is 1, and a block
  // known to be full takes a lane's four columns by 16-byte loads: transposed,
  // order 2500 with 1701 right-hand sides 502 -> 453 us); rows and columns
  // outside are zero
  template <bool STEP1>
  __device__ __forceinline__ void load(const S* __restrict__ p, long step, int lk, int cols, bool in,
                                       bool full) {
    if (STEP1 && full) {
#pragma unroll
      for (int c = 0; c < kTxB / 16; c++) {
        typedef S quad __attribute__((ext_vector_type(4), aligned(sizeof(S))));
        const quad w = *reinterpret_cast<const quad*>(p + 16 * c + 4 * lk);
#pragma unroll
        for (int s = 0; s < 4; s++) v[c][s] = w[s];
      }
      return;
    }
#pragma unroll
    for (int c = 0; c < kTxB / 16; c++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int k = 16 * c + 4 * lk + s;
        v[c][s] = in && k < cols ? p[(size_t)k * (STEP1 ? 1 : step)] : S(0);
      }
  }
};

// Column (of 16) that lane ln supplies as a step's row, for accumulator
// register s of lane (n, k) to be column 4 k + s.
template <class S>
__device__ __forceinline__ int tx_lane_col(int ln) {
  return sizeof(S) == 8 ? 4 * (ln & 3) + (ln >> 2) : ln;
}

// FOLD: the last block's product is folded into the inverse (see above)
template <class S, bool TR, bool FOLD>
__global__ void __launch_bounds__(kTxThreads)
trsv_xcd(int n, int nb, int nrhs, int gpad, int upper, S alpha, const S* __restrict__ A, long lda,
         const S* __restrict__ Dinv, int dtrans, S* __restrict__ B, long bi, long bj,
         tx_word* __restrict__ xb, int* __restrict__ err, int* __restrict__ status, int* info,
         long limit, const int* skip) {  // (info may be skip)
  typedef TriMfma<S> M;
  typedef typename M::acc_t acc_t;
  const int grp = blockIdx.x % gpad, li = blockIdx.x / gpad;
  const int c0 = grp * kTxCols;  // the group's first right-hand side
  if (c0 >= nrhs || (skip && *skip)) return;
  const int nc = min(kTxCols, nrhs - c0);
  __shared__ S xs[2][kTxB * kTxLd], ys[kTxB * kTxLd];
  __shared__ S al[FOLD ? kTxB : 1][kTxB + 1];
  __shared__ int bad;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int ln = lane & 15, lk = lane >> 4;
  const int p = upper ? nb - 1 - li : li;  // li counts in solve order
  const int r0 = p * kTxB, rows = min(kTxB, n - r0);
  if (t == 0) bad = 0;
  xb += (size_t)grp * nb * kTxBlock;
  if (w >= kTxWaves) {  // fetch the solved blocks: right-hand sides v, v + 4, ..., a row per lane
    const int v = w - kTxWaves;
    lds_barrier();
    for (int lj = 0; lj < li; lj++) {
      const tx_word* src = xb + (size_t)lj * kTxBlock + lane;
      tx_word x[4];
      long spins = 0;
      for (bool miss = true; miss;) {
        miss = false;
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int c = v + 4 * u;
          x[u] = c < nc ? __hip_atomic_load(const_cast<tx_word*>(src) + c * kTxB, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT)
                        : 0ull;
          miss = miss || x[u] == kTxSent;
        }
        miss = __any(miss);
        if (miss && (++spins >= limit || ((spins & 255) == 0 && ld_flag(err)))) {
          st_flag(err, 1);
          bad = 1;
          miss = false;
        }
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
        xs[lj & 1][lane * kTxLd + v + 4 * u] =
            (S)__longlong_as_double(static_cast<long long>(x[u]));
      if (FOLD && lj + 1 == li) lds_barrier();
      lds_barrier();
      if (bad) return;
    }
    if (!FOLD) lds_barrier();
    return;
  }
  const int row = 16 * w + ln;
  const bool in = row < rows;
  // this wave's rows of op(A), of the block's inverse, of the right-hand sides
  TxRows<S> a0, a1, d, f;
  auto load_a = [&](TxRows<S>& a, int lj) {
    const int q0 = (upper ? nb - 1 - lj : lj) * kTxB;
    const bool full = rows == kTxB && n - q0 >= kTxB;
    if (TR)
      a.template load<true>(A + (size_t)(r0 + row) * lda + q0, 1, lk, n - q0, in, full);
    else
      a.template load<false>(A + (r0 + row) + (size_t)q0 * lda, lda, lk, n - q0, in, full);
  };
  if (FOLD && li > 0) load_a(f, li - 1);
  const S* D = Dinv + (size_t)(r0 / NB) * NB * NB + (size_t)(r0 % NB) * (NB + 1);
  if (dtrans)
    d.template load<true>(D + (size_t)row * NB, 1, lk, rows, in, rows == kTxB);
  else
    d.template load<false>(D + row, NB, lk, rows, in, rows == kTxB);
  S rhs[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int c = M::row(lane, r);
    rhs[r] = in && c < nc ? alpha * B[(r0 + row) * bi + (c0 + c) * bj] : S(0);
  }
  const int ls = FOLD ? li - 1 : li;  // blocks folded in one by one
  if (ls > 0) load_a(a0, 0);
  if (ls > 1) load_a(a1, 1);
  acc_t acc, acc2;
  auto mul = [&](const S* xl, const TxRows<S>& m) {
#pragma unroll
    for (int c = 0; c < kTxB / 16; c++)
#pragma unroll
      for (int s = 0; s < 4; s += 2) {
        acc = M::op(xl[(16 * c + 4 * lk + s) * kTxLd + ln], m.v[c][s], acc);
        acc2 = M::op(xl[(16 * c + 4 * lk + s + 1) * kTxLd + ln], m.v[c][s + 1], acc2);
      }
  };
  // f = -inv(A_pp) A_pq, q the block solved right before this one: one product
  // only follows q on the chain
  if (FOLD && li > 0) {
#pragma unroll
    for (int c = 0; c < kTxB / 16; c++)
#pragma unroll
      for (int s = 0; s < 4; s++) al[row][16 * c + 4 * lk + s] = -f.v[c][s];
  }
  lds_barrier();
  if (FOLD && li > 0) {
    const int fm = tx_lane_col<S>(ln);
#pragma unroll
    for (int c = 0; c < kTxB / 16; c++) {
      acc = acc2 = acc_t{0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < kTxB / 16; e++)
#pragma unroll
        for (int s = 0; s < 4; s += 2) {
          acc = M::op(al[16 * e + 4 * lk + s][16 * c + fm], d.v[e][s], acc);
          acc2 = M::op(al[16 * e + 4 * lk + s + 1][16 * c + fm], d.v[e][s + 1], acc2);
        }
#pragma unroll
      for (int s = 0; s < 4; s++) f.v[c][s] = acc[s] + acc2[s];
    }
  }
  acc = acc2 = acc_t{0, 0, 0, 0};
  auto step = [&](TxRows<S>& a, int lj) -> bool {
    lds_barrier();
    if (bad) return false;
    mul(xs[lj & 1], a);
    if (lj + 2 < ls) load_a(a, lj + 2);
    return true;
  };
  bool ok = true;
  for (int lj = 0; lj < ls && ok; lj += 2) {
    ok = step(a0, lj);
    if (ok && lj + 1 < ls) ok = step(a1, lj + 1);
  }
  if (ok) {
    // inv(A_pp) (alpha b - the blocks before q), then q's share
#pragma unroll
    for (int r = 0; r < 4; r++)
      ys[row * kTxLd + M::row(lane, r)] = in ? rhs[r] - (acc[r] + acc2[r]) : S(0);
    lds_barrier();
    acc = acc2 = acc_t{0, 0, 0, 0};
    mul(ys, d);
    if (FOLD && li > 0) {
      lds_barrier();
      ok = !bad;
      mul(xs[(li - 1) & 1], f);
    }
  }
  if (!ok) {
    if (t == 0) {
      atomicOr(status, ATLG_FAIL_TRSV);
      if (info) *info = INT_MIN;
    }
    return;
  }
  tx_word* out = xb + (size_t)li * kTxBlock + row;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int c = M::row(lane, r);
    const S x = __builtin_canonicalize(acc[r] + acc2[r]);
    if (c < nc) {
      __hip_atomic_store(out + c * kTxB, static_cast<tx_word>(__double_as_longlong((double)x)),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (in) B[(r0 + row) * bi + (c0 + c) * bj] = x;
    }
  }
}

// Largest order solved in one launch.  Longer triangles are halved first, so
// that the whole device reads what lies off the diagonal blocks; the more
// right-hand sides, the more its large products save over the 16-column
// groups, which take turns on a compute unit.  Order 2500 by launches up to
// order 2048 / 1024 / 512 / none: 200 right-hand sides 152 / 178 / 220 / 347
// us, 500 181 / 208 / 251 / 375, 1701 455 / 425 / 492 / 549, 2500 - / 567 /
// 597 / 669, 4000 - / 831 / 828 / 842; order 4096, transposed, 500 467 / 436.
inline long tx_order(long nrhs) {
  return nrhs <= 384 ? 2048 : nrhs <= 3072 ? 1024 : nrhs <= 4096 ? 512 : 0;
}
// The largest exchange area that this asks for (kNoAllocTxBlocks blocks), with
// its error word.
constexpr size_t kTxFixedBytes = 256 + sizeof(tx_word) * kTxBlock * kNoAllocTxBlocks;
static_assert(kNoAllocTxBlocks >= 384 / kTxCols * (2048 / kTxB) &&
              kNoAllocTxBlocks >= 3072 / kTxCols * (1024 / kTxB) &&
              kNoAllocTxBlocks >= 4096 / kTxCols * (512 / kTxB), "fixed exchange area");
static_assert(kTxFixedBytes + 4 * kNoAllocWords == kNoAllocTxBytes, "fixed exchange area");

// Solves op(A) X = alpha B, op(A) lower (or upper) triangular of order n <=
// tx_order(nrhs), element (i, j) of X and B at i bi + j bj; Dinv holds the inverses
// of op(A)'s NB x NB diagonal blocks, or their transposes (dtrans).  `fixed`,
// when not null, is memory for the exchange area (kTxFixedBytes) in place of
// the stream's own.  False, with nothing queued,
// where the exchange area cannot be had.
template <class S>
bool trsv_one_launch(hipStream_t s, bool lower, bool tr, long n, long nrhs, S alpha, const S* A,
                     long lda, const S* Dinv, int dtrans, S* B, long bi, long bj, const int* skip,
                     const WaitReport& rep, unsigned char* fixed) {
  const int nb = (int)((n + kTxB - 1) / kTxB);
  const int groups = (int)((nrhs + kTxCols - 1) / kTxCols);
  const long words = (long)groups * nb * kTxBlock;
  tx_word* xb = static_cast<tx_word*>(
      fixed ? fixed
            : scratch_in_capture(s, kSlotTrsv, 256 + sizeof(tx_word) * words, !rep.status));
  if (!xb) return false;
  int* err = reinterpret_cast<int*>(xb);
  xb += 256 / sizeof(tx_word);
  hipLaunchKernelGGL(tx_reset, dim3((unsigned)std::min(256L, (words + 511) / 512)), dim3(512), 0,
                     s, xb, words, err);
  ATLG_LAUNCHED();
  const int gpad = (groups + kTxGroups - 1) / kTxGroups * kTxGroups;
  const dim3 grid(gpad * (nb - 1) + groups), block(kTxThreads);
  const int up = lower ? 0 : 1;
  int* status = rep.status ? rep.status : status_word(s);
  const long limit = wait_limit(kSvSpin);
  // more groups than XCDs: throughput counts, and folding adds to the products
  const bool fold = groups <= kTxGroups;
  const auto fn = tr ? (fold ? trsv_xcd<S, true, true> : trsv_xcd<S, true, false>)
                     : (fold ? trsv_xcd<S, false, true> : trsv_xcd<S, false, false>);
  hipLaunchKernelGGL(fn, grid, block, 0, s, (int)n, nb, (int)nrhs, gpad, up, alpha, A, lda, Dinv,
                     dtrans, B, bi, bj, xb, err, status, rep.info, limit, skip);
  ATLG_LAUNCHED();
  return true;
}
