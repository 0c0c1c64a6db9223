// LU leaf panel of up to kXpRows rows held in registers by workgroups of one
// XCD, included by getrf.hip.
//
// What bounds a leaf: the chain of its columns, each a pivot search over all
// rows, an exchange, and a rank-1 update.  panel_coop (taller panels) spends
// 3.8 us per column in one workgroup and 4.6 us in many: a row per lane means
// that every lane reads all 32 entries of the pivot row from LDS, and an
// agent-scope exchange travels through device memory because the workgroups
// sit on different XCDs.  Here
//
//  * the rows are held in the layout of the matrix core's accumulator: a wave
//    has 64 rows x 32 columns, lane l the rows 16 rt + (l & 15), rt < 4, and
//    the columns 4 b + (l >> 4), b < 8.  Four consecutive columns (a block)
//    sit in the four 16-lane quarters of one register, which is exactly the
//    operand layout of a 16x16x4 MFMA: after the block's four columns are
//    factored with updates inside the block only (one FMA per row), one MFMA
//    per 16x16 tile applies all four to the columns right of the block;
//  * a row never moves between lanes: every row carries its current position
//    and interchanges only exchange positions; the rows are stored to their
//    final positions at the end;
//  * a column's exchange is six words per candidate (key, position and the
//    row's four block entries); the rest of a pivot row is published beside
//    the next columns and only needed at the block's end;
//  * one workgroup (M <= kXpRows1) exchanges through LDS alone.  More (at
//    most 16) must share an XCD, whose L2 all its compute units see:
//    workgroups are dealt to the XCDs in turn, so of a grid of 8 (G - 1) + 1
//    only every eighth works and the others leave at once.  Words are written
//    once per leaf.  They are polled with agent-scope loads, which pass the
//    compute unit's own cache, and stored with workgroup-scope stores, which
//    stop at the XCD's L2: an exchange of eight workgroups takes 840 cycles,
//    against 1500 with agent-scope stores and 2000 across XCDs (one line per
//    candidate, timed by itself).  The waits are bounded as panel_coop's are,
//    so a device that dealt the workgroups otherwise would report a failure;
//  * workgroups wait for each other only once all of a panel's are resident.
//    A full one fills a compute unit and sixteen take half an XCD's, so panels
//    of several streams or processes, or other kernels, may each hold units
//    that the others need.  A workgroup therefore first counts itself in and
//    waits, some milliseconds at most, for the others (xp_gather); when they
//    do not come all give up at once, and the first factors the panel alone,
//    in memory (xp_alone, 1.4 ms for 8192 rows).  The panel is unchanged until
//    the end, so nothing is lost, and no launch needs to be cooperative (N=1500
//    4.9 ms with that, 4.3 without; counting in costs a leaf 2 of its 80 us).
//    Successive factorizations take the XCDs in turn, to keep out of each
//    other's way.
//
// A column takes 4000-4500 cycles (about 1.8 us), most of it the issue of
// some 450 dependent instructions by one or two waves per SIMD.  M x 32 LU,
// set-up launches included (panel_coop -> here, by one measurement): M = 256
// 136 -> 74 us, 1000 168 -> 88, 4096 178 -> 88, 8192 186 -> 96; without the
// copies in it 59, 78, 80 and 94 us.  128 rows per wave (half the
// workgroups) did not fit the registers: 160 us at M = 1000.
#pragma once

constexpr int kXpMaxG = 16;                    // workgroups (one compute unit each)
constexpr int kXpWaves = 8;                    // most waves of a workgroup
constexpr int kXpRowsWg = 64 * kXpWaves;       // rows of a full workgroup
constexpr int kXpRows = kXpMaxG * kXpRowsWg;   // tallest panel
// Tallest panel of one workgroup, and rows per workgroup of a panel of
// several while the grid allows it (one wave per SIMD).
#ifndef ATLG_XP_ROWS1
#define ATLG_XP_ROWS1 512
#endif
constexpr int kXpRows1 = ATLG_XP_ROWS1;
static_assert(kXpRows1 <= kXpRowsWg, "one workgroup's rows");
#ifndef ATLG_XP_ROWS_PER_WG
#define ATLG_XP_ROWS_PER_WG 256
#endif
// The block-column arithmetic below is written for 32-column leaves.
constexpr int kXpW = 32;
static_assert(PW == kXpW, "leaf width of the XCD panel");
constexpr int kXpCand = 6;  // words of a candidate: key, position, four entries
constexpr int RT = 4;       // row tiles of a wave

typedef unsigned long long xp_word;
constexpr xp_word kXpSent = Word<double>::kSent;

// One leaf's exchange area.  Slots are written once per leaf; the next leaf,
// which uses the other area, refills them with sentinels.
struct XpBox {
  xp_word cand[kXpW][kXpCand][kXpMaxG];  // word-major: xp_pick reads a word per lane
  xp_word trail[kXpW][kXpW];  // pivot row of column j: its entries right of the block
  int err;
  int here;  // workgroups that have arrived, and kXpAlone
  int pad[14];
};
constexpr int kXpAlone = 1 << 16;
// Polls (each a round trip to the L2) before a panel's workgroups stop waiting
// for one of them to become resident.
constexpr long kXpGather = 1L << 13;

__device__ inline xp_word xp_ld(const xp_word* p) {
  return __hip_atomic_load(const_cast<xp_word*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void xp_st(xp_word* p, xp_word v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline xp_word xp_bits(double x) { return static_cast<xp_word>(__double_as_longlong(x)); }
__device__ inline double xp_val(xp_word u) { return __longlong_as_double(static_cast<long long>(u)); }
__device__ inline void xp_clear(XpBox* m, int t, int nt) {
  for (int e = t; e < kXpW * kXpCand * kXpMaxG; e += nt) xp_st(&m->cand[0][0][0] + e, kXpSent);
  for (int e = t; e < kXpW * kXpW; e += nt) xp_st(&m->trail[0][0] + e, kXpSent);
  if (t == 0) {
    st_agent(&m->err, 0);
    __hip_atomic_store(&m->here, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
}
__global__ void xp_init(XpBox* m) {
  xp_clear(m + blockIdx.x, threadIdx.x, blockDim.x);
}

__device__ __forceinline__ double xp_max(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float xp_max(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// pivot key: |x|, -1 for a (quiet) NaN (volatile: not moved into a branch)
__device__ __forceinline__ double xp_key(double x) {
  double r;
  asm volatile("v_max_f64 %0, |%1|, -1.0" : "=v"(r) : "v"(x));
  return r;
}
__device__ __forceinline__ float xp_key(float x) {
  float r;
  asm volatile("v_max_f32 %0, |%1|, -1.0" : "=v"(r) : "v"(x));
  return r;
}
// DPP moves within 16-lane rows whose source lanes all exist
template <int CTRL>
__device__ __forceinline__ float xp_dpp(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ double xp_dpp(double x) {
  const long long u = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp(static_cast<int>(u), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(static_cast<int>(u >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}
__device__ __forceinline__ double xp_lane(double x, int l) { return readlane_d(x, l); }
__device__ __forceinline__ float xp_lane(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}
// value of the lane at byte address 4 * lane
__device__ __forceinline__ float xp_from(int addr, float x) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(x)));
}
__device__ __forceinline__ double xp_from(int addr, double x) {
  const long long u = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_ds_bpermute(addr, static_cast<int>(u));
  const int hi = __builtin_amdgcn_ds_bpermute(addr, static_cast<int>(u >> 32));
  return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}
// largest value of each 16-lane row, in all its lanes
template <class S>
__device__ __forceinline__ S xp_row_max(S x) {
  x = xp_max(x, xp_dpp<0xB1>(x));
  x = xp_max(x, xp_dpp<0x4E>(x));
  x = xp_max(x, xp_dpp<0x141>(x));
  return xp_max(x, xp_dpp<0x140>(x));
}
__device__ __forceinline__ int xp_wave_min(int x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = min(x, __shfl_xor(x, o));
  return x;
}

// The candidates of a column, at most 16 of six words: lane 16 i + c holds
// word i (key, position, entries 0 and 1) of candidate c in w0 and, i < 2,
// word 4 + i (entries 2 and 3) in w1.
struct XpWords {
  xp_word w0, w1;
};
// Best of n candidates: largest key, the smallest position among equal ones.
__device__ __forceinline__ int xp_pick(const XpWords& w, int n, int lane) {
  const double key = lane < n ? xp_val(w.w0) : -3.0;
  const double m = readlane_d(xp_row_max(key), 0);
  unsigned b = (unsigned)__ballot(key == m) & 0xFFFFu;
  if (b & (b - 1)) {  // equal keys
    const int p = __shfl(static_cast<int>(w.w0), (lane & 15) + 16);
    const int c = xp_wave_min(lane < n && key == m ? p : INT_MAX);
    b = (unsigned)__ballot(lane < n && key == m && p == c) & 0xFFFFu;
  }
  return __builtin_amdgcn_readfirstlane(__builtin_ctz(b | 0x10000u) & 15);
}

// Whether all G workgroups are resident; when they are not within `patience`
// polls (negative: in any case) every one of them gets the same no.  (Atomics
// that end at the XCD's L2, as the exchange's stores do.)
__device__ bool xp_gather(XpBox* m, int G, long patience) {
  if (patience < 0)
    __hip_atomic_fetch_or(&m->here, kXpAlone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  for (long spins = 0;;) {
    int v = ld_agent(&m->here);
    if (v & kXpAlone) return false;
    if (v == G) return true;
    // (fails when one arrived meanwhile: at most G times)
    if (++spins > patience &&
        __hip_atomic_compare_exchange_strong(&m->here, &v, v | kXpAlone, __ATOMIC_RELAXED,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))
      return false;
  }
}

// The panel by one workgroup, column by column in memory.  slot: 32 words;
// urow: w entries; pa, pb, zcol as panel_xcd fills them.  (Not inlined: it
// would spill the panel's scalar registers.)
template <class S>
__device__ __attribute__((noinline)) void xp_alone(int M, int w, int off, S* P, long lda,
                                                   xp_word* slot, S* urow, int* pa, int* pb,
                                                   int* zcol) {
  const int t = threadIdx.x, nt = blockDim.x, mn = min(M, w);
#pragma unroll 1
  for (int j = 0; j < mn; j++) {
    S* cj = P + (size_t)j * lda;
    S key = S(-2);
    int p = INT_MAX;
    for (int i = j + t; i < M; i += nt) {  // (ascending: the first of equal keys stays)
      const S a = xp_key(__builtin_canonicalize(cj[i]));
      if (a > key) {
        key = a;
        p = i;
      }
    }
    S m = key;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = xp_max(m, __shfl_xor(m, o));
    p = xp_wave_min(key == m ? p : INT_MAX);
    if ((t & 63) == 0) {
      slot[t >> 6] = xp_bits((double)m);
      slot[16 + (t >> 6)] = (xp_word)(unsigned)p;
    }
    __syncthreads();
    double best = -3.0;
    p = j;
    for (int q = 0; q < nt / 64; q++) {
      const double k = xp_val(slot[q]);
      const int c = static_cast<int>(slot[16 + q]);
      if (k > best || (k == best && c < p)) {
        best = k;
        p = c;
      }
    }
    if (t < w) {  // rows j and p change places
      S* c = P + (size_t)t * lda;
      const S x = c[j], u = c[p];
      c[j] = u;
      c[p] = x;
      urow[t] = u;
    }
    __syncthreads();
    const S piv = urow[j];
    if (piv != S(0)) {
      const bool small = !(fabs(piv) >= std::numeric_limits<S>::min());
      const S up = !small ? S(1) : std::is_same<S, double>::value ? S(0x1p600) : S(0x1p100f);
      const S ps = piv * up, rinv = S(1) / ps;
      for (int i = j + 1 + t; i < M; i += nt) {
        const S x = cj[i] * up;
        S l = x * rinv;
        if (small) l += (x - l * ps) * rinv;
        cj[i] = l;
#pragma unroll 4
        for (int c = j + 1; c < w; c++) P[i + (size_t)c * lda] -= l * urow[c];
      }
    }
    if (t == 0) {
      pa[j] = off + j;
      pb[j] = off + p;
      if (piv == S(0) && *zcol < 0) *zcol = j;
    }
    __syncthreads();
  }
}

// Factors the M x w (w <= 32) panel P, row 0 of which is absolute row `off`
// on the matrix's diagonal; 32 columns of P span less than 2 GiB.  Outputs
// as panel_coop's.  G workgroups of blockDim.x / 64 waves on XCD `xcd`; grid
// 8 (G - 1) + xcd + 1 (see above).
// ONE: G is 1, and what several workgroups need is not compiled in (M = 256
// 59 us, 65 in the general form; N = 1500 4.24 ms, 4.31).
template <class S, bool ONE>
__global__ void __launch_bounds__(64 * kXpWaves)
panel_xcd(int M, int w, int off, S* __restrict__ P, long lda, int* __restrict__ ipiv,
          int* __restrict__ dinfo, XpBox* __restrict__ box, int par, int groups, int xcd,
          int* __restrict__ list, int* __restrict__ status, long limit, long gather) {
  typedef TriMfma<S> Mf;
  typedef typename Mf::acc_t acc_t;
  const int G = ONE ? 1 : groups;
  if (!ONE && (blockIdx.x & 7) != xcd) return;
  __shared__ xp_word slot[2][kXpCand][16];  // the waves' candidates, word-major
  __shared__ S ubuf[4][kXpW];  // G == 1: trailing entries of the block's pivot rows
  __shared__ S l11[kXpWaves][4][4];  // each wave's copy of the block's pivot rows
  __shared__ int pa[kXpW], pb[kXpW];
  __shared__ int sbad, zcol, together;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int NW = blockDim.x >> 6, g = ONE ? 0 : blockIdx.x >> 3;
  const int n = lane & 15, k = lane >> 4;
  XpBox* mb = box + par;
  if (G > 1 && t == 0)
    __hip_atomic_fetch_add(&mb->here, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  if (G > 1) xp_clear(box + (par ^ 1), g * blockDim.x + t, G * blockDim.x);
  for (int e = t; e < 2 * kXpCand * 16; e += blockDim.x) (&slot[0][0][0])[e] = xp_bits(-3.0);
  if (t == 0) {
    sbad = 0;
    zcol = -1;
  }
  // rows row0 + 16 rt + n, columns 4 b + k in v[rt][b >> 2][b & 3]
  const int row0 = (g * NW + wv) * 16 * RT + n;
  acc_t v[RT][2];
  int pos[RT];
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(P, 0, 0x7fffffff, kBufDword3);
  const int cstride = static_cast<int>(lda * (long)sizeof(S));
  // all in flight; rows past the panel are clamped and then zeroed
#pragma unroll
  for (int rt = 0; rt < RT; rt++) pos[rt] = min(row0 + 16 * rt, M - 1) * (int)sizeof(S);
  if (w == kXpW) {
#pragma unroll
    for (int b = 0; b < 8; b++)
#pragma unroll
      for (int rt = 0; rt < RT; rt++)
        v[rt][b >> 2][b & 3] = buf_ld(S(0), rs, static_cast<unsigned>(pos[rt] + k * cstride),
                                      4 * b * cstride);
  } else {
#pragma unroll
    for (int b = 0; b < 8; b++)
#pragma unroll
      for (int rt = 0; rt < RT; rt++) {
        v[rt][b >> 2][b & 3] = S(0);
        if (4 * b + k < w)
          v[rt][b >> 2][b & 3] = buf_ld(S(0), rs, static_cast<unsigned>(pos[rt] + k * cstride),
                                        4 * b * cstride);
      }
  }
  // (and any signalling NaN made quiet: the pivot keys' maximum expects
  // that, and no published value can then equal the sentinel, one of those)
#pragma unroll
  for (int rt = 0; rt < RT; rt++) {
    const bool in = row0 + 16 * rt < M;
#pragma unroll
    for (int b = 0; b < 8; b++)
      v[rt][b >> 2][b & 3] = in ? __builtin_canonicalize(v[rt][b >> 2][b & 3]) : S(0);
  }
#pragma unroll
  for (int rt = 0; rt < RT; rt++) pos[rt] = row0 + 16 * rt;
  const int mn = min(M, w);
  bool bad = false;  // this wave gave up waiting (no further waits or updates)
  // every row is in registers before any workgroup can finish and store
  __builtin_amdgcn_s_waitcnt(0);
  if (G > 1 && t == 0) together = xp_gather(mb, G, gather);
  __syncthreads();
  const bool alone = G > 1 && !together;
  if (alone) {
    if (g > 0) return;
    xp_alone(M, w, off, P, lda, &slot[0][0][0], &ubuf[0][0], pa, pb, &zcol);
  }
  const int held = alone ? 0 : mn;  // columns factored in registers
#pragma unroll 1
  for (int b = 0; 4 * b < held; b++) {
    const int jb = 4 * b, nq = min(4, mn - jb);
    // the block's entries of this lane's rows, and back below: selects by the
    // uniform b (a switch makes the compiler copy whole accumulator tuples)
    S x[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      x[rt] = v[rt][0][0];
#pragma unroll
      for (int b2 = 1; b2 < 8; b2++) x[rt] = b == b2 ? v[rt][b2 >> 2][b2 & 3] : x[rt];
    }
    int zmask = 0;  // columns with a zero pivot: neither scaled nor eliminated
#pragma unroll 1
    for (int q = 0; q < nq; q++) {
      const int j = jb + q, sp = j & 1;
      // column j of this lane's rows in every quarter (used once the pivot
      // is known: the exchange hides the moves)
      S xq[RT];
#pragma unroll
      for (int rt = 0; rt < RT; rt++) xq[rt] = xp_from(4 * (16 * q + n), x[rt]);
      // the wave's candidate: largest |x| of the rows at positions j..M-1
      S key[RT], m = S(-2);
      const unsigned left = k == q ? M - j : 0;
#pragma unroll
      for (int rt = 0; rt < RT; rt++) {
        const S a = xp_key(x[rt]);
        key[rt] = (unsigned)(pos[rt] - j) < left ? a : S(-2);
        m = xp_max(m, key[rt]);
      }
      m = xp_lane(xp_row_max(m), 16 * q);
      unsigned long long bl[RT];
      int cnt = 0;
#pragma unroll
      for (int rt = 0; rt < RT; rt++) {
        bl[rt] = __ballot(key[rt] == m);
        cnt += __popcll(bl[rt]);
      }
      if (cnt > 1) {  // equal keys (or no rows): the smallest position
        int c = INT_MAX;
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
          if (key[rt] == m) c = min(c, pos[rt]);
        c = xp_wave_min(c);
#pragma unroll
        for (int rt = 0; rt < RT; rt++) bl[rt] = __ballot(key[rt] == m && pos[rt] == c);
      }
      {
        unsigned long long bb = bl[RT - 1];
        S xs = x[RT - 1];
        int px = pos[RT - 1];
#pragma unroll
        for (int rt = RT - 2; rt >= 0; rt--) {
          const bool h = bl[rt] != 0;
          bb = h ? bl[rt] : bb;
          xs = h ? x[rt] : xs;
          px = h ? pos[rt] : px;
        }
        const int src = __builtin_ctzll(bb | (1ull << 63));
        xp_word* sl = &slot[sp][0][wv];
        if (n == (src & 15)) sl[(2 + k) * 16] = xp_bits((double)xs);
        if (lane == src) {
          sl[0] = xp_bits((double)m);
          sl[16] = (xp_word)(unsigned)px;
        }
      }
      __syncthreads();
      XpWords ww = {0, 0};
      int pc = 0;  // the pivot row's candidate
      if (G == 1 || wv == 0) {
        const xp_word* sw = &slot[sp][0][0];
        ww.w0 = sw[lane];
        ww.w1 = sw[64 + (lane & 31)];
        if (G > 1) {
          pc = xp_pick(ww, NW, lane);
          if (n == pc) {
            xp_st(&mb->cand[j][k][g], ww.w0);
            if (k < 2) xp_st(&mb->cand[j][4 + k][g], ww.w1);
          }
        }
      }
      if (G > 1) {
        const xp_word* src = &mb->cand[j][k][n];
        const bool w0 = n < G, w1 = w0 && k < 2;
        ww.w0 = ww.w1 = 0;
        long spins = 0;
        while (!bad) {
          if (w0) ww.w0 = xp_ld(src);
          if (w1) ww.w1 = xp_ld(src + 4 * kXpMaxG);
          if (!__any(ww.w0 == kXpSent || ww.w1 == kXpSent)) break;
          if (++spins >= limit || ((spins & 255) == 0 && ld_agent(&mb->err))) {
            st_agent(&mb->err, 1);
            sbad = 1;
            bad = true;
          }
        }
      }
      // every candidate's reciprocal of this column beside the search for the
      // best one (the entry of column q: w0 of quarters 2, 3 or w1 of 0, 1)
      S rw = (S)xp_val(q < 2 ? ww.w0 : ww.w1);
      rw = S(1) / rw;
      pc = xp_pick(ww, G == 1 ? NW : G, lane);
      // rows j..M-1 always hold a candidate, so the position is in [j, M);
      // the clamp only keeps a failed exchange in range
      int p = __builtin_amdgcn_readlane(static_cast<int>(ww.w0), pc + 16);
      p = (p >= j && p < M) ? p : j;
      S e[4];  // the pivot row's block entries
      e[0] = (S)readlane_d(xp_val(ww.w0), pc + 32);
      e[1] = (S)readlane_d(xp_val(ww.w0), pc + 48);
      e[2] = (S)readlane_d(xp_val(ww.w1), pc);
      e[3] = (S)readlane_d(xp_val(ww.w1), pc + 16);
      S rinv = xp_lane(rw, pc + 16 * ((q + 2) & 3));
      S piv = e[0], u = e[0];  // column j's entry, and this quarter's
#pragma unroll
      for (int a = 1; a < 4; a++) {
        piv = q == a ? e[a] : piv;
        u = k == a ? e[a] : u;
      }
      if (bad) piv = S(0);
      if (piv != S(0)) {
        // the reciprocal of a subnormal pivot can overflow: pivot and entries
        // (no larger) are then scaled up, and the quotient corrected once
        S l[RT];
#pragma unroll
        for (int rt = 0; rt < RT; rt++) l[rt] = xq[rt] * rinv;
        if (!(fabs(piv) >= std::numeric_limits<S>::min())) {
          const S up = std::is_same<S, double>::value ? S(0x1p600) : S(0x1p100f);
          const S ps = piv * up;
          rinv = S(1) / ps;
#pragma unroll
          for (int rt = 0; rt < RT; rt++) {
            const S xs = xq[rt] * up;
            l[rt] = xs * rinv;
            l[rt] += (xs - l[rt] * ps) * rinv;
          }
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
          // rows below the pivot (position p keeps its row only when p is j;
          // the row at j moves to p): the multiplier in quarter q, the
          // update right of it, nothing left of it
          const S y = k == q ? l[rt] : x[rt] - l[rt] * u;
          const bool low = pos[rt] >= j && pos[rt] != p;
          x[rt] = (k >= q && low) ? y : x[rt];
        }
      } else {
        zmask |= 1 << q;
      }
      // the pivot row's entries right of the block, for the block's end
      if (n == 0) l11[wv][q][k] = u;
      if (jb + 4 < w) {
        bool mine = false;
#pragma unroll
        for (int rt = 0; rt < RT; rt++) mine = mine || pos[rt] == p;
        if (__any(mine)) {
#pragma unroll
          for (int rt = 0; rt < RT; rt++)
            if (pos[rt] == p) {
#pragma unroll
              for (int b2 = 1; b2 < 8; b2++) {
                if (G == 1) ubuf[q][4 * b2 + k] = v[rt][b2 >> 2][b2 & 3];
                else if (b2 > b)
                  xp_st(&mb->trail[j][4 * b2 + k], xp_bits((double)v[rt][b2 >> 2][b2 & 3]));
              }
            }
        }
      }
#pragma unroll
      for (int rt = 0; rt < RT; rt++) pos[rt] = pos[rt] == j ? p : (pos[rt] == p ? j : pos[rt]);
      if (g == 0 && t == 0) {
        pa[j] = off + j;
        pb[j] = off + p;
        if (piv == S(0) && zcol < 0) zcol = j;
      }
    }
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
      for (int b2 = 0; b2 < 8; b2++)
        v[rt][b2 >> 2][b2 & 3] = b == b2 ? x[rt] : v[rt][b2 >> 2][b2 & 3];
    if (jb + 4 >= w) break;
    // the columns right of the block: U12 = inv(L11) A12 from the published
    // rows, then one MFMA per tile
    if (G == 1) __syncthreads();
    const int mr = std::is_same<S, double>::value ? n >> 2 : n & 3;
    const int mk = std::is_same<S, double>::value ? n & 3 : n >> 2;
    S a[2][4], x1[2];  // tile ct's column of this lane, all four pivot rows
    if (G == 1) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        a[0][i] = ubuf[i][4 * mr + mk];
        a[1][i] = ubuf[i][16 + 4 * mr + mk];
      }
    } else {
      const xp_word* src = &mb->trail[jb][4 * mr + mk];
      xp_word wt[2][4];
      long spins = 0;
      bool miss = !bad;
#pragma unroll
      for (int i = 0; i < 4; i++) wt[0][i] = wt[1][i] = 0ull;
      while (miss) {
        miss = false;
#pragma unroll
        for (int ct = 0; ct < 2; ct++)
          if (4 * ct + 3 > b) {
#pragma unroll
            for (int i = 0; i < 4; i++) wt[ct][i] = xp_ld(src + i * kXpW + 16 * ct);
          }
#pragma unroll
        for (int ct = 0; ct < 2; ct++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            miss = miss || (4 * ct + mr > b && i < nq && wt[ct][i] == kXpSent);
        miss = __any(miss);
        if (miss && (++spins >= limit || ((spins & 255) == 0 && ld_agent(&mb->err)))) {
          st_agent(&mb->err, 1);
          sbad = 1;
          bad = true;
          miss = false;
        }
      }
#pragma unroll
      for (int ct = 0; ct < 2; ct++)
#pragma unroll
        for (int i = 0; i < 4; i++) a[ct][i] = (S)xp_val(wt[ct][i]);
    }
#pragma unroll
    for (int i = 1; i < 4; i++)
#pragma unroll
      for (int c2 = 0; c2 < i; c2++) {
        const S l = l11[wv][i][c2];
        const bool el = !(zmask >> c2 & 1);
#pragma unroll
        for (int ct = 0; ct < 2; ct++) a[ct][i] = el ? a[ct][i] - l * a[ct][c2] : a[ct][i];
      }
#pragma unroll
    for (int ct = 0; ct < 2; ct++) {
      S u = a[ct][0];
#pragma unroll
      for (int i = 1; i < 4; i++) u = k == i ? a[ct][i] : u;
      x1[ct] = (4 * ct + mr > b && k < nq && !bad) ? -u : S(0);
    }
    // multipliers of this lane's column for its rows; none for a row chosen
    // at or before that column
    bool fin = isfinite(x1[0]) && isfinite(x1[1]);
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      const bool use = pos[rt] > jb + k && k < nq && !(zmask >> k & 1);
      x[rt] = use ? x[rt] : S(0);
      fin = fin && isfinite(x[rt]);
    }
    if (__all(fin)) {
      if (b < 3) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++) v[rt][0] = Mf::op(x1[0], x[rt], v[rt][0]);
      }
#pragma unroll
      for (int rt = 0; rt < RT; rt++) v[rt][1] = Mf::op(x1[1], x[rt], v[rt][1]);
    } else {
      // infinities or NaN: a product with a masked zero must not reach
      // finished entries, so the columns go one by one and only the active
      // entries take the products
#pragma unroll 1
      for (int kk = 0; kk < nq; kk++) {
        if (zmask >> kk & 1) continue;
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
          const bool act = pos[rt] > jb + kk;
#pragma unroll
          for (int ct = 0; ct < 2; ct++) {
            const acc_t d = Mf::op(k == kk ? x1[ct] : S(0), k == kk ? x[rt] : S(0),
                                   acc_t{0, 0, 0, 0});
#pragma unroll
            for (int r = 0; r < 4; r++)
              if (4 * ct + r > b && act) v[rt][ct][r] += d[r];
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
    if (!alone && row0 + 16 * rt < M) {
      const unsigned vo = static_cast<unsigned>(pos[rt] * (int)sizeof(S) + k * cstride);
      if (w == kXpW) {
#pragma unroll
        for (int b = 0; b < 8; b++) buf_st(v[rt][b >> 2][b & 3], rs, vo, 4 * b * cstride);
      } else {
#pragma unroll
        for (int b = 0; b < 8; b++)
          if (4 * b + k < w) buf_st(v[rt][b >> 2][b & 3], rs, vo, 4 * b * cstride);
      }
    }
  __syncthreads();
  if (sbad) {
    if (t == 0) {
      *dinfo = INT_MIN;
      atomicOr(status, ATLG_FAIL_PANEL);
    }
    if (g == 0) {
      if (t < mn) ipiv[off + t] = off + t;  // identity: later users stay in bounds
      if (t == 0) list[0] = 0;              // apply no interchanges
    }
    return;
  }
  if (g == 0) {
    if (t < mn) ipiv[off + t] = pb[t];
    if (t == 0 && zcol >= 0 && *dinfo == 0) *dinfo = off + zcol + 1;
    if (t < 64) compose_swaps_wave(pa, pb, mn, list);
  }
}
