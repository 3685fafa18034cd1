/*
 * The screened kernels: one workgroup per permutation, cells dropped by
 * comparing their overlap with a critical count.
 *
 * For one job every cell (i, j) has fixed K_i, n_j and N, so whether its tail
 * P(X >= k) can lie at or below a level e^L depends on k alone.  The job's cut
 * tables (k_cut_table, built once by its first screened launch) hold, for each
 * of a few levels, the largest k whose tail is certain to lie above the level;
 * level 0 drops only cells whose tail is exactly 1.  A permutation is swept
 * against the start level's table: per pair of columns the screen is one
 * packed 16-bit saturating subtraction, where evaluating a first-term bound
 * takes four table lookups and some 30 instructions a cell (that sweep and
 * its second pass over rows within reach of the minimum took 84 % of the
 * genome-scale job).  Cells above their cut go to a per-wave list and through
 * the first-term, bracket and exact FP64 tiers; the bounds these find move the
 * sweep on to tighter tables.  When the best exact p is at or below the start
 * level, no dropped cell can reach or tie it and the result is final;
 * otherwise (2-10 % of null permutations) the sweep is repeated with the
 * next, looser table.
 */
#pragma once
#include "dto_kernels.h"

#pragma clang fp contract(off)

namespace dto {

/* A cell's sweep segment: kCutWords count words (2 columns each) per lane,
 * 768 columns a wave.  Every grid of reference thresholds has fewer (719 at
 * the longest accepted list), so its rows are one segment. */
constexpr uint32_t kCutWords = 6;
constexpr uint32_t kCutSpan = 64u * kCutWords;

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

/* max(0, a - b) in both 16-bit halves. */
__device__ __forceinline__ uint32_t sub_sat_u16x2(uint32_t a, uint32_t b) {
  const u16x2 d = __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b));
  return __builtin_bit_cast(uint32_t, d);
}

/* The counts of a word's first column, and of both: w + (w << 16).  As C this
 * becomes a 64-bit multiply-add by 0x10001, four times the cost. */
__device__ __forceinline__ uint32_t word_prefix(uint32_t w) {
  uint32_t v;
  asm("v_lshl_add_u32 %0, %1, 16, %1" : "=v"(v) : "v"(w));
  return v;
}

/* The shared bound, read from LDS (through a generic pointer the read would
 * be a flat load, whose wait covers every outstanding global load). */
__device__ __forceinline__ float shared_bound(const Lds &S) {
  return fkey_value(*(const volatile __attribute__((address_space(3))) int *)lds_addr(S.ushare));
}

/* log P(X = k) in FP64 (no particular operation order). */
__device__ __forceinline__ double log_term(const DevJob &J, uint32_t K, uint32_t n, uint32_t k) {
  const double *LF = J.LF;
  const uint32_t N = J.N;
  return ((LF[K] - LF[k]) - LF[K - k]) + ((LF[N - K] - LF[n - k]) - LF[(N - K) - (n - k)]) -
         ((LF[N] - LF[n]) - LF[N - n]);
}

/* The cut tables: out[(((level * T1 + i) * segs + s) * kCutWords + u) * 64 +
 * lane] packs the cuts of columns 2 w and 2 w + 1, w = kCutSpan s + kCutWords
 * lane + u.  A cell is dropped when k <= its cut.  One thread per cell.  For
 * the low levels the cut is the largest k found with P(X = k) alone above the
 * level.  From there it adds terms downwards in FP32: at every k the sum is a
 * lower bound of P(X >= k) up to its rounding: each term's ratio has a
 * relative error of up to 6 * 2^-24 (four roundings and a reciprocal of 1
 * ulp), and fewer than 1,000 steps lead from the low levels to 1.2 standard
 * deviations (at most 99) below the mean, where the sum exceeds the highest
 * level: under 0.04 %.  Above populations of 2^24, where subtracting 1 from a
 * count is rounded too, the deviation is at most 16, and fewer than 200 steps
 * add under 0.12 %.  So P(X >= k) > e^l is certain once the sum exceeds 1.01
 * e^l, and for every smaller k too.  A tail that never gets there keeps the cut max(0, K + n - N), the
 * largest k with P(X >= k) = 1, which is also level 0's.  Columns past T2 get
 * 0xFFFF: never listed.  89 us at 599 x 599 cells and 14 levels; adding every
 * term from the lowest level up took 245 us. */
static __global__ __launch_bounds__(256) void k_cut_table(DevJob J, uint16_t *__restrict__ out) {
  const uint32_t cols = 2u * kCutSpan * J.cut_segs;
  const uint64_t per_level = (uint64_t)J.T1 * cols;
  for (uint64_t c = (uint64_t)blockIdx.x * 256 + threadIdx.x; c < per_level; c += (uint64_t)gridDim.x * 256) {
    const uint32_t i = (uint32_t)(c / cols), j = (uint32_t)(c % cols);
    const uint32_t s = j / (2u * kCutSpan), wi = (j % (2u * kCutSpan)) / 2u;
    uint16_t *o =
        out + ((((uint64_t)i * J.cut_segs + s) * kCutWords + wi % kCutWords) * 64u + wi / kCutWords) * 2u + (j & 1u);
    if (j >= J.T2) {
      for (uint32_t l = 0; l < kCutLevels; ++l) o[l * per_level] = 0xFFFFu;
      continue;
    }
    const uint32_t N = J.N, K = J.K[i], n = J.n[j];
    const uint32_t lo = K + n > N ? K + n - N : 0u, hi = K < n ? K : n;
    uint32_t mode = (uint32_t)(((double)K + 1.0) * ((double)n + 1.0) / ((double)N + 2.0));
    mode = mode < lo ? lo : (mode > hi ? hi : mode);
    /* the low levels, by the first term alone: Newton steps down from the
     * largest k (log P(X = k) is concave, so a step rounded down stays on the
     * far side of the level until the last ones) */
    uint32_t k = hi, l = kCutLevels - 1u;
    double x = log_term(J, K, n, k);
    for (; l >= kCutDeep; --l) {
      const double level = (double)J.cut_level[l] + 0.01;
      while (x < level && k > mode) {
        const float s = __logf((float)k * (float)((N - K) - (n - k)) / ((float)(K - k + 1u) * (float)(n - k + 1u)));
        const float d = s > 1e-3f ? fminf((float)(level - x) / s, 1e9f) : 1.f;
        const uint32_t step = d > 1.f ? (uint32_t)d : 1u;
        k -= step < k - mode ? step : k - mode;
        x = log_term(J, K, n, k);
      }
      if (x < level) break;
      o[l * per_level] = (uint16_t)k;
    }
    if (l < kCutDeep) {
      /* the others, by the sum from here down, in units of the first term */
      const float off = (float)x;
      float t = 1.f, S = 1.f, th = 1.01f * __expf(J.cut_level[l] - off);
      /* t_{k-1} / t_k = k (N - K - n + k) / ((K - k + 1) (n - k + 1)) */
      float f0 = (float)k, f1 = (float)((N - K) - (n - k)), f2 = (float)(K - k + 1u), f3 = (float)(n - k + 1u);
      for (; k > lo; --k) {
        while (S > th) {
          o[l * per_level] = (uint16_t)k;
          --l;
          th = l ? 1.01f * __expf(J.cut_level[l] - off) : __builtin_inff();
        }
        if (l == 0u) break;
        t *= (f0 * f1) * __builtin_amdgcn_rcpf(f2 * f3);
        S += t;
        f0 -= 1.f;
        f1 -= 1.f;
        f2 += 1.f;
        f3 += 1.f;
      }
    }
    for (uint32_t v = 0; v <= l; ++v) o[v * per_level] = (uint16_t)lo;
  }
}

/* How a job's pairs are built: kBuildRegs keeps each list-2 position's pair
 * in its thread's registers and the join in LDS; the others stage pairs in
 * LDS or in a global slice (build_rows). */
enum { kBuildGlobal = 0, kBuildLds = 1, kBuildRegs = 2 };
/* Elements a thread holds at most in kBuildRegs. */
constexpr uint32_t kRegPairs = 32;

/* Per-job tables that stay in LDS while a workgroup works on that job. */
template <int NT, int BUILD>
__device__ __forceinline__ void load_cut_tables(const DevJob &J, const LdsLayout &Lo, const Lds &S,
                                                unsigned char *smem) {
  for (uint32_t t = threadIdx.x; t < 256; t += NT) S.tab[t] = kExpTabC[t];
  for (uint32_t t = threadIdx.x; t < J.T2; t += NT) S.coln[t] = J.n[t];
  if (BUILD == kBuildRegs) {
    uint16_t *jn = (uint16_t *)(smem + Lo.join);
    for (uint32_t t = threadIdx.x; t < J.N2; t += NT) jn[t] = (uint16_t)J.join[t]; /* none: 0xFFFF */
  }
}

/* build_rows for lists whose pairs fit the workgroup's registers (both
 * shuffle domains at most kRegPairs * NT elements, no repeated ids).  What
 * bounds the build is the gather of the join at random positions: from L2
 * it is one cache line a lane; the LDS answers 64 lanes in a few cycles.
 * The pairs' staging in registers is what leaves the LDS room for it.  Loads
 * take clamped indices instead of conditions: under a condition each load
 * is a basic block of its own and its wait comes before the next one. */
template <int NT, bool EXPLICIT>
__device__ __forceinline__ void build_regs(const DevJob &J, const LdsLayout &Lo, const Lds &S, const uint16_t *jn,
                                           const uint32_t *i1, const uint32_t *i2, const Shuffle &s1,
                                           const Shuffle &s2, int *err) {
  constexpr uint32_t W = NT / 64, U = kShufU, CH = kRegPairs / U;
  uint32_t tid = threadIdx.x;
  /* opaque: else the positions and addresses of every element, the same in
   * every task, are computed before the task loop and kept in scratch */
  asm volatile("" : "+v"(tid));
  const uint32_t T1 = J.T1, T2 = J.T2, N1 = J.N1, N2 = J.N2, T2wp = Lo.T2w_pad;
  const uint16_t *bin1 = J.bin1, *bin2 = J.bin2;
  for (uint32_t t = tid; t <= T1; t += NT) S.rowstart[t] = 0;
  for (uint32_t t = tid; t < W * T2wp; t += NT) S.cw[t] = 0;
  if (tid == 0) *S.ushare = fkey(__builtin_inff());
  /* list-1 bins by position */
  uint32_t carried = 0;
#pragma unroll 1
  for (uint32_t base = 0; base < (EXPLICIT ? N1 : s1.dom); base += NT * U) {
    uint32_t k[U], m[U], bn[U];
    if (EXPLICIT) {
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) k[u] = base + u * NT + tid;
      if (i1) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) m[u] = at32(i1, min(k[u], N1 - 1u));
      } else {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) m[u] = k[u];
      }
    } else {
      shuffle_chunk<NT>(s1, S.redS, base, carried, k, m);
    }
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) bn[u] = at32(bin1, min(k[u], N1 - 1u));
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const bool in = EXPLICIT ? k[u] < N1 : true;
      if (EXPLICIT && in && m[u] >= N1) atomicOr(err, 1);
      if (in && m[u] < N1) S.nb[m[u]] = (uint16_t)bn[u];
    }
  }
  __syncthreads();
  /* pairs (a << 16 | b) per list-2 position, counted per row */
  uint32_t pr[kRegPairs];
  carried = 0;
#pragma unroll
  for (uint32_t c = 0; c < CH; ++c) {
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) pr[c * U + u] = kNone;
    if (c * NT * U < (EXPLICIT ? N2 : s2.dom)) {
      uint32_t e[U], q[U], b[U], a[U];
      if (EXPLICIT) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) e[u] = (c * U + u) * NT + tid;
        if (i2) {
#pragma unroll
          for (uint32_t u = 0; u < U; ++u) q[u] = at32(i2, min(e[u], N2 - 1u));
        } else {
#pragma unroll
          for (uint32_t u = 0; u < U; ++u) q[u] = e[u];
        }
      } else {
        shuffle_chunk<NT>(s2, S.redS, c * NT * U, carried, e, q);
      }
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) b[u] = at32(bin2, min(e[u], N2 - 1u));
      if (EXPLICIT) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
          if (e[u] < N2 && q[u] >= N2) atomicOr(err, 1);
          q[u] = e[u] < N2 ? q[u] : N2;
        }
      }
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) a[u] = jn[min(q[u], N2 - 1u)];
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) a[u] = q[u] < N2 ? a[u] : 0xFFFFu;
      /* positions without a partner read entry 0, and are left out */
#pragma unroll
      for (uint32_t u = 0; u < U; ++u) {
        const uint32_t x = S.nb[a[u] != 0xFFFFu ? a[u] : 0u];
        a[u] = a[u] != 0xFFFFu ? x : kBinNone;
      }
#pragma unroll
      for (uint32_t u = 0; u < U; ++u)
        if (a[u] < T1 && b[u] < T2) {
          pr[c * U + u] = (a[u] << 16) | b[u];
          atomicAdd(&S.rowstart[a[u]], 1u);
        }
    }
  }
  __syncthreads();
  block_excl_scan<NT>(S.rowstart, T1, S.redS);
  for (uint32_t t = tid; t < T1; t += NT) S.cursor[t] = S.rowstart[t];
  __syncthreads();
  /* the columns in row order, over the list-1 bins (all read above) */
#pragma unroll
  for (uint32_t c = 0; c < CH; ++c) {
    uint32_t pos[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u)
      if (pr[c * U + u] != kNone) pos[u] = atomicAdd(&S.cursor[pr[c * U + u] >> 16], 1u);
#pragma unroll
    for (uint32_t u = 0; u < U; ++u)
      if (pr[c * U + u] != kNone) S.nb[pos[u]] = (uint16_t)pr[c * U + u];
  }
  __syncthreads();
}

/* The listed cells, in full-lane batches: each lane takes one cell, keeps it
 * as a p == 0 cell, or forms its first-term screen value x and bounds its log
 * p from both sides (x minus the margin plus a lower bound of the tail; x
 * plus the margin and the geometric bound of the tail, 1 / (1 - r), since the
 * term ratios r only fall).  The upper ends tighten Uw before the batch is
 * tested, so that a permutation whose small p-values fill many cells does not
 * send them all to tier 2. */
template <int NT>
__device__ __forceinline__ void flush_cut(const DevJob &J, const Lds &S, uint2 *cand0, uint32_t &n0, uint2 *cand,
                                          uint32_t &nc, uint4 *c3, uint32_t &n3, BestKey &xb, ZeroKey &zb, float &Uw,
                                          float &U2w, WaveStats &st) {
  const uint32_t lane = lane_id(), N = J.N;
  const float *H = J.H32;
  uint64_t tf = cycles();
  if (lane == 0) st.cheap += n0;
  wave_sync();
#pragma unroll 1
  for (uint32_t r0 = 0; r0 < n0; r0 += 64) {
    const float us = shared_bound(S);
    U2w = fminf(U2w, us);
    Uw = fminf(Uw, us);
    float L = __builtin_inff(), U = __builtin_inff();
    uint2 cd = make_uint2(0u, 0u);
    if (r0 + lane < n0) {
      cd = cand0[r0 + lane];
      const uint32_t i = cd.x >> 16, j = cd.x & 0xFFFFu, k = cd.y;
      const uint32_t K = J.K[i], n = S.coln[j], mx = min(K, n);
      float x = 0.f;
      if (k <= mx) x = (J.A32[i] + J.B32[j]) - ((H[k] + H[K - k]) + (H[n - k] + H[(N - K) - (n - k)]));
      if (k > mx || (x + J.margin < -745.2f && exact_zero(J, K, n, k, x))) {
        take_zero(zb, k, cd.x);
        U = -__builtin_inff();
      } else {
        L = x - J.margin;
        L = L >= -708.f ? L + tail_lower_log(N, K, n, k) : -__builtin_inff(); /* below: sums may be subnormal */
        const float r = k < mx ? term_ratio(N, K, n, k) * (1.f + 8.f * 0x1p-24f) : 0.f;
        U = 1e-6f; /* every p <= 1 (+ rounding) */
        if (r < 0.999f) {
          float hi = x + J.margin - __logf(1.f - r) + 3e-4f;
          if (hi < -690.f) hi = fmaxf(hi, __logf((float)(mx - k + 1u)) - 744.44f) + 0.7f;
          U = fminf(U, hi);
        }
      }
    }
    U = wave_minf(U);
    if (U < U2w) {
      U2w = U;
      share_bound(S, U2w);
    }
    Uw = fminf(Uw, U2w);
    const bool f = L < __builtin_inff() && L <= Uw;
    const uint64_t m = __ballot(f);
    const uint32_t cnt = (uint32_t)__popcll(m);
    if (cnt) {
      if (nc + cnt > (uint32_t)kCandCap) flush_candidates<NT>(J, S, cand, nc, c3, n3, xb, Uw, U2w, st);
      if (f) cand[nc + mask_lt(m)] = cd;
      nc += cnt;
      st.push1 += cnt;
    }
  }
  n0 = 0;
  wave_sync();
  st.cyc[3] += cycles() - tf;
}

/* First row of wave w's block: rows are split so that the sum of rows
 * (kRowPairs pairs' worth of work each) and pairs is about equal per wave.
 * The lanes probe 64 rows at a time. */
constexpr uint32_t kRowPairs = 512;
__device__ __forceinline__ uint32_t block_row(const uint32_t *rowstart, uint32_t T1, uint32_t w, uint32_t W) {
  if (w == 0u) return 0u;
  if (w >= W) return T1;
  const uint32_t lane = lane_id();
  const uint64_t want = ((uint64_t)T1 * kRowPairs + rowstart[T1]) * w / W;
  uint32_t lo = 0u, len = T1; /* the answer, the first row with a cost prefix >= want, is in [lo, lo + len] */
  while (len) {
    const uint32_t step = (len + 63u) / 64u;
    const uint32_t r = lo + lane * step; /* lane's probe */
    const bool below = lane * step < len && (uint64_t)r * kRowPairs + rowstart[min(r, T1)] < want;
    const uint32_t c = (uint32_t)__popcll(__ballot(below)); /* probes 0 .. c-1 lie below */
    if (c == 0u) break;
    const uint32_t nlo = lo + (c - 1u) * step + 1u, nhi = min(lo + c * step, lo + len);
    lo = nlo;
    len = nhi > nlo ? nhi - nlo : 0u;
  }
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)min(lo, T1));
}

/* One permutation: overlap grid -> best cell, in thread 0 (others:
 * undefined).  Each wave owns a block of consecutive rows: it counts its
 * rows' pairs by column, an exclusive prefix over the waves turns those into
 * the counts above each block, and the wave then adds its rows one by one and
 * scans each, so every pair is added twice, not once per wave.  Two waves a
 * SIMD or more: the sweep is bound by VALU issue and by the latency of each
 * row's chain (adds, reads, scan) together.  10,001 explicit tasks at N =
 * 20,000: 3.65 ms at 0.51 of the VALU issue rate, where the first-term screen
 * took 8.00 ms; 1,000 drawn ones at N = 40,961: 0.94 instead of 4.4 ms. */
template <int NT, bool EXPLICIT, int BUILD>
__device__ __forceinline__ BestKey optimize_cut(const DevJob &J, const LdsLayout &Lo, const Lds &S, const uint32_t *i1,
                                                const uint32_t *i2, const Shuffle &s1, const Shuffle &s2, int *err,
                                                WaveStats &st, unsigned char *smem, uint16_t *gpairs, uint32_t *counter,
                                                uint32_t *slot) {
  constexpr uint32_t W = NT / 64;
  const uint32_t tid = threadIdx.x, lane = lane_id(), w = wave_id();
  uint64_t tc0 = cycles();
  if (BUILD == kBuildRegs)
    build_regs<NT, EXPLICIT>(J, Lo, S, (const uint16_t *)(smem + Lo.join), i1, i2, s1, s2, err);
  else
    build_rows<NT, EXPLICIT, false, BUILD == kBuildLds, true>(J, Lo, S, i1, i2, s1, s2, err, gpairs);
  uint64_t tc1 = cycles();
  st.cyc[0] += tc1 - tc0;
  /* claim the next task once the build is done: every workgroup of the
   * launch that fits the chip has started by then */
  if (counter && tid == 0) *slot = atomicAdd(counter, 1u);

  const uint32_t T1 = J.T1, T2w_pad = Lo.T2w_pad, segs = J.cut_segs;
  const uint32_t zero_word = T2w_pad - kCutWords; /* the wave's last kCutWords words stay zero */
  uint32_t *C = S.cw + w * T2w_pad;
  const uint32_t rbeg = block_row(S.rowstart, T1, w, W), rend = block_row(S.rowstart, T1, w + 1u, W);
  const uint32_t pbeg = S.rowstart[rbeg], pend = S.rowstart[rend];

  ZeroKey zb = {0u, kNone, 0u, 0u}; /* p == 0 cells */
  BestKey xb = no_best();           /* exactly evaluated cells */
  static_assert(kCandCap >= 64 && kCand0Cap >= 128, "one ballot (64 cells) must fit beside a partly filled list");
  uint2 *cand0 = S.cand0 + w * kCand0Cap;
  uint2 *cand = S.cand + w * kCandCap;
  uint4 *c3 = S.cand3 + w * kCand3Cap;

#pragma unroll 1
  for (uint32_t lev = kCutStart;; --lev) {
    /* column counts of this wave's rows, then of all rows before them */
    if (w + 1u < W)
      for (uint32_t e = pbeg + lane; e < pend; e += 256u) {
        uint32_t b[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) b[u] = S.nb[min(e + 64u * u, pend - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
          if (e + 64u * u < pend) atomicAdd(&C[b[u] >> 1], 1u << ((b[u] & 1u) * 16u));
      }
    __syncthreads();
    for (uint32_t t = tid; t < zero_word; t += NT) {
      uint32_t x[W], run = 0u;
#pragma unroll
      for (uint32_t v = 0; v < W; ++v) x[v] = S.cw[v * T2w_pad + t];
#pragma unroll
      for (uint32_t v = 0; v < W; ++v) {
        S.cw[v * T2w_pad + t] = run;
        run += x[v];
      }
    }
    __syncthreads();

    uint64_t tc2 = cycles();
    st.cyc[1] += tc2 - tc1;
    st.rows++;
    float U2w = 1e-6f; /* upper bound of the minimum log p */
    float Uw = fminf(J.cut_level[lev] + 1e-3f, U2w); /* cells above it cannot decide this pass */
    /* the table in use: once a bound of the minimum lies below a lower level,
     * that level's table (a cell it drops has p > e^level >= the minimum) */
    uint32_t use = lev;
    float next_level = use + 1u < kCutLevels ? J.cut_level[use + 1u] : -__builtin_inff();
    const uint64_t per_level = (uint64_t)T1 * segs * (kCutWords * 64u);
    uint32_t n0 = 0, nc = 0, n3 = 0;
    const uint32_t *cut = J.cut + lev * per_level + (uint64_t)rbeg * segs * (kCutWords * 64u);
    uint32_t pe0 = pbeg, pe1 = rbeg < rend ? S.rowstart[rbeg + 1u] : pbeg;
    uint32_t pb[2];
#pragma unroll
    for (uint32_t u = 0; u < 2; ++u) pb[u] = S.nb[pe1 > pe0 ? min(pe0 + lane + 64u * u, pe1 - 1u) : 0u];
    /* a segment's cuts are loaded while the one before it is scanned; one
     * row past the last is read (the tables end with a padding row) */
    uint32_t kd[kCutWords];
#pragma unroll
    for (uint32_t u = 0; u < kCutWords; ++u) kd[u] = cut[64u * u + lane];
#pragma unroll 1
    for (uint32_t i = rbeg; i < rend; ++i) {
      const uint32_t ne1 = i + 2u <= rend ? S.rowstart[i + 2u] : pe1;
      /* this row's pairs: the first 128 from registers */
#pragma unroll
      for (uint32_t u = 0; u < 2; ++u)
        if (pe0 + lane + 64u * u < pe1) atomicAdd(&C[pb[u] >> 1], 1u << ((pb[u] & 1u) * 16u));
      for (uint32_t e = pe0 + 128u + lane; e < pe1; e += 64u) {
        const uint32_t b = S.nb[e];
        atomicAdd(&C[b >> 1], 1u << ((b & 1u) * 16u));
      }
      pe0 = pe1;
      pe1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)ne1);
#pragma unroll
      for (uint32_t u = 0; u < 2; ++u) pb[u] = S.nb[pe1 > pe0 ? min(pe0 + lane + 64u * u, pe1 - 1u) : 0u];
      const float us = shared_bound(S);
      uint32_t carry = 0u;
#pragma unroll 1
      for (uint32_t s = 0; s < segs; ++s) {
        uint32_t wv[kCutWords], tot = 0u;
        const uint32_t w0 = min(s * kCutSpan + lane * kCutWords, zero_word);
#pragma unroll
        for (uint32_t u = 0; u < kCutWords; u += 2) {
          const uint2 v = *(const uint2 *)(C + w0 + u);
          wv[u] = v.x;
          wv[u + 1] = v.y;
        }
        uint32_t kn[kCutWords];
        while (__builtin_amdgcn_readfirstlane((int)(us < next_level))) {
          ++use;
          cut += per_level;
          next_level = use + 1u < kCutLevels ? J.cut_level[use + 1u] : -__builtin_inff();
        }
        cut += kCutWords * 64u;
#pragma unroll
        for (uint32_t u = 0; u < kCutWords; ++u) kn[u] = cut[64u * u + lane];
#pragma unroll
        for (uint32_t u = 0; u < kCutWords; ++u) tot += wv[u];
        tot = (tot & 0xFFFFu) + (tot >> 16);
        const uint32_t incl = wave_incl_scan(tot);
        uint32_t run2 = carry + incl - tot;
        run2 |= run2 << 16;
        carry += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        uint32_t kv[kCutWords], d[kCutWords], any = 0u;
#pragma unroll
        for (uint32_t u = 0; u < kCutWords; ++u) {
          /* prefixes after the word's first and second column */
          kv[u] = word_prefix(wv[u]) + run2;
          run2 = __builtin_amdgcn_perm(kv[u], kv[u], 0x03020302u); /* the high half, twice */
          d[u] = sub_sat_u16x2(kv[u], kd[u]);
          any |= d[u];
        }
        if (__ballot(any != 0u)) {
          /* listed cells as a bit per column, then one per lane and step */
          uint32_t left = 0u;
#pragma unroll
          for (uint32_t u = 0; u < kCutWords; ++u)
            left |= ((d[u] & 0xFFFFu) ? 1u << (2u * u) : 0u) | (d[u] > 0xFFFFu ? 2u << (2u * u) : 0u);
          uint64_t m = __ballot(left != 0u);
#pragma unroll 1
          do {
            if (n0 > (uint32_t)kCand0Cap - 64u)
              flush_cut<NT>(J, S, cand0, n0, cand, nc, c3, n3, xb, zb, Uw, U2w, st);
            if (left) {
              const uint32_t c = (uint32_t)__builtin_ctz(left);
              uint32_t k = kv[0];
#pragma unroll
              for (uint32_t u = 1; u < kCutWords; ++u) k = (c >> 1) == u ? kv[u] : k;
              k = (c & 1u) ? k >> 16 : k & 0xFFFFu;
              cand0[n0 + mask_lt(m)] = make_uint2((i << 16) | (2u * (s * kCutSpan + lane * kCutWords) + c), k);
              left &= left - 1u;
            }
            n0 += (uint32_t)__popcll(m);
            m = __ballot(left != 0u);
          } while (m);
        }
#pragma unroll
        for (uint32_t u = 0; u < kCutWords; ++u) kd[u] = kn[u];
      }
    }
    uint64_t tc3 = cycles();
    st.cyc[2] += tc3 - tc2;
    if (n0) flush_cut<NT>(J, S, cand0, n0, cand, nc, c3, n3, xb, zb, Uw, U2w, st);
    if (nc) flush_candidates<NT>(J, S, cand, nc, c3, n3, xb, Uw, U2w, st);
    {
      const float U2o = fminf(U2w, log_bound_of(xb));
      share_bound(S, U2o);
      const float U2s = fminf(U2o, shared_bound(S));
      if (n3) flush_exact(J, S, c3, n3, U2s, xb, st);
    }
    const ZeroKey zw = wave_zero(zb);
    if (lane == 0) {
      S.redB[w] = class_key(0.0, zw);
      S.redB[2 * W + w] = xb;
    }
    __syncthreads();
    st.cyc[4] += cycles() - tc3;
    double pmin = __builtin_inf();
    for (uint32_t v = 0; v < W; ++v) {
      if (S.redB[v].ij != kNone) pmin = 0.0;
      if (S.redB[2 * W + v].ij != kNone) pmin = fmin(pmin, S.redB[2 * W + v].p);
    }
    if (lev == 0u || pmin <= exp((double)J.cut_level[lev])) {
      /* p == 1 cells matter only when no cell has p < 1 */
      if (pmin < 1.0) {
        if (lane == 0) S.redB[W + w] = no_best();
      } else {
        const ZeroKey o = class1_best<NT, true>(J, Lo, S, C);
        if (lane == 0) S.redB[W + w] = class_key(1.0, o);
      }
      __syncthreads();
      break;
    }
    /* no cell at or below the level: again with the next table */
    xb = no_best();
    zb = {0u, kNone, 0u, 0u};
    tc1 = cycles();
    for (uint32_t t = lane; t < T2w_pad; t += 64u) C[t] = 0u;
    __syncthreads();
  }
  /* the classes hold disjoint cells: p == 0, p == 1 (k <= max(0, K + n - N))
   * and evaluated cells; the tie counts add up across them */
  BestKey b = no_best();
  if (tid == 0)
    for (uint32_t v = 0; v < 3 * W; ++v) merge_best(b, S.redB[v]);
  __syncthreads();
  return b;
}

/* Permutations [perm_base, perm_base + n_perm) of one job, optionally after
 * the unpermuted task (lead = 1: task 0, record 0).  EXPLICIT: idx1 / idx2
 * hold n_perm permutations back to back (NULL: identity); otherwise the Philox
 * shuffle keyed by (seed, job_id, permutation id, list).  ws: per workgroup
 * pair staging (N2 u16 each) in kBuildGlobal.  Workgroups take tasks from a device
 * counter (zeroed before the launch); every workgroup exits once the counter
 * passes the task count. */
template <int NT, bool EXPLICIT, int BUILD>
__global__ __launch_bounds__(NT, 4) void k_cut(DevJob J, LdsLayout Lo, const uint32_t *__restrict__ idx1,
                                            const uint32_t *__restrict__ idx2, uint64_t n_perm, uint64_t perm_base,
                                            uint64_t seed, uint32_t job_id, int32_t permuted, uint32_t lead,
                                            dto_record *__restrict__ out, int *__restrict__ err,
                                            uint16_t *__restrict__ ws, uint32_t *__restrict__ counter) {
  extern __shared__ __align__(16) unsigned char smem[];
  uint32_t &s_next = *(uint32_t *)(smem + Lo.misc);
  const Lds S = lds_view<true>(smem, Lo, NT / 64, nullptr);
  load_cut_tables<NT, BUILD>(J, Lo, S, smem);
  uint16_t *gpairs = BUILD != kBuildGlobal ? nullptr : ws + (uint64_t)blockIdx.x * J.N2;
  WaveStats st = {0u, 0u, 0u, {0, 0, 0, 0, 0}, 0u, 0u, 0u, 0u, 0u};
  if (threadIdx.x == 0) s_next = atomicAdd(counter, 1u);
  __syncthreads();
  uint64_t pp = s_next;
  __syncthreads();
  const uint64_t tasks = n_perm + lead;
  while (pp < tasks) {
    const bool first = pp < lead;
    const uint64_t q = pp - lead;
    const uint32_t *i1 = (EXPLICIT && idx1 && !first) ? idx1 + q * J.N1 : nullptr;
    const uint32_t *i2 = (EXPLICIT && idx2 && !first) ? idx2 + q * J.N2 : nullptr;
    Shuffle s1, s2;
    if (!EXPLICIT) {
      s1 = shuffle_make(seed, job_id, (uint32_t)(perm_base + q), 1u, J.N1);
      s2 = shuffle_make(seed, job_id, (uint32_t)(perm_base + q), 2u, J.N2);
      s1.ident = s2.ident = first ? 1u : 0u;
    }
    const BestKey b = optimize_cut<NT, EXPLICIT, BUILD>(J, Lo, S, i1, i2, s1, s2, err, st, smem, gpairs, counter, &s_next);
    /* the value claimed during this task, published by its barriers */
    const uint64_t pn = s_next;
    if (threadIdx.x == 0) write_record(J, b, first ? 0 : permuted, out + pp, err);
    wave_sync(); /* keeps thread 0's block apart from the next iteration's (see k_plain) */
    pp = pn;
  }
  flush_stats(J, st);
}

/* k_batch for jobs with cut tables (see there for the queue). */
template <int NT, int BUILD>
__global__ __launch_bounds__(NT, 4) void k_batch_cut(const BatchJob *__restrict__ jobs, const WorkItem *__restrict__ items,
                                                  uint32_t n_items, uint64_t seed, uint32_t *__restrict__ counter,
                                                  int *__restrict__ err, uint16_t *__restrict__ ws, uint32_t ws_stride,
                                                  uint32_t item_slot) {
  extern __shared__ __align__(16) unsigned char smem[];
  uint32_t &s_item = *(uint32_t *)(smem + item_slot);
  uint16_t *gpairs = BUILD != kBuildGlobal ? nullptr : ws + (uint64_t)blockIdx.x * ws_stride;
  uint32_t cur = kNone;
  WaveStats st = {0u, 0u, 0u, {0, 0, 0, 0, 0}, 0u, 0u, 0u, 0u, 0u};
  for (;;) {
    if (threadIdx.x == 0) s_item = atomicAdd(counter, 1u);
    __syncthreads();
    const uint32_t it = s_item;
    __syncthreads();
    if (it >= n_items) break;
    const WorkItem wi = items[it];
    const BatchJob &B = jobs[wi.job];
    const Lds S = lds_view<true>(smem, B.lo, NT / 64, nullptr);
    if (wi.job != cur) {
      load_cut_tables<NT, BUILD>(B.J, B.lo, S, smem);
      __syncthreads();
      cur = wi.job;
    }
    for (uint32_t t = wi.t0; t < wi.t0 + wi.count; ++t) {
      Shuffle s1 = shuffle_make(seed, B.job_id, t - 1u, 1u, B.J.N1);
      Shuffle s2 = shuffle_make(seed, B.job_id, t - 1u, 2u, B.J.N2);
      s1.ident = s2.ident = t == 0 ? 1u : 0u;
      const BestKey b =
          optimize_cut<NT, false, BUILD>(B.J, B.lo, S, nullptr, nullptr, s1, s2, err, st, smem, gpairs, nullptr, nullptr);
      if (threadIdx.x == 0) write_record(B.J, b, t == 0 ? 0 : 1, B.out + t, err);
      wave_sync(); /* keeps thread 0's block apart from the next iteration's (see k_plain) */
    }
  }
}

}  // namespace dto
