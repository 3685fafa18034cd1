/*
 * The plain kernels: every cell's exact FP64 tail, as the plain mode's best
 * cell (k_plain) or as the full record grid (k_grid_pvalues).
 */
#pragma once
#include "dto_kernels.h"

#pragma clang fp contract(off)

namespace dto {

/* dto_tail_exact with U terms in flight: their table loads and exps are
 * independent, and only the additions, made in the same ascending order with
 * the same early exit, are serial, so the sum is bit-identical.  One term at a
 * time waits for four table reads and an exp per addition.  Four where the
 * tasks fill the GPU (49 plain tasks at N = 6,000: 2.45 ms, 2.87 with eight);
 * eight for the one grid of a call, which waits for its longest tails (599 x
 * 599 records: 247 us, 256 with four). */
template <uint32_t U>
__device__ __forceinline__ double tail_exact_wide(const double *LF, uint32_t N, uint32_t K, uint32_t n, uint32_t k,
                                                  double d, const uint64_t *tab) {
  if (k == 0) return 1.0;
  const uint32_t x = k - 1, mn = (K + n > N) ? K + n - N : 0, mx = K < n ? K : n;
  if (x < mn) return 1.0;
  if (x >= mx) return 0.0;
  const double lfK = LF[K], lfNK = LF[N - K];
  const uint32_t NK = N - K;
  double acc = 0.0;
  for (uint32_t i0 = k; i0 <= mx; i0 += U) {
    double t[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint32_t i = min(i0 + u, mx);
      const double lb1 = (lfK - LF[i]) - LF[K - i];
      const double lb2 = (lfNK - LF[n - i]) - LF[NK - (n - i)];
      t[u] = (lb1 + lb2) - d;
    }
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) t[u] = dto_exp(t[u], tab);
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint32_t i = i0 + u;
      if (i > mx) return acc;
      acc = acc + t[u];
      if (t[u] * 0x1p56 <= acc) {
        /* rho_i <= 1 - 2^-20, checked as num <= den - ceil(den / 2^20) */
        const uint64_t num = (uint64_t)(K - i) * (uint64_t)(n - i);
        const uint64_t den = (uint64_t)(i + 1) * (uint64_t)(NK - n + i + 1);
        if (num <= den - ((den + 0xFFFFFull) >> 20)) return acc;
      }
    }
  }
  return acc;
}

/* Plain mode.  A work item is one task's rows i with (i / W) % parts == part:
 * a launch of few tasks splits each over several workgroups, each building
 * the task's rows for itself (a few per cent of the tails' time), and leaves
 * its best cell in partial[item] for k_plain_reduce; with parts == 1 it
 * writes the record.  The lanes of a wave take 128 neighbouring columns at a
 * time, whose tails are of similar length.  Items come from a device counter
 * (zeroed before the launch); every workgroup exits once it passes n_perm *
 * parts.  49 tasks at N = 6,000: 2.45 ms, 25.7 ms with a workgroup a task,
 * ten neighbouring columns a lane and one term at a time. */
template <int NT, bool EXPLICIT, bool PL>
__global__ __launch_bounds__(NT) void k_plain(DevJob J, LdsLayout Lo, const uint32_t *__restrict__ idx1,
                                              const uint32_t *__restrict__ idx2, uint64_t n_perm, uint64_t perm_base,
                                              uint64_t seed, uint32_t job_id, int32_t permuted, uint32_t parts,
                                              BestKey *__restrict__ partial, dto_record *__restrict__ out,
                                              int *__restrict__ err, uint16_t *__restrict__ ws,
                                              uint32_t *__restrict__ counter) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr uint32_t W = NT / 64;
  uint32_t &s_next = *(uint32_t *)(smem + Lo.misc);
  const Lds S = lds_view<true>(smem, Lo, W, nullptr);
  const uint32_t lane = lane_id(), w = wave_id();
  for (uint32_t t = threadIdx.x; t < 256; t += NT) S.tab[t] = kExpTabC[t];
  for (uint32_t t = threadIdx.x; t < J.T2; t += NT) S.coln[t] = J.n[t];
  uint16_t *gpairs = PL ? nullptr : ws + (uint64_t)blockIdx.x * J.N2;
  uint32_t *C = S.cw + w * Lo.T2w_pad;
  const uint32_t T1 = J.T1, T2 = J.T2, T2w = J.T2w;
  for (;;) {
    if (threadIdx.x == 0) s_next = atomicAdd(counter, 1u);
    __syncthreads();
    const uint64_t item = s_next;
    __syncthreads();
    const uint64_t pp = item / parts;
    const uint32_t part = (uint32_t)(item % parts);
    if (pp >= n_perm) break;
    const uint32_t *i1 = (EXPLICIT && idx1) ? idx1 + pp * J.N1 : nullptr;
    const uint32_t *i2 = (EXPLICIT && idx2) ? idx2 + pp * J.N2 : nullptr;
    Shuffle s1, s2;
    if (!EXPLICIT) {
      s1 = shuffle_make(seed, job_id, (uint32_t)(perm_base + pp), 1u, J.N1);
      s2 = shuffle_make(seed, job_id, (uint32_t)(perm_base + pp), 2u, J.N2);
    }
    build_rows<NT, EXPLICIT, false, PL, true>(J, Lo, S, i1, i2, s1, s2, err, gpairs);
    BestKey xb = no_best();
    uint32_t added = 0;
    for (uint32_t i = part * W + w; i < T1; i += parts * W) {
      rows_update<true>(S, C, added, i + 1u, true);
      added = i + 1u;
      const uint32_t K = J.K[i];
      uint32_t carry = 0;
      for (uint32_t w0 = 0; w0 < T2w; w0 += 64u) {
        const uint32_t wi = w0 + lane, x = wi < T2w ? C[wi] : 0u;
        const uint32_t tot = (x & 0xFFFFu) + (x >> 16), incl = wave_incl_scan(tot);
        uint32_t k = carry + incl - tot;
        carry += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
#pragma unroll 1
        for (uint32_t h = 0; h < 2; ++h) {
          const uint32_t j = 2u * wi + h;
          k += h ? x >> 16 : x & 0xFFFFu;
          if (j < T2) take_better(xb, tail_exact_wide<4>(J.LF, J.N, K, S.coln[j], k, J.D[j], S.tab), k, (i << 16) | j);
        }
      }
    }
    xb = wave_best(xb);
    if (lane == 0) S.redB[w] = xb;
    __syncthreads();
    if (threadIdx.x == 0) {
      BestKey b = no_best();
      for (uint32_t v = 0; v < W; ++v) merge_best(b, S.redB[v]);
      if (parts > 1u)
        partial[item] = b;
      else
        write_record(J, b, permuted, out + pp, err);
    }
    /* without a barrier here the compiler joins this iteration's "thread 0
     * only" block to the next one's, and lets the other lanes of its wave go
     * round the loop, past the claim's barrier, ahead of thread 0 */
    __syncthreads();
  }
}

/* The parts' best cells of each task -> its record. */
static __global__ __launch_bounds__(64) void k_plain_reduce(DevJob J, const BestKey *__restrict__ partial,
                                                            uint32_t parts, uint32_t n_perm, int32_t permuted,
                                                            dto_record *__restrict__ out, int *__restrict__ err) {
  const uint32_t t = blockIdx.x * 64u + threadIdx.x;
  if (t >= n_perm) return;
  BestKey b = no_best();
  for (uint32_t v = 0; v < parts; ++v) merge_best(b, partial[(uint64_t)t * parts + v]);
  write_record(J, b, permuted, out + t, err);
}

/* Overlap counts of every cell of one permutation: the workgroups build the
 * rows each for itself, and wave s of all takes rows s, s + waves, ...
 * (a launch of one workgroup swept every row after the other: with 64, 45 us
 * for the 599 rows at N = 20,000, most of it the build). */
template <int NT, bool PL>
__global__ __launch_bounds__(NT) void k_grid_counts(DevJob J, LdsLayout Lo, const uint32_t *__restrict__ idx1,
                                                    const uint32_t *__restrict__ idx2, uint32_t *__restrict__ kout,
                                                    int *__restrict__ err, uint16_t *__restrict__ ws) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr uint32_t W = NT / 64;
  const Lds S = lds_view<true>(smem, Lo, W, nullptr);
  Shuffle s1, s2;
  build_rows<NT, true, false, PL>(J, Lo, S, idx1, idx2, s1, s2, err, PL ? nullptr : ws + (uint64_t)blockIdx.x * J.N2);
  const uint32_t w = wave_id(), lane = lane_id();
  const uint32_t T1 = J.T1, T2 = J.T2, T2w = J.T2w;
  uint32_t *C = S.cw + w * Lo.T2w_pad;
  uint32_t added = 0;
  for (uint32_t i = blockIdx.x * W + w; i < T1; i += gridDim.x * W) {
    rows_update<true>(S, C, added, i + 1u, true);
    added = i + 1u;
    uint32_t carry = 0;
    for (uint32_t w0 = 0; w0 < T2w; w0 += 64u) {
      const uint32_t wi = w0 + lane, x = wi < T2w ? C[wi] : 0u;
      const uint32_t tot = (x & 0xFFFFu) + (x >> 16), incl = wave_incl_scan(tot);
      const uint32_t k1 = carry + incl, k0 = k1 - (x >> 16);
      carry += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
      if (2u * wi < T2) kout[(uint64_t)i * T2 + 2u * wi] = k0;
      if (2u * wi + 1u < T2) kout[(uint64_t)i * T2 + 2u * wi + 1u] = k1;
    }
  }
}

/* Exact p-value of every cell from the count grid.  A wave's 64 records are
 * put together in LDS and stored as consecutive 8-byte words (72-byte
 * records written lane by lane touch every line 18 times). */
static __global__ __launch_bounds__(256) void k_grid_pvalues(DevJob J, const uint32_t *__restrict__ kin,
                                                             int32_t permuted, dto_record *__restrict__ out) {
  __shared__ uint64_t tab[256];
  __shared__ __align__(16) dto_record stage[4][64];
  tab[threadIdx.x] = kExpTabC[threadIdx.x];
  __syncthreads();
  const uint32_t lane = lane_id(), w = wave_id();
  const uint64_t cells = (uint64_t)J.T1 * J.T2;
  /* from the last cells on: the long tails are in the later rows, and would
   * otherwise run on when the rest is done */
  const uint64_t batches = (cells + 63u) / 64u;
  for (uint64_t q = (uint64_t)blockIdx.x * 4u + w; q < batches; q += (uint64_t)gridDim.x * 4u) {
    const uint64_t c0 = (batches - 1u - q) * 64u;
    const uint64_t c = c0 + lane;
    if (c < cells) {
      const uint32_t i = (uint32_t)(c / J.T2), j = (uint32_t)(c % J.T2);
      const uint32_t k = kin[c];
      const double p = tail_exact_wide<8>(J.LF, J.N, J.K[i], J.n[j], k, J.D[j], tab);
      write_record(J, BestKey{p, k, (i << 16) | j, 0u, 0u}, permuted, &stage[w][lane], nullptr);
    }
    wave_sync();
    const uint32_t cnt = (uint32_t)(cells - c0 < 64u ? cells - c0 : 64u);
    static_assert(sizeof(dto_record) % 8 == 0, "records are stored as 8-byte words");
    const uint64_t *src = (const uint64_t *)stage[w];
    uint64_t *dst = (uint64_t *)(out + c0);
    for (uint32_t t = lane; t < cnt * (uint32_t)(sizeof(dto_record) / 8u); t += 64u) dst[t] = src[t];
    wave_sync();
  }
}

}  // namespace dto
