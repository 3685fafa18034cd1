/*
 * Launches of the plain kernels (dto_plain.h): the plain mode and the debug
 * grid.
 */
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/dto.h"
#include "dto_internal.h"
#include "dto_plain.h"

using namespace dto;

/* The launch's slot of the buffer of partial results that the job keeps from
 * its first split launch on, or NULL where there is no memory for it (the
 * launch is then not split). */
static BestKey *partial_slot(dto_job *j, uint32_t slot) {
  std::lock_guard<std::mutex> g(j->cut_mu);
  if (!j->partial) {
    const size_t bytes = (size_t)kCounterSlots * kSplitItems * sizeof(BestKey);
    if (j->alloc(&j->partial, bytes) != hipSuccess) {
      (void)hipGetLastError();
      j->partial = nullptr;
      return nullptr;
    }
    j->partial_bytes = bytes;
  }
  return (BestKey *)j->partial + (size_t)slot * kSplitItems;
}

template <bool E, bool PL>
static hipError_t launch_t(dto_job *j, uint32_t max_grid, hipStream_t st, const uint32_t *i1, const uint32_t *i2,
                           uint64_t n_perm, uint64_t base, uint64_t seed, uint32_t job_id, int32_t permuted,
                           dto_record *out, BestKey *part) {
  auto kern = k_plain<kNT, E, PL>;
  const LdsLayout &lo = j->lo_plain;
  (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lo.total);
  const uint32_t slot = j->slots.take(st);
  uint32_t *ctr = j->d_ctr + slot;
  uint32_t parts = 1;
  BestKey *partial = part;
  if (n_perm <= kSplitTasks) {
    parts = std::min<uint32_t>(kSplitItems / (uint32_t)n_perm, (j->dev.T1 + kNT / 64 - 1) / (kNT / 64));
    if (parts > 1 && !partial && !(partial = partial_slot(j, slot))) parts = 1;
  }
  const uint32_t grid = (uint32_t)std::min<uint64_t>(n_perm * parts, max_grid);
  StagingOrder order(j, lo, st);
  hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(64), 0, st, ctr);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kNT), lo.total, st, j->dev, lo, i1, i2, n_perm, base, seed, job_id,
                     permuted, parts, partial, out, j->d_err, j->ws, ctr);
  if (parts > 1)
    hipLaunchKernelGGL(k_plain_reduce, dim3(((uint32_t)n_perm + 63u) / 64u), dim3(64), 0, st, j->dev, partial, parts,
                       (uint32_t)n_perm, permuted, out, j->d_err);
  return hipGetLastError();
}

hipError_t dto::launch_plain(dto_job *j, bool expl, uint32_t max_grid, hipStream_t st, const uint32_t *i1,
                             const uint32_t *i2, uint64_t n_perm, uint64_t base, uint64_t seed, uint32_t job_id,
                             int32_t permuted, dto_record *out, BestKey *part) {
  if (j->lo_plain.pairs_in_lds)
    return expl ? launch_t<true, true>(j, max_grid, st, i1, i2, n_perm, base, seed, job_id, permuted, out, part)
                : launch_t<false, true>(j, max_grid, st, i1, i2, n_perm, base, seed, job_id, permuted, out, part);
  return expl ? launch_t<true, false>(j, max_grid, st, i1, i2, n_perm, base, seed, job_id, permuted, out, part)
              : launch_t<false, false>(j, max_grid, st, i1, i2, n_perm, base, seed, job_id, permuted, out, part);
}

/* The debug grid of one permutation on a stream: overlap counts into kcnt
 * (T1 * T2 words), then every cell's exact record into out; an out-of-range
 * permutation index sets *err. */
hipError_t dto::launch_grid(dto_job *job, const uint32_t *d1, const uint32_t *d2, uint32_t *kcnt, dto_record *out,
                            int *err, hipStream_t st) {
  const size_t cells = (size_t)job->dev.T1 * job->dev.T2;
  const LdsLayout &lo = job->lo_plain;
  /* one row a wave, up to 64 workgroups: past that the redundant builds only
   * load the caches */
  const uint32_t gc = std::min<uint32_t>((job->dev.T1 + kNT / 64 - 1) / (kNT / 64), 64u);
  if (lo.pairs_in_lds) {
    auto kern = k_grid_counts<kNT, true>;
    (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lo.total);
    hipLaunchKernelGGL(kern, dim3(gc), dim3(kNT), lo.total, st, job->dev, lo, d1, d2, kcnt, err, job->ws);
  } else {
    auto kern = k_grid_counts<kNT, false>;
    (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lo.total);
    StagingOrder order(job, lo, st);
    hipLaunchKernelGGL(kern, dim3(gc), dim3(kNT), lo.total, st, job->dev, lo, d1, d2, kcnt, err, job->ws);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int32_t permuted = (d1 || d2) ? 1 : 0;
  const uint32_t g = (uint32_t)std::min<size_t>((cells + 255) / 256, 8192);
  hipLaunchKernelGGL(k_grid_pvalues, dim3(g), dim3(256), 0, st, job->dev, (const uint32_t *)kcnt, permuted, out);
  return hipGetLastError();
}
