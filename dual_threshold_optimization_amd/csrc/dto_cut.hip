/*
 * Launches of the screened kernels (dto_cut.h): a job's cut tables, the
 * permutations of one job, and batches of jobs.
 */
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <string>

#include "../../include/dto.h"
#include "dto_cut.h"
#include "dto_internal.h"

using namespace dto;

static uint32_t align16(uint32_t x) { return (x + 15u) & ~15u; }

bool dto::cut_layout(const HostJob &h, int W, int build, LdsLayout *out) {
  LdsLayout L{};
  const uint32_t N1 = (uint32_t)h.l1.ids.size(), N2 = (uint32_t)h.l2.ids.size();
  const uint32_t T1 = (uint32_t)h.thr1.size(), T2 = (uint32_t)h.thr2.size();
  const uint32_t T2w = (T2 + 1) / 2, w = (uint32_t)W;
  if (build == kBuildRegs) {
    const uint32_t most = kRegPairs * 64u * w;
    if (h.dup || shuffle_make(0, 0, 0, 1, N1).dom > most || shuffle_make(0, 0, 0, 2, N2).dom > most) return false;
  }
  L.T2w_pad = ((T2w + 1u) & ~1u) + kCutWords; /* a lane's run of zero words ends each wave's counts */
  L.pairs_in_lds = build != kBuildGlobal ? 1u : 0u;
  L.nb_in_lds = 1u;
  /* the build's staging and cursors, then the sweep's lists in their place */
  L.cursor = build == kBuildLds ? align16(2u * std::max(N2, 1u)) : 0u;
  L.cand0 = 0u;
  L.cand = L.cand0 + 8u * w * (uint32_t)kCand0Cap;
  L.cand3 = L.cand + 8u * w * (uint32_t)kCandCap;
  uint32_t at = align16(std::max(L.cursor + 4u * T1, L.cand3 + 16u * w * (uint32_t)kCand3Cap));
  auto region = [&](uint32_t &field, uint32_t bytes) {
    field = at;
    at = align16(at + bytes);
  };
  region(L.nb, 2u * std::max(std::max(N1, N2), 1u));
  region(L.join, build == kBuildRegs ? 2u * N2 : 0u);
  region(L.rowstart, 4u * (T1 + 1u));
  region(L.cw, 4u * w * L.T2w_pad);
  region(L.coln, 4u * T2);
  region(L.exptab, 8u * 256u);
  region(L.red, (16u + 3u * (uint32_t)sizeof(BestKey) + 16u) * w);
  region(L.misc, 16u);
  L.total = at;
  *out = L;
  return true;
}

/* One shape for a set of jobs: 512-thread workgroups where two or more fit a
 * CU (the waves of one hide the barriers of another), else 1,024 threads, so
 * that a CU holds 16 waves either way; the first build that every job fits.
 * Where 16 waves' column counts do not fit beside the lists or the thresholds
 * (reference thresholds: above 49,800 entries), 512 threads, 8 waves a CU. */
int dto::cut_shape(const HostJob *const *jobs, size_t n, size_t lim, CutShape *out) {
  const struct {
    int nt, build;
    uint32_t per_cu;
  } tries[] = {{512, kBuildRegs, 2},  {512, kBuildLds, 2}, {1024, kBuildRegs, 1},  {1024, kBuildLds, 1},
               {1024, kBuildGlobal, 1}, {512, kBuildLds, 1}, {512, kBuildGlobal, 1}};
  for (const auto &t : tries) {
    uint32_t most = 0;
    bool fit = true;
    for (size_t i = 0; i < n && fit; ++i) {
      LdsLayout L;
      fit = cut_layout(*jobs[i], t.nt / 64, t.build, &L);
      if (fit) most = std::max(most, L.total);
    }
    if (!fit || (size_t)most * t.per_cu > lim) continue;
    *out = {t.nt, t.build, most};
    return DTO_OK;
  }
  return fail(DTO_ERR_TOO_LARGE, "job does not fit in LDS");
}

void dto::cut_levels(const HostJob &h, DevJob &d) {
  d.cut_segs = (uint32_t)((h.thr2.size() + 2u * kCutSpan - 1u) / (2u * kCutSpan));
  const double cells = (double)h.thr1.size() * (double)h.thr2.size();
  /* the start level: about where nine null permutations in ten have a cell
   * below it (their minimum falls with the log of the number of cells); then
   * steps for null minima, and wide ones for planted overlaps.  Above it,
   * small steps down to nearly p = 1: level 0 lists every cell with p < 1
   * (on a 4M-cell grid milliseconds for one permutation).  With 10 levels
   * the genome-scale job was 8 % slower and the 4M-cell grid 1.8 times. */
  const double l0 = std::min(-1.0, 1.1 - 0.45 * log(cells));
  const double level[kCutLevels] = {0.0,      0.15 * l0, 0.3 * l0,  0.5 * l0,  0.75 * l0, l0,         l0 - 1.5,
                                    l0 - 4.0, l0 - 8.0,  l0 - 16.0, l0 - 35.0, l0 - 75.0, l0 - 160.0, l0 - 340.0};
  for (uint32_t l = 0; l < kCutLevels; ++l) d.cut_level[l] = (float)level[l];
}

int dto::cut_tables(dto_job *j, hipStream_t st, const uint32_t **out) {
  std::lock_guard<std::mutex> g(j->cut_mu);
  *out = j->cut;
  if (j->cut && !j->cut_pending) return DTO_OK;
  RelaxedCapture relaxed;
  const bool capturing = stream_capturing(st);
  if (j->cut) {
    const hipError_t q = hipEventQuery(j->cut_ev);
    if (q == hipSuccess) {
      j->cut_pending = false;
      return DTO_OK;
    }
    (void)hipGetLastError();
    if (q != hipErrorNotReady) return fail(DTO_ERR_DEVICE, std::string("cut tables: ") + hipGetErrorString(q));
    /* a capture cannot wait on work recorded outside it */
    if (capturing) HIP_TRY(hipEventSynchronize(j->cut_ev));
    else HIP_TRY(hipStreamWaitEvent(st, j->cut_ev, 0));
    return DTO_OK;
  }
  const size_t per_level = (size_t)j->dev.T1 * j->dev.cut_segs * 2u * kCutSpan;
  if (!j->cut_ev) HIP_TRY(hipEventCreateWithFlags(&j->cut_ev, hipEventDisableTiming));
  void *p = nullptr;
  /* the sweep loads one row's segment past the last */
  const size_t bytes = (kCutLevels * per_level + 2u * kCutSpan) * sizeof(uint16_t);
  if (j->alloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return DTO_OK;
  }
  /* a captured launch would only build them when it is replayed: they are
   * built beside the capture, and are complete before it goes on */
  hipStream_t b = st;
  hipError_t e = capturing ? hipStreamCreateWithFlags(&b, hipStreamNonBlocking) : hipSuccess;
  if (e == hipSuccess) {
    const uint32_t grid = (uint32_t)std::min<size_t>((per_level + 255) / 256, 65536);
    hipLaunchKernelGGL(k_cut_table, dim3(grid), dim3(256), 0, b, j->dev, (uint16_t *)p);
    e = hipGetLastError();
    if (e == hipSuccess) e = capturing ? hipStreamSynchronize(b) : hipEventRecord(j->cut_ev, b);
    if (capturing) (void)hipStreamDestroy(b);
  }
  if (e != hipSuccess) {
    (void)hipFree(p);
    return fail(DTO_ERR_DEVICE, std::string("cut tables: ") + hipGetErrorString(e));
  }
  *out = j->cut = (uint32_t *)p;
  j->cut_bytes = bytes;
  j->cut_pending = !capturing;
  return DTO_OK;
}

template <int NT, int BUILD, bool E>
static hipError_t launch_t(dto_job *j, const uint32_t *cut, uint32_t grid, hipStream_t st, const uint32_t *i1, const uint32_t *i2,
                           uint64_t n_perm, uint64_t base, uint64_t seed, uint32_t job_id, int32_t permuted,
                           uint32_t lead, dto_record *out) {
  auto kern = k_cut<NT, E, BUILD>;
  const LdsLayout &lo = j->lo_cut;
  (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lo.total);
  uint32_t *ctr = j->d_ctr + j->slots.take(st);
  DevJob dev = j->dev;
  dev.cut = cut;
  StagingOrder order(j, lo, st);
  hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(64), 0, st, ctr);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(NT), lo.total, st, dev, lo, i1, i2, n_perm, base, seed, job_id, permuted,
                     lead, out, j->d_err, j->ws, ctr);
  return hipGetLastError();
}

hipError_t dto::launch_cut(dto_job *j, const uint32_t *cut, bool expl, uint32_t grid, hipStream_t st,
                           const uint32_t *i1, const uint32_t *i2, uint64_t n_perm, uint64_t base, uint64_t seed, uint32_t job_id,
                           int32_t permuted, uint32_t lead, dto_record *out) {
#define DTO_CUT(NT, B)                                                                                               \
  if (j->cut_sh.nt == NT && j->cut_sh.build == B)                                                                    \
    return expl ? launch_t<NT, B, true>(j, cut, grid, st, i1, i2, n_perm, base, seed, job_id, permuted, lead, out)   \
                : launch_t<NT, B, false>(j, cut, grid, st, i1, i2, n_perm, base, seed, job_id, permuted, lead, out);
  DTO_CUT(512, kBuildRegs)
  DTO_CUT(512, kBuildLds)
  DTO_CUT(512, kBuildGlobal)
  DTO_CUT(1024, kBuildRegs)
  DTO_CUT(1024, kBuildLds)
  DTO_CUT(1024, kBuildGlobal)
#undef DTO_CUT
  return hipErrorInvalidValue;
}

template <int NT, int BUILD>
static hipError_t batch_t(uint32_t grid, uint32_t lds, hipStream_t st, const BatchJob *jobs, const WorkItem *items,
                          uint32_t n_items, uint64_t seed, uint32_t *counter, int *err, uint16_t *ws,
                          uint32_t ws_stride) {
  auto kern = k_batch_cut<NT, BUILD>;
  (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  /* every layout ends with its 16-byte misc slot: the largest one's is free in all */
  hipLaunchKernelGGL(kern, dim3(grid), dim3(NT), lds, st, jobs, items, n_items, seed, counter, err, ws, ws_stride,
                     lds - 16u);
  return hipGetLastError();
}

hipError_t dto::launch_batch_cut(const CutShape &sh, uint32_t grid, hipStream_t st, const BatchJob *jobs,
                                 const WorkItem *items, uint32_t n_items, uint64_t seed, uint32_t *counter, int *err,
                                 uint16_t *ws, uint32_t ws_stride) {
#define DTO_CUT(NT, B)            \
  if (sh.nt == NT && sh.build == B) \
    return batch_t<NT, B>(grid, sh.lds, st, jobs, items, n_items, seed, counter, err, ws, ws_stride);
  DTO_CUT(512, kBuildRegs)
  DTO_CUT(512, kBuildLds)
  DTO_CUT(512, kBuildGlobal)
  DTO_CUT(1024, kBuildRegs)
  DTO_CUT(1024, kBuildLds)
  DTO_CUT(1024, kBuildGlobal)
#undef DTO_CUT
  return hipErrorInvalidValue;
}
