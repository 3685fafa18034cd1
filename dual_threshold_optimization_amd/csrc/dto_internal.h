/*
 * Library-internal state shared by the translation units of libdto_amd.so.
 */
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <mutex>
#include <string>
#include <vector>

#include "dto_device.h"
#include "dto_host.hpp"

#define HIP_TRY(expr)                                                                                      \
  do {                                                                                                     \
    hipError_t e_ = (expr);                                                                                \
    if (e_ != hipSuccess) return dto::fail(DTO_ERR_DEVICE, std::string(#expr ": ") + hipGetErrorString(e_)); \
  } while (0)

namespace dto {
constexpr int kNT = 512; /* threads per workgroup of the grid kernels (8 waves) */

struct DevProps {
  int ok = 0;
  int cus = 0;
  size_t lds_per_block = 0;
};
int current_device(int *dev);
int device_props(int dev, DevProps *out);
/* with_h: the screen table in LDS; nb_lds: the bins array in LDS (else a
 * per-workgroup global slice of max(N1, N2) u16). */
LdsLayout make_layout(const HostJob &h, int W, bool with_h, size_t lds_limit, bool nb_lds = true);
/* The screened kernels' layout for a job: table and bins in LDS when they
 * fit, else the table in LDS and the bins global, else the table global. */
LdsLayout screen_layout(const HostJob &h, int W, size_t lds_limit);
/* The cut kernels (dto_cut.h): how pairs are built, the layout at W waves
 * (false: the job's lists rule the build out), the shape taken for a set of
 * jobs, and the levels of a job's cut tables. */
bool cut_layout(const HostJob &h, int W, int build, LdsLayout *out);
struct CutShape {
  int nt = 0, build = 0;
  uint32_t lds = 0; /* the largest layout's */
};
int cut_shape(const HostJob *const *jobs, size_t n, size_t lds_limit, CutShape *out);
void cut_levels(const HostJob &h, DevJob &d);
}  // namespace dto

inline bool stream_capturing(hipStream_t st) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cs) != hipSuccess) (void)hipGetLastError();
  return cs != hipStreamCaptureStatusNone;
}

/* Slots of a job's work counters (and of its partial results), one per
 * launch, so that launches on different streams do not share one: a ring for
 * launches that run at once, and one for captured launches, which keep their
 * slot for every replay and would otherwise share it with each 256th ordinary
 * launch.  Only more launches in flight at once than the ring has slots, or
 * replays of captured launches more than kCaptureRing apart, meet. */
constexpr uint32_t kCounterRing = 256, kCaptureRing = 64, kCounterSlots = kCounterRing + kCaptureRing;
struct LaunchSlots {
  std::atomic<uint32_t> ordinary{0}, captured{0};
  uint32_t take(bool capturing) {
    return capturing ? kCounterRing + captured.fetch_add(1u) % kCaptureRing : ordinary.fetch_add(1u) % kCounterRing;
  }
  uint32_t take(hipStream_t st) { return take(stream_capturing(st)); }
};
/* Plain launches of at most kSplitTasks tasks split each over several
 * workgroups, kSplitItems in all, whose partial results go to a buffer of that
 * size: two for each of this GPU's 256 CUs (a task alone fills it; 257 tasks
 * and more occupy it as they are). */
constexpr uint32_t kSplitTasks = 256, kSplitItems = 512;
/* A resident job's room for small calls (upload_job), after its tables: the
 * error word's block, records (a run of 1,000 permutations), the partial
 * results of one plain launch, and one pair of index arrays. */
constexpr size_t kErrBytes = 256, kCallRecords = 1025;
constexpr size_t kRoomPart = kErrBytes + kCallRecords * sizeof(dto_record);
constexpr size_t kRoomIdx = kRoomPart + kSplitItems * sizeof(dto::BestKey);
static_assert(kRoomPart % alignof(dto::BestKey) == 0, "partial results follow the records");

/* Byte offsets of a job's tables inside its device arena. */
struct ArenaOffsets {
  size_t bin1, bin2, join, joff, jpos, K, n, thr1, thr2, LF, D, H, A, B, err, ctr, stats;
};

/* The thread's stream-capture mode set to relaxed while in scope. */
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

/* A job: host tables plus their device copy (one HBM arena).  The arena is
 * the job's own allocation (`arena`), or, for a job created with
 * DTO_DEFER_UPLOAD and admitted by a server, a region of the server's pool
 * (`arena` stays NULL; the server owns the memory). */
struct dto_job {
  dto::HostJob h;
  dto::DevJob dev{};
  void *arena = nullptr;
  size_t arena_bytes = 0; /* size of the arena image */
  /* sizes of the job's own allocations, 0 where there is none; those of the
   * cut tables and partial results under cut_mu */
  size_t own_bytes = 0, ws_bytes = 0, cut_bytes = 0, partial_bytes = 0;
  bool resident = false;  /* dev points at an arena (own or pooled) */
  std::vector<unsigned char> image; /* the arena's contents (kept for deferred jobs) */
  ArenaOffsets off{};
  int *d_err = nullptr;
  uint32_t *d_ctr = nullptr; /* work counters of permutation launches, kCounterSlots */
  LaunchSlots slots;
  int device = -1;
  dto::LdsLayout lo_screen{}, lo_plain{}; /* lo_screen: a server's slices */
  dto::CutShape cut_sh{};
  dto::LdsLayout lo_cut{};
  /* the cut tables, set under cut_mu by the first screened launch; while
   * cut_pending, launches on other streams wait for cut_ev first */
  uint32_t *cut = nullptr;
  hipEvent_t cut_ev = nullptr;
  bool cut_pending = false;
  void *partial = nullptr; /* split plain launches' partial results, set under cut_mu */
  std::mutex cut_mu;
  uint16_t *ws = nullptr; /* global pair staging (only when the LDS cannot hold the pairs) */
  uint32_t ws_slots = 0;
  /* launches using ws run in order: each waits for the previous one's event */
  hipEvent_t ws_ev = nullptr;
  bool ws_used = false;
  std::mutex ws_mu;
  std::mutex call_mu; /* the arena's call room is in use */
  std::atomic<uint32_t> fail_alloc{0}; /* test hook: the n-th allocation from now on fails */
  /* The job's device allocations that later calls depend on.  Some are made
   * by a launch: while any thread captures a stream in global mode, hipMalloc
   * is refused to every thread (and may end that capture) unless the calling
   * one is in relaxed mode. */
  hipError_t alloc(void **p, size_t bytes) {
    if (fail_alloc && --fail_alloc == 0) return hipErrorOutOfMemory;
    RelaxedCapture relaxed;
    return hipMalloc(p, bytes);
  }
};
/* Tables, layouts and arena image of a job on the current device (no device
 * memory); then either its own arena (upload_job) or a caller's region
 * (bind_job, after the caller has copied j->image there). */
int prepare_job(dto_job *j);
int upload_job(dto_job *j);
void bind_job(dto_job *j, unsigned char *base);
/* Uploads a deferred job into its own arena on first use; fails when the
 * job sits in a server's pool (the server owns it). */
int ensure_resident(dto_job *j);
/* Launches that stage their pairs in the job's global buffer (lists too long
 * for the LDS) run one after another, whatever their streams: each waits for
 * the previous one's completion event.  Inside a stream capture the wait is
 * left out (a capture cannot wait on work recorded outside it), so captured
 * launches of one such job must not overlap. */
struct StagingOrder {
  dto_job *j;
  hipStream_t st;
  bool on = false;
  StagingOrder(const dto_job *job, const dto::LdsLayout &lo, hipStream_t s) : j(const_cast<dto_job *>(job)), st(s) {
    if (lo.pairs_in_lds || !j->ws_ev || stream_capturing(st)) return;
    j->ws_mu.lock();
    on = true;
    if (j->ws_used) (void)hipStreamWaitEvent(st, j->ws_ev, 0);
  }
  ~StagingOrder() {
    if (!on) return;
    if (hipEventRecord(j->ws_ev, st) == hipSuccess) j->ws_used = true;
    j->ws_mu.unlock();
  }
};

namespace dto {
/* The debug grid of one permutation on a stream (k_grid_counts then
 * k_grid_pvalues): overlap counts into kcnt (T1 * T2 words), every cell's
 * record into out; an out-of-range permutation index sets *err. */
hipError_t launch_grid(dto_job *job, const uint32_t *d1, const uint32_t *d2, uint32_t *kcnt, dto_record *out, int *err,
                       hipStream_t st);
/* A job's cut tables for work on stream st: built there if it has none yet,
 * and st waits where another stream still builds them.  *out is NULL where
 * the device has no memory for them. */
int cut_tables(dto_job *j, hipStream_t st, const uint32_t **out);
hipError_t launch_cut(dto_job *j, const uint32_t *cut, bool expl, uint32_t grid, hipStream_t st, const uint32_t *i1, const uint32_t *i2,
                      uint64_t n_perm, uint64_t base, uint64_t seed, uint32_t job_id, int32_t permuted, uint32_t lead,
                      dto_record *out);
/* part: the caller's room for the partial results (kSplitItems), or NULL for
 * a slot of the job's own buffer. */
hipError_t launch_plain(dto_job *j, bool expl, uint32_t max_grid, hipStream_t st, const uint32_t *i1,
                        const uint32_t *i2, uint64_t n_perm, uint64_t base, uint64_t seed, uint32_t job_id,
                        int32_t permuted, dto_record *out, BestKey *part);
struct BatchJob;
struct WorkItem;
hipError_t launch_batch_cut(const CutShape &sh, uint32_t grid, hipStream_t st, const BatchJob *jobs,
                            const WorkItem *items, uint32_t n_items, uint64_t seed, uint32_t *counter, int *err,
                            uint16_t *ws, uint32_t ws_stride);
}  // namespace dto
