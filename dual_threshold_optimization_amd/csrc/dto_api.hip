/*
 * C ABI of the DTO library (include/dto.h): device residency of jobs, kernel
 * launches, and the reference's run / empirical p-value / JSON steps.
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/dto.h"
#include "dto_host.hpp"
#include "dto_kernels.h"
#include "dto_internal.h"

namespace dto {
const char *last_error_cstr();
}

using namespace dto;



/* ------------------------------------------------------------------ */
/* devices                                                               */
/* ------------------------------------------------------------------ */
static std::mutex g_dev_mu;
static DevProps g_props[64];

int dto::current_device(int *dev) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) {
    (void)hipGetLastError();
    return fail(DTO_ERR_NO_DEVICE, "no HIP device available: the DTO kernels need an MI355X (gfx950)");
  }
  HIP_TRY(hipGetDevice(dev));
  return DTO_OK;
}

int dto::device_props(int dev, DevProps *out) {
  std::lock_guard<std::mutex> g(g_dev_mu);
  if (dev < 0 || dev >= 64) return fail(DTO_ERR_DEVICE, "device id out of range");
  if (!g_props[dev].ok) {
    hipDeviceProp_t p;
    HIP_TRY(hipGetDeviceProperties(&p, dev));
    g_props[dev].cus = p.multiProcessorCount;
    g_props[dev].lds_per_block = p.sharedMemPerBlock;
    g_props[dev].ok = 1;
  }
  *out = g_props[dev];
  return DTO_OK;
}

/* ------------------------------------------------------------------ */
/* job                                                                   */
/* ------------------------------------------------------------------ */
static uint32_t align16(uint32_t x) { return (x + 15u) & ~15u; }

LdsLayout dto::make_layout(const HostJob &h, int W, bool with_h, size_t lds_limit, bool nb_lds) {
  LdsLayout L{};
  const uint32_t N1 = (uint32_t)h.l1.ids.size(), N2 = (uint32_t)h.l2.ids.size();
  const uint32_t T1 = (uint32_t)h.thr1.size(), T2 = (uint32_t)h.thr2.size();
  const uint32_t T2w = (T2 + 1) / 2;
  L.T2w_pad = (T2w + 4u) & ~3u; /* at least one zero padding word */
  /* the screen table (or, without it, the pair staging) sits at offset 0 so
   * that table reads address it with the scaled index alone */
  /* pairs: u32 (row << 16 | column) where they alias the screen table, else the row alone as a u16 */
  const uint32_t hb = with_h ? 4u * (uint32_t)(h.N + 1) : 0u, pb = (with_h ? 4u : 2u) * std::max(N2, 1u);
  uint32_t fixed = 0;
  auto region = [&](uint32_t &field, uint32_t bytes) {
    field = fixed;
    fixed = align16(fixed + bytes);
  };
  region(L.nb, nb_lds ? 2u * std::max(std::max(N1, N2), 1u) : 0u);
  L.nb_in_lds = nb_lds ? 1u : 0u;
  region(L.rowstart, 4u * (T1 + 1));
  /* cursor is used while building the rows, cand0 in the reverse sweep */
  region(L.cursor, std::max(4u * T1, 8u * (uint32_t)W * (uint32_t)kCand0Cap));
  L.cand0 = L.cursor;
  region(L.cw, 4u * (uint32_t)W * L.T2w_pad);
  region(L.rowmin, 4u * T1);
  region(L.coln, 4u * T2);
  region(L.colb, 4u * T2);
  region(L.cand, 8u * (uint32_t)W * (uint32_t)kCandCap);
  region(L.cand3, 16u * (uint32_t)W * (uint32_t)kCand3Cap);
  region(L.exptab, 8u * 256u);
  region(L.red, (16u + 3u * (uint32_t)sizeof(BestKey) + 16u) * (uint32_t)W);
  region(L.misc, 16u);
  uint32_t base = 0;
  L.h = L.pairs = 0;
  if (with_h) {
    L.h_in_lds = 1;
    L.pairs_in_lds = 1;
    base = align16(std::max(hb, pb));
  } else if (align16(pb) + fixed <= lds_limit) {
    L.h_in_lds = 0;
    L.pairs_in_lds = 1;
    base = align16(pb);
  } else {
    L.h_in_lds = 0;
    L.pairs_in_lds = 0;
  }
  for (uint32_t *f : {&L.nb, &L.rowstart, &L.cursor, &L.cw, &L.rowmin, &L.coln, &L.colb, &L.cand, &L.cand3,
                      &L.exptab, &L.red, &L.misc})
    *f += base;
  L.cand0 = L.cursor;
  L.total = base + fixed;
  /* the batch kernel keeps its work item in the largest layout's misc slot,
   * which must therefore end the layout */
  if (L.misc + 16u != L.total) abort();
  return L;
}

template <typename T>
static size_t put(std::vector<unsigned char> &buf, const std::vector<T> &v) {
  size_t off = (buf.size() + 255) & ~(size_t)255;
  buf.resize(off + std::max<size_t>(v.size() * sizeof(T), 4));
  if (!v.empty()) memcpy(buf.data() + off, v.data(), v.size() * sizeof(T));
  return off;
}

LdsLayout dto::screen_layout(const HostJob &h, int W, size_t lim) {
  LdsLayout L = make_layout(h, W, true, lim, true);
  if (L.total <= lim) return L;
  L = make_layout(h, W, true, lim, false);
  if (L.total <= lim) return L;
  return make_layout(h, W, false, lim, true);
}

int prepare_job(dto_job *j) {
  int dev;
  int rc = current_device(&dev);
  if (rc) return rc;
  DevProps pr;
  if ((rc = device_props(dev, &pr))) return rc;
  const HostJob &h = j->h;
  /* LDS: keep the screen table resident when it fits */
  const size_t lim = pr.lds_per_block;
  LdsLayout without_h = make_layout(h, kNT / 64, false, lim);
  if (without_h.total > lim)
    return fail(DTO_ERR_TOO_LARGE, "job needs " + std::to_string(without_h.total) + " B of LDS per workgroup, device has " +
                                       std::to_string(lim));
  j->lo_plain = without_h;
  j->lo_screen = screen_layout(h, kNT / 64, lim);
  const HostJob *hp = &h;
  if ((rc = cut_shape(&hp, 1, lim, &j->cut_sh))) return rc;
  (void)cut_layout(h, j->cut_sh.nt / 64, j->cut_sh.build, &j->lo_cut);
  if (j->cut) (void)hipFree(j->cut);
  j->cut = nullptr;
  j->cut_bytes = 0;
  j->cut_pending = false;
  std::vector<unsigned char> &buf = j->image;
  buf.clear();
  ArenaOffsets &o = j->off;
  o.bin1 = put(buf, h.bin1);
  o.bin2 = put(buf, h.bin2);
  o.join = put(buf, h.join);
  o.joff = put(buf, h.join_off);
  o.jpos = put(buf, h.join_pos);
  o.K = put(buf, h.K);
  o.n = put(buf, h.n);
  o.thr1 = put(buf, h.thr1);
  o.thr2 = put(buf, h.thr2);
  o.LF = put(buf, h.LF);
  o.D = put(buf, h.D);
  o.H = put(buf, h.H32);
  o.A = put(buf, h.A32);
  o.B = put(buf, h.B32);
  o.err = put(buf, std::vector<int>(4, 0));
  o.ctr = put(buf, std::vector<uint32_t>(kCounterSlots, 0));
  o.stats = put(buf, std::vector<unsigned long long>(16, 0));
  buf.resize((buf.size() + 255) & ~(size_t)255);
  j->arena_bytes = buf.size();
  j->device = dev;
  DevJob &d = j->dev;
  d = DevJob{};
  d.N = (uint32_t)h.N;
  d.N1 = (uint32_t)h.l1.ids.size();
  d.N2 = (uint32_t)h.l2.ids.size();
  d.T1 = (uint32_t)h.thr1.size();
  d.T2 = (uint32_t)h.thr2.size();
  d.T2w = (d.T2 + 1) / 2;
  d.dup = h.dup ? 1u : 0u;
  d.kle = h.kle ? 1u : 0u;
  d.margin = h.margin;
  cut_levels(h, d);
  return DTO_OK;
}

void bind_job(dto_job *j, unsigned char *b) {
  const ArenaOffsets &o = j->off;
  DevJob &d = j->dev;
  d.bin1 = (const uint16_t *)(b + o.bin1);
  d.bin2 = (const uint16_t *)(b + o.bin2);
  d.join = (const int32_t *)(b + o.join);
  d.join_off = (const uint32_t *)(b + o.joff);
  d.join_pos = (const uint32_t *)(b + o.jpos);
  d.K = (const uint32_t *)(b + o.K);
  d.n = (const uint32_t *)(b + o.n);
  d.thr1 = (const uint32_t *)(b + o.thr1);
  d.thr2 = (const uint32_t *)(b + o.thr2);
  d.LF = (const double *)(b + o.LF);
  d.D = (const double *)(b + o.D);
  d.H32 = (const float *)(b + o.H);
  d.A32 = (const float *)(b + o.A);
  d.B32 = (const float *)(b + o.B);
  j->d_err = (int *)(b + o.err);
  j->d_ctr = (uint32_t *)(b + o.ctr);
  d.stats = (unsigned long long *)(b + o.stats);
  j->resident = true;
}

int upload_job(dto_job *j) {
  int rc = prepare_job(j);
  if (rc) return rc;
  DevProps pr;
  if ((rc = device_props(j->device, &pr))) return rc;
  if (j->arena) (void)hipFree(j->arena);
  if (j->ws) (void)hipFree(j->ws);
  j->arena = nullptr;
  j->ws = nullptr;
  j->own_bytes = j->ws_bytes = 0;
  j->resident = false;
  /* global pair staging for layouts whose pairs do not fit in LDS; before the
   * job is resident, so that no launch finds it missing */
  j->ws_slots = (uint32_t)pr.cus * 4u;
  if (!j->lo_plain.pairs_in_lds || !j->lo_cut.pairs_in_lds) {
    const size_t ws_bytes = (size_t)j->ws_slots * std::max<uint32_t>(j->dev.N2, 1) * sizeof(uint16_t);
    HIP_TRY(j->alloc((void **)&j->ws, ws_bytes));
    j->ws_bytes = ws_bytes;
    if (!j->ws_ev) HIP_TRY(hipEventCreateWithFlags(&j->ws_ev, hipEventDisableTiming));
  }
  /* after the tables: the room of a small call, which then needs no
   * allocation of its own; one copy brings its error word and records back */
  const size_t tables = j->image.size();
  j->image.resize(tables + kErrBytes, 0);
  const size_t own_bytes = tables + kRoomIdx + ((size_t)j->dev.N1 + j->dev.N2) * sizeof(uint32_t);
  HIP_TRY(j->alloc(&j->arena, own_bytes));
  j->own_bytes = own_bytes;
  HIP_TRY(hipMemcpy(j->arena, j->image.data(), j->image.size(), hipMemcpyHostToDevice));
  bind_job(j, (unsigned char *)j->arena);
  j->d_err = (int *)((unsigned char *)j->arena + tables);
  std::vector<unsigned char>().swap(j->image); /* the device copy is the job's now */
  return DTO_OK;
}

int ensure_resident(dto_job *j) {
  if (j->resident) return DTO_OK;
  return upload_job(j);
}

/* ------------------------------------------------------------------ */
/* launches                                                              */
/* ------------------------------------------------------------------ */
/* Number of workgroups for a permutation launch: enough to fill every CU at
 * the occupancy the LDS footprint allows, never more than the work. */
static uint32_t perm_grid(const dto_job *j, const LdsLayout &lo, uint64_t n_perm, uint64_t max_per_cu) {
  DevProps pr;
  if (device_props(j->device, &pr)) return 1;
  uint64_t per_cu = std::max<uint64_t>(1, pr.lds_per_block ? (160u * 1024u) / std::max<uint32_t>(lo.total, 1) : 1);
  per_cu = std::min<uint64_t>(per_cu, max_per_cu);
  uint64_t g = std::min<uint64_t>(n_perm, (uint64_t)pr.cus * per_cu);
  if (!lo.pairs_in_lds) g = std::min<uint64_t>(g, j->ws_slots); /* one global slot per workgroup */
  return (uint32_t)std::max<uint64_t>(g, 1);
}

/* lead = 1: the unpermuted task runs first, in the same launch, into record 0
 * (screened mode with drawn permutations only).  part: see launch_plain. */
static int launch_perms(dto_job *j, uint32_t mode, bool expl, const uint32_t *d1, const uint32_t *d2, uint64_t n_perm,
                        uint64_t base, uint64_t seed, uint32_t job_id, int32_t permuted, dto_record *d_out,
                        hipStream_t st, uint32_t lead = 0, BestKey *part = nullptr) {
  if (n_perm + lead == 0) return DTO_OK;
  if (n_perm >= (1ull << 32) - 65536ull) return fail(DTO_ERR_TOO_LARGE, "too many permutations in one launch");
  hipError_t e;
  if (mode == DTO_MODE_PLAIN) {
    /* at most one workgroup per staging slot */
    const uint32_t g = perm_grid(j, j->lo_plain, ~0ull, 4);
    e = launch_plain(j, expl, g, st, d1, d2, n_perm, base, seed, job_id, permuted, d_out, part);
  } else if (mode == DTO_MODE_SCREENED) {
    const uint32_t *cut = nullptr;
    int rc = cut_tables(j, st, &cut);
    if (rc) return rc;
    if (!cut) {
      /* no memory for the tables: the plain kernels give the same records */
      if (lead && (rc = launch_perms(j, DTO_MODE_PLAIN, true, nullptr, nullptr, 1, 0, 0, 0, 0, d_out, st, 0, part)))
        return rc;
      return launch_perms(j, DTO_MODE_PLAIN, expl, d1, d2, n_perm, base, seed, job_id, permuted, d_out + lead, st, 0,
                          part);
    }
    const uint32_t g = perm_grid(j, j->lo_cut, n_perm + lead, j->cut_sh.nt == 512 ? 4 : 2);
    e = launch_cut(j, cut, expl, g, st, d1, d2, n_perm, base, seed, job_id, permuted, lead, d_out);
  } else {
    return fail(DTO_ERR_INVALID_ARGUMENT, "unknown mode");
  }
  if (e != hipSuccess) return fail(DTO_ERR_DEVICE, std::string("kernel launch: ") + hipGetErrorString(e));
  return DTO_OK;
}

static int check_err_flag(dto_job *j) {
  int h[1] = {0};
  HIP_TRY(hipMemcpy(h, j->d_err, sizeof(int), hipMemcpyDeviceToHost));
  if (h[0]) {
    int z = 0;
    HIP_TRY(hipMemcpy(j->d_err, &z, sizeof(int), hipMemcpyHostToDevice));
    if (h[0] & 2) return fail(DTO_ERR_DEVICE, "internal error: a permutation selected no grid cell");
    return fail(DTO_ERR_BAD_PERMUTATION, "a permutation index is out of range");
  }
  return DTO_OK;
}

struct DevBuf {
  void *p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
};

/* Device room for one call's records (and, for a single explicit pair, its
 * index arrays; for plain launches, their partial results): the job's own
 * where it is free and large enough, else allocated for the call. */
struct CallRoom {
  dto_job *j;
  std::unique_lock<std::mutex> own;
  DevBuf tmp;
  dto_record *rec = nullptr;
  uint32_t *idx = nullptr;
  BestKey *part = nullptr;
  size_t records = 0;
  explicit CallRoom(dto_job *job) : j(job) {}
  int open(size_t n, bool with_idx) {
    records = n;
    const size_t rec_b = n * sizeof(dto_record);
    if (j->arena && n <= kCallRecords) {
      own = std::unique_lock<std::mutex>(j->call_mu, std::try_to_lock);
      if (own.owns_lock()) {
        unsigned char *const room = (unsigned char *)j->d_err;
        rec = (dto_record *)(room + kErrBytes);
        part = (BestKey *)(room + kRoomPart);
        idx = (uint32_t *)(room + kRoomIdx);
        return DTO_OK;
      }
    }
    const size_t idx_b = with_idx ? ((size_t)j->dev.N1 + j->dev.N2) * sizeof(uint32_t) : 0;
    HIP_TRY(hipMalloc(&tmp.p, rec_b + idx_b));
    rec = (dto_record *)tmp.p;
    idx = (uint32_t *)((unsigned char *)tmp.p + rec_b);
    return DTO_OK;
  }
  /* Waits for the launches of this call and brings its records back. */
  int fetch(std::vector<unsigned char> &buf, const dto_record **out) {
    const size_t rec_b = records * sizeof(dto_record);
    buf.resize(kErrBytes + rec_b);
    *out = (const dto_record *)(buf.data() + kErrBytes);
    if (!own.owns_lock()) {
      HIP_TRY(hipMemcpy(buf.data() + kErrBytes, rec, rec_b, hipMemcpyDeviceToHost));
      return check_err_flag(j);
    }
    HIP_TRY(hipMemcpy(buf.data(), j->d_err, kErrBytes + rec_b, hipMemcpyDeviceToHost));
    int err;
    memcpy(&err, buf.data(), sizeof err);
    return err ? check_err_flag(j) : DTO_OK;
  }
};

/* explicit permutations must be permutations of [0, len) */
static int validate_perms(const uint32_t *idx, uint64_t P, uint64_t len) {
  if (!idx) return DTO_OK;
  std::vector<uint8_t> stamp(len, 0); /* the last of 255 rounds of rows that held the value */
  for (uint64_t p = 0; p < P; ++p) {
    const uint32_t *row = idx + p * len;
    const uint8_t mark = (uint8_t)(p % 255u + 1u);
    if (p && mark == 1u) std::fill(stamp.begin(), stamp.end(), (uint8_t)0);
    for (uint64_t k = 0; k < len; ++k) {
      uint32_t v = row[k];
      if (v >= len || stamp[v] == mark)
        return fail(DTO_ERR_BAD_PERMUTATION, "permutation " + std::to_string(p) + " is not a permutation of [0, " +
                                                 std::to_string(len) + ")");
      stamp[v] = mark;
    }
  }
  return DTO_OK;
}


/* ------------------------------------------------------------------ */
/* C ABI                                                                  */
/* ------------------------------------------------------------------ */
extern "C" {

const char *dto_last_error(void) { return dto::last_error_cstr(); }

int dto_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return n;
}

double dto_fdr(uint64_t l1, uint64_t l2, uint64_t overlap, uint64_t population, double sensitivity) {
  /* fdr.rs:29-60; where the reference panics (sensitivity <= 0, fdr.rs:36-39)
   * the result is NaN and dto_last_error() holds the panic message */
  if (sensitivity <= 0.0) {
    fail(DTO_ERR_INVALID_ARGUMENT, "Sensitivity must be greater than 0.");
    return __builtin_nan("");
  }
  double df = fmax((double)overlap / sensitivity, 0.0);
  double b = fmax((double)l1 - df, 0.0);
  double r = fmax((double)l2 - df, 0.0);
  double num = b * r;
  double den = (double)population * (double)overlap;
  return den > 0.0 ? num / den : 0.0;
}

int dto_fdr_checked(uint64_t l1, uint64_t l2, uint64_t overlap, uint64_t population, double sensitivity,
                    double *out) {
  if (!out) return fail(DTO_ERR_INVALID_ARGUMENT, "null output");
  if (sensitivity <= 0.0) return fail(DTO_ERR_INVALID_ARGUMENT, "Sensitivity must be greater than 0.");
  *out = dto_fdr(l1, l2, overlap, population, sensitivity);
  return DTO_OK;
}

uint32_t dto_generate_thresholds(uint32_t max_rank, uint32_t *out, uint32_t cap) {
  std::vector<uint32_t> t = generate_thresholds(max_rank);
  if (out)
    for (uint32_t i = 0; i < cap && i < t.size(); ++i) out[i] = t[i];
  return (uint32_t)t.size();
}

int dto_ln_factorial_table(uint64_t n_max, double *out) {
  if (!out) return fail(DTO_ERR_INVALID_ARGUMENT, "null output");
  for (uint64_t x = 0; x <= n_max; ++x) out[x] = ln_factorial(x);
  return DTO_OK;
}

int dto_hypergeometric_pvalue(const uint64_t *N, const uint64_t *K, const uint64_t *n, const uint64_t *k,
                              uint64_t count, double *out) {
  if (count == 0) return DTO_OK;
  if (!N || !K || !n || !k || !out) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  uint64_t maxN = 0;
  for (uint64_t c = 0; c < count; ++c) {
    /* Hypergeometric::new(N, K, n).expect(...) */
    if (K[c] > N[c] || n[c] > N[c]) return fail(DTO_ERR_HYPERGEOMETRIC, "Failed to create hypergeometric distribution");
    if (N[c] >= (1ull << 31)) return fail(DTO_ERR_TOO_LARGE, "population size too large");
    maxN = std::max(maxN, N[c]);
  }
  int dev, rc;
  if ((rc = current_device(&dev))) return rc;
  std::vector<double> LF(maxN + 1);
  for (uint64_t x = 0; x <= maxN; ++x) LF[x] = ln_factorial(x);
  DevBuf dLF, dq, dout;
  HIP_TRY(hipMalloc(&dLF.p, LF.size() * 8));
  HIP_TRY(hipMalloc(&dq.p, count * 8 * 4));
  HIP_TRY(hipMalloc(&dout.p, count * 8));
  uint64_t *q = (uint64_t *)dq.p;
  HIP_TRY(hipMemcpy(dLF.p, LF.data(), LF.size() * 8, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(q, N, count * 8, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(q + count, K, count * 8, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(q + 2 * count, n, count * 8, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(q + 3 * count, k, count * 8, hipMemcpyHostToDevice));
  uint32_t g = (uint32_t)std::min<uint64_t>((count + 255) / 256, 4096);
  hipLaunchKernelGGL(k_hypergeom, dim3(g), dim3(256), 0, 0, (const double *)dLF.p, q, q + count, q + 2 * count,
                     q + 3 * count, count, (double *)dout.p);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpy(out, dout.p, count * 8, hipMemcpyDeviceToHost));
  return DTO_OK;
}

/* internal test hooks (not in dto.h): device exp and device shuffle */
int dto_internal_exp(const double *x, uint64_t count, double *out) {
  int dev, rc;
  if ((rc = current_device(&dev))) return rc;
  DevBuf dx, dy;
  HIP_TRY(hipMalloc(&dx.p, count * 8));
  HIP_TRY(hipMalloc(&dy.p, count * 8));
  HIP_TRY(hipMemcpy(dx.p, x, count * 8, hipMemcpyHostToDevice));
  uint32_t g = (uint32_t)std::min<uint64_t>((count + 255) / 256, 8192);
  hipLaunchKernelGGL(k_exp, dim3(g), dim3(256), 0, 0, (const double *)dx.p, count, (double *)dy.p);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpy(out, dy.p, count * 8, hipMemcpyDeviceToHost));
  return DTO_OK;
}

int dto_internal_exp_host(const double *x, uint64_t count, double *out) {
  static const uint64_t tab[256] = DTO_EXP_TAB_INIT;
  for (uint64_t c = 0; c < count; ++c) out[c] = dto_exp(x[c], tab);
  return DTO_OK;
}

/* one Philox4x32-10 block (host), for the published known-answer vectors */
int dto_internal_philox(const uint32_t *ctr, const uint32_t *key, uint32_t *out) {
  if (!ctr || !key || !out) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  U32x4 c;
  c.x = ctr[0];
  c.y = ctr[1];
  c.z = ctr[2];
  c.w = ctr[3];
  const U32x4 r = philox4x32_10(c, key[0], key[1]);
  out[0] = r.x;
  out[1] = r.y;
  out[2] = r.z;
  out[3] = r.w;
  return DTO_OK;
}

int dto_internal_shuffle_device(uint64_t seed, uint32_t job, uint32_t perm, uint32_t list, uint32_t n, uint32_t *out) {
  int dev, rc;
  if ((rc = current_device(&dev))) return rc;
  DevBuf d;
  HIP_TRY(hipMalloc(&d.p, std::max<uint32_t>(n, 1) * 4));
  hipLaunchKernelGGL(k_shuffle, dim3(1), dim3(256), 0, 0, seed, job, perm, list, n, (uint32_t *)d.p);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpy(out, d.p, (size_t)n * 4, hipMemcpyDeviceToHost));
  return DTO_OK;
}

/* work counters of a job's screened launches (test / profiling hook, not in
 * dto.h), 16 values: exact cells, exact terms, passes, cycles of the build /
 * column counts / sweep / list flushes / what follows the sweep, cells past
 * the first-term test, tier-2 survivors, tier-2 flushes, 0, listed cells; in a
 * server's slices what the first-term screen counts in their places
 * (WaveStats) */
int dto_internal_stats(dto_job *job, uint64_t *out, int reset) {
  if (!job || !out) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  if (!DTO_STATS) return fail(DTO_ERR_INVALID_ARGUMENT, "the library was built without DTO_STATS (make STATS=1)");
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(out, job->dev.stats, 16 * sizeof(uint64_t), hipMemcpyDeviceToHost));
  if (reset) HIP_TRY(hipMemset(job->dev.stats, 0, 16 * sizeof(uint64_t)));
  return DTO_OK;
}

/* test hook (not in dto.h): the counter slots of n launches, captured[i] of
 * them captured, in order */
int dto_internal_launch_slots(const int32_t *captured, uint32_t n, uint32_t *out) {
  if (!captured || !out) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  LaunchSlots s;
  for (uint32_t i = 0; i < n; ++i) out[i] = s.take(captured[i] != 0);
  return DTO_OK;
}

/* test hook (not in dto.h): threads and build of the job's screened launches */
int dto_internal_cut_shape(const dto_job *job, int32_t *nt, int32_t *build) {
  if (!job || !nt || !build) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  *nt = job->cut_sh.nt;
  *build = job->cut_sh.build;
  return DTO_OK;
}

/* test hook (not in dto.h): the n-th device allocation of the job from now on
 * fails (0: none does) */
int dto_internal_fail_alloc(dto_job *job, uint32_t n) {
  if (!job) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  job->fail_alloc = n;
  return DTO_OK;
}

int dto_philox_permutation(uint64_t seed, uint32_t job_id, uint32_t perm, uint32_t list, uint32_t len, uint32_t *out) {
  if (!out && len) return fail(DTO_ERR_INVALID_ARGUMENT, "null output");
  Shuffle s = shuffle_make(seed, job_id, perm, list, len);
  shuffle_fill(s, out);
  return DTO_OK;
}

int dto_job_create(const char *const *ids1, const uint32_t *ranks1, uint64_t n1, const char *const *ids2,
                   const uint32_t *ranks2, uint64_t n2, const char *const *bg, uint64_t nbg, uint32_t flags,
                   dto_job **out) {
  if (!out) return fail(DTO_ERR_INVALID_ARGUMENT, "null output");
  *out = nullptr;
  dto_job *j = new dto_job();
  int rc = build_host_job(ids1, ranks1, n1, ids2, ranks2, n2, bg, nbg, flags & ~DTO_DEFER_UPLOAD, j->h);
  if (!rc) rc = (flags & DTO_DEFER_UPLOAD) ? prepare_job(j) : upload_job(j);
  if (rc) {
    dto_job_destroy(j);
    return rc;
  }
  *out = j;
  return DTO_OK;
}

int dto_job_create_with_population(const char *const *ids1, const uint32_t *ranks1, uint64_t n1,
                                   const char *const *ids2, const uint32_t *ranks2, uint64_t n2,
                                   uint64_t population_size, dto_job **out) {
  if (!out) return fail(DTO_ERR_INVALID_ARGUMENT, "null output");
  *out = nullptr;
  dto_job *j = new dto_job();
  int rc = build_host_job_with_population(ids1, ranks1, n1, ids2, ranks2, n2, population_size, j->h);
  if (!rc) rc = upload_job(j);
  if (rc) {
    dto_job_destroy(j);
    return rc;
  }
  *out = j;
  return DTO_OK;
}

int dto_job_create_from_files(const char *path1, const char *path2, const char *bg_path, uint32_t flags,
                              dto_job **out) {
  std::vector<std::string> i1, i2, ib;
  std::vector<uint32_t> r1, r2;
  int rc;
  if ((rc = read_ranked_csv(path1, i1, r1))) return rc;
  if ((rc = read_ranked_csv(path2, i2, r2))) return rc;
  if (bg_path && (rc = read_feature_lines(bg_path, ib))) return rc;
  std::vector<const char *> p1, p2, pb;
  for (auto &s : i1) p1.push_back(s.c_str());
  for (auto &s : i2) p2.push_back(s.c_str());
  for (auto &s : ib) pb.push_back(s.c_str());
  static const char *empty_bg[1] = {""};
  const char *const *bgp = bg_path ? (pb.empty() ? empty_bg : pb.data()) : nullptr;
  return dto_job_create(p1.data(), r1.data(), i1.size(), p2.data(), r2.data(), i2.size(), bgp, pb.size(), flags, out);
}

int dto_job_set_thresholds(dto_job *job, const uint32_t *thr1, uint32_t t1, const uint32_t *thr2, uint32_t t2) {
  if (!job || (t1 && !thr1) || (t2 && !thr2)) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  if (job->resident && !job->arena) return fail(DTO_ERR_INVALID_ARGUMENT, "the job belongs to a server");
  const bool own = job->resident;
  HostJob saved = job->h;
  job->h.thr1.assign(thr1, thr1 + t1);
  job->h.thr2.assign(thr2, thr2 + t2);
  int rc = job->h.derive();
  if (!rc) rc = own ? upload_job(job) : prepare_job(job);
  if (rc) {
    std::string msg = dto_last_error();
    job->h = saved;
    (void)(own ? upload_job(job) : prepare_job(job));
    return fail(rc, msg);
  }
  return DTO_OK;
}

int dto_job_info_get(const dto_job *job, dto_job_info *info) {
  if (!job || !info) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  info->population_size = job->h.N;
  info->len1 = job->h.l1.ids.size();
  info->len2 = job->h.l2.ids.size();
  info->n_thresholds1 = (uint32_t)job->h.thr1.size();
  info->n_thresholds2 = (uint32_t)job->h.thr2.size();
  info->dropped1 = job->h.dropped1;
  info->dropped2 = job->h.dropped2;
  std::lock_guard<std::mutex> g(const_cast<dto_job *>(job)->cut_mu);
  /* a job without an arena of its own: what it takes of a server's pool */
  info->device_bytes = (job->own_bytes ? job->own_bytes : job->arena_bytes) + job->ws_bytes + job->cut_bytes +
                       job->partial_bytes;
  return DTO_OK;
}

int dto_job_thresholds(const dto_job *job, int list, uint32_t *out, uint32_t cap) {
  if (!job || (list != 1 && list != 2)) return -fail(DTO_ERR_INVALID_ARGUMENT, "bad job or list");
  const std::vector<uint32_t> &t = list == 1 ? job->h.thr1 : job->h.thr2;
  if (out)
    for (uint32_t i = 0; i < cap && i < t.size(); ++i) out[i] = t[i];
  return (int)t.size();
}

void dto_job_destroy(dto_job *job) {
  if (!job) return;
  if (job->arena) (void)hipFree(job->arena);
  if (job->ws) (void)hipFree(job->ws);
  if (job->cut) (void)hipFree(job->cut);
  if (job->partial) (void)hipFree(job->partial);
  if (job->ws_ev) (void)hipEventDestroy(job->ws_ev);
  if (job->cut_ev) (void)hipEventDestroy(job->cut_ev);
  delete job;
}

int dto_run_device(dto_job *job, uint64_t n_perm, uint64_t perm_base, uint64_t seed, const uint32_t *d_idx1,
                   const uint32_t *d_idx2, uint32_t mode, dto_record *d_out, void *stream) {
  if (!job || (!d_out && n_perm)) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  int rc;
  if ((rc = ensure_resident(job))) return rc;
  bool expl = d_idx1 || d_idx2;
  return launch_perms(job, mode, expl, d_idx1, d_idx2, n_perm, perm_base, seed, 0, 1, d_out, (hipStream_t)stream);
}

int dto_optimize(dto_job *job, const uint32_t *idx1, const uint32_t *idx2, uint32_t mode, dto_record *out) {
  if (!job || !out) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  int rc;
  if ((rc = ensure_resident(job))) return rc;
  if ((rc = validate_perms(idx1, 1, job->dev.N1)) || (rc = validate_perms(idx2, 1, job->dev.N2))) return rc;
  const size_t n1 = job->dev.N1, n2 = job->dev.N2;
  CallRoom room(job);
  if ((rc = room.open(1, true))) return rc;
  uint32_t *d1 = idx1 ? room.idx : nullptr, *d2 = idx2 ? room.idx + n1 : nullptr;
  if (idx1 && idx2) {
    std::vector<uint32_t> both(n1 + n2);
    memcpy(both.data(), idx1, n1 * 4);
    memcpy(both.data() + n1, idx2, n2 * 4);
    HIP_TRY(hipMemcpy(d1, both.data(), (n1 + n2) * 4, hipMemcpyHostToDevice));
  } else if (idx1) {
    HIP_TRY(hipMemcpy(d1, idx1, n1 * 4, hipMemcpyHostToDevice));
  } else if (idx2) {
    HIP_TRY(hipMemcpy(d2, idx2, n2 * 4, hipMemcpyHostToDevice));
  }
  int32_t permuted = (idx1 || idx2) ? 1 : 0;
  if ((rc = launch_perms(job, mode, true, d1, d2, 1, 0, 0, 0, permuted, room.rec, 0, 0, room.part))) return rc;
  std::vector<unsigned char> buf;
  const dto_record *rec = nullptr;
  if ((rc = room.fetch(buf, &rec))) return rc;
  *out = *rec;
  return DTO_OK;
}

int dto_process_threshold_pairs(dto_job *job, const uint32_t *idx1, const uint32_t *idx2, dto_record *out) {
  if (!job || !out) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  int rc;
  if ((rc = ensure_resident(job))) return rc;
  if ((rc = validate_perms(idx1, 1, job->dev.N1)) || (rc = validate_perms(idx2, 1, job->dev.N2))) return rc;
  const size_t n1 = job->dev.N1, n2 = job->dev.N2, cells = (size_t)job->dev.T1 * job->dev.T2;
  DevBuf di, dk, dr;
  HIP_TRY(hipMalloc(&di.p, (n1 + n2 + 2) * 4));
  HIP_TRY(hipMalloc(&dk.p, cells * 4));
  HIP_TRY(hipMalloc(&dr.p, cells * sizeof(dto_record)));
  uint32_t *d1 = nullptr, *d2 = nullptr;
  if (idx1) {
    d1 = (uint32_t *)di.p;
    HIP_TRY(hipMemcpy(d1, idx1, n1 * 4, hipMemcpyHostToDevice));
  }
  if (idx2) {
    d2 = (uint32_t *)di.p + n1 + 1;
    HIP_TRY(hipMemcpy(d2, idx2, n2 * 4, hipMemcpyHostToDevice));
  }
  HIP_TRY(launch_grid(job, d1, d2, (uint32_t *)dk.p, (dto_record *)dr.p, job->d_err, 0));
  HIP_TRY(hipMemcpy(out, dr.p, cells * sizeof(dto_record), hipMemcpyDeviceToHost));
  return check_err_flag(job);
}


int dto_empirical_pvalue(const dto_record *unpermuted, const dto_record *perm, uint64_t n_perm, dto_result *result) {
  if (!unpermuted || !result || (n_perm && !perm)) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  /* empirical_pvalue.rs:136-173 */
  result->unpermuted = *unpermuted;
  result->fdr = dto_fdr(unpermuted->set1_len, unpermuted->set2_len, unpermuted->intersection_size,
                        unpermuted->population_size, 0.8);
  result->n_permutations = n_perm;
  uint64_t le = 0;
  for (uint64_t p = 0; p < n_perm; ++p) le += perm[p].pvalue <= unpermuted->pvalue;
  result->n_le = le;
  result->empirical_pvalue = n_perm ? (double)le / (double)n_perm : 1.0;
  return DTO_OK;
}

int dto_run(dto_job *job, uint64_t n_perm, uint64_t seed, const uint32_t *idx1, const uint32_t *idx2, uint32_t mode,
            dto_result *result, dto_record *perm_out) {
  if (!job || !result) return fail(DTO_ERR_INVALID_ARGUMENT, "null pointer");
  if ((idx1 == nullptr) != (idx2 == nullptr))
    return fail(DTO_ERR_INVALID_ARGUMENT, "give explicit permutations for both lists or neither");
  int rc;
  if ((rc = ensure_resident(job))) return rc;
  const uint64_t n1 = job->dev.N1, n2 = job->dev.N2;
  if ((rc = validate_perms(idx1, n_perm, n1)) || (rc = validate_perms(idx2, n_perm, n2))) return rc;
  CallRoom room(job);
  if ((rc = room.open(n_perm + 1, false))) return rc;
  dto_record *d_rec = room.rec;
  /* task 0: unpermuted (main.rs:122-125); with drawn permutations it joins
   * their launch, where it costs no workgroup's latency of its own */
  const uint32_t lead = mode == DTO_MODE_SCREENED && n_perm && !idx1 ? 1 : 0;
  if (!lead && (rc = launch_perms(job, mode, true, nullptr, nullptr, 1, 0, 0, 0, 0, d_rec, 0, 0, room.part))) return rc;
  if (n_perm) {
    if (idx1) {
      /* explicit permutations, streamed in chunks of at most ~512 MiB */
      uint64_t chunk = std::max<uint64_t>(1, (512ull << 20) / ((n1 + n2) * 4));
      chunk = std::min(chunk, n_perm);
      DevBuf di;
      HIP_TRY(hipMalloc(&di.p, chunk * (n1 + n2) * 4));
      uint32_t *d1 = (uint32_t *)di.p, *d2 = d1 + chunk * n1;
      for (uint64_t p0 = 0; p0 < n_perm; p0 += chunk) {
        uint64_t c = std::min(chunk, n_perm - p0);
        HIP_TRY(hipMemcpy(d1, idx1 + p0 * n1, c * n1 * 4, hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(d2, idx2 + p0 * n2, c * n2 * 4, hipMemcpyHostToDevice));
        if ((rc = launch_perms(job, mode, true, d1, d2, c, p0, seed, 0, 1, d_rec + 1 + p0, 0, 0, room.part))) return rc;
        HIP_TRY(hipDeviceSynchronize());
      }
    } else {
      if ((rc = launch_perms(job, mode, false, nullptr, nullptr, n_perm, 0, seed, 0, 1, d_rec + 1 - lead, 0, lead,
                             room.part)))
        return rc;
    }
  }
  std::vector<unsigned char> buf;
  const dto_record *rec = nullptr;
  if ((rc = room.fetch(buf, &rec))) return rc;
  if (perm_out && n_perm) memcpy(perm_out, rec + 1, n_perm * sizeof(dto_record));
  return dto_empirical_pvalue(&rec[0], rec + 1, n_perm, result);
}

int dto_result_json(const dto_result *result, char *buf, size_t cap) {
  if (!result) return -1;
  std::string s = result_json(*result);
  if (!buf || cap < s.size() + 1) return -1;
  memcpy(buf, s.c_str(), s.size() + 1);
  return (int)s.size();
}

}  // extern "C"
