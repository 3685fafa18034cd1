"""The work a user has this framework do, as cases that can be timed and compared.

A case is a dict of plain values: `kind` says which public entry point runs it, the
rest are sizes and options.  The ranges: lists of 30 (the README example) to 41,000
features, reference thresholds or dense custom grids, 1 to 10,000 permutations, drawn
on the device or given, the screened and the plain mode, duplicate ids, batches of
uneven jobs, and the full grid export.

    listed()             the listed cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  lists, resident jobs, permutations and output buffers
    run(state)           one pass through the public entry points, and its outputs
    work(case)           bytes and operations one pass cannot do without
    exact(case, seed)    p-values of the same inputs from plain torch in 64 bits

Records come back as their 64-bit words (threshold values, set sizes, overlap, the bits
of the p-value, flags, tie counts), next to the p-values as floats.
"""
import math

import numpy as np
import torch

import dual_threshold_optimization_amd as dto
from dual_threshold_optimization_amd import _lib
from dual_threshold_optimization_amd import workloads as W

RECORD_BYTES = 72
RECORD_WORDS = RECORD_BYTES // 8
P_WORD = 6  # the p-value's word in a record


def listed():
    return [
        # The README example through the CLI's run: 30 features, 1,000 permutations.  The
        # smallest job a user runs, all latency.
        {"name": "run_readme_30", "kind": "run", "n": 30, "extras": 0, "planted": 0, "ties": 0.1, "perms": 1000},
        # One optimize() call on genome-sized lists, as a program that steps through list
        # pairs makes it: one task, host in and out.
        {"name": "optimize_20k", "kind": "optimize", "n": 20000, "extras": 2000, "planted": 600, "ties": 0.1,
         "permuted": True},
        # An ordinary yeast-sized run at the CLI's default of 1,000 permutations.
        {"name": "run_6k", "kind": "run", "n": 6000, "extras": 0, "planted": 200, "ties": 0.05, "perms": 1000},
        # The same with ids that repeat in list 2 (probes of one gene), which joins them to
        # the same feature of list 1.
        {"name": "run_dup_6k", "kind": "run", "n": 6007, "extras": 0, "planted": 200, "ties": 0.05, "perms": 1000,
         "dup": 150},
        # The genome-scale job with explicit permutations resident on the GPU: the headline.
        {"name": "explicit_20k", "kind": "device", "n": 20000, "extras": 2000, "planted": 600, "ties": 0.1,
         "perms": 10000, "explicit": True},
        # The genome-scale job as the CLI runs it with -p 10000, permutations drawn on the GPU.
        {"name": "run_20k", "kind": "run", "n": 20000, "extras": 2000, "planted": 600, "ties": 0.1, "perms": 10000},
        # A transcript-level list, of a ragged length.
        {"name": "device_27k", "kind": "device", "n": 27431, "extras": 2000, "planted": 800, "ties": 0.1,
         "perms": 1500, "explicit": False},
        # Long lists, whose tables are the largest.
        {"name": "device_41k", "kind": "device", "n": 40961, "extras": 2000, "planted": 1200, "ties": 0.1,
         "perms": 1000, "explicit": False},
        # A dense custom grid: 2,000 thresholds on both lists, 4M cells a permutation.
        {"name": "dense_2k", "kind": "device", "n": 20000, "extras": 2000, "planted": 600, "ties": 0.1, "perms": 700,
         "explicit": False, "step": 10},
        # The plain mode, which a user takes to check the screened one: every cell exact.
        {"name": "plain_6k", "kind": "device", "n": 6000, "extras": 0, "planted": 200, "ties": 0.05, "perms": 48,
         "explicit": True, "mode": "plain"},
        # Many uneven jobs in one persistent launch.
        {"name": "batch_32", "kind": "batch", "jobs": 32, "n_min": 2000, "n_max": 20000, "perms": 400},
        # The full record grid of one permutation (debug output) on the caller's buffers.
        {"name": "grid_20k", "kind": "grid", "n": 20000, "extras": 2000, "planted": 600, "ties": 0.1,
         "permuted": True},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes over the logarithm of their ranges, permutation counts bounded
    by the work of the largest listed case."""
    kind = rng.choice(["run", "run", "device", "device", "device", "optimize", "batch", "grid"])
    if kind == "batch":
        n_max = _log_uniform(rng, 3000, 20000)
        return {"kind": "batch", "jobs": rng.randint(4, 40), "n_min": rng.randint(500, n_max // 2), "n_max": n_max,
                "perms": _log_uniform(rng, 30, 300)}
    n = _log_uniform(rng, 25 if kind == "run" else 500, 41000)
    case = {"kind": kind, "n": n, "extras": rng.choice([0, 0, rng.randint(1, max(1, n // 10))]),
            "planted": rng.randint(0, max(1, n // 20)), "ties": rng.choice([0.0, 0.05, 0.1, 0.3])}
    if kind in ("optimize", "grid"):
        case["permuted"] = rng.random() < 0.5
        return case
    case["perms"] = _log_uniform(rng, 50, 4000)
    if kind == "run":
        if rng.random() < 0.2:
            case["dup"] = max(1, n // rng.randint(20, 200))
        return case
    case["explicit"] = rng.random() < 0.5
    if rng.random() < 0.15:
        case["mode"] = "plain"
        case["n"] = min(n, 6000)
        case["extras"] = min(case["extras"], case["n"] // 10)
        case["planted"] = min(case["planted"], case["n"] // 20)
        case["perms"] = rng.randint(8, 40)
    elif rng.random() < 0.25:
        case["n"] = n = min(n, 30000)
        case["extras"] = min(case["extras"], n // 10)
        case["planted"] = min(case["planted"], n // 20)
        case["step"] = max(1, n // rng.randint(300, 2000))
        case["perms"] = max(30, min(case["perms"], int(2.5e9) // (n // case["step"]) ** 2))
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _lists(case, seed):
    n, planted = case["n"], case["planted"]
    top1, top2 = max(n // 10, planted, 1), max(3 * n // 40, planted, 1)
    ids1, r1, ids2, r2, bg = W.planted_lists(n, planted, top1, top2, case["ties"], seed, extras=case["extras"])
    if case.get("dup"):
        rng = np.random.default_rng(seed + 77)
        for q in rng.choice(len(ids2) - 1, size=case["dup"], replace=False):
            ids2[q + 1] = ids2[q]
    return ids1, r1, ids2, r2, bg


def _population(case):
    return case["n"] + (50 if case.get("dup") else 0)


def _job(case, seed):
    ids1, r1, ids2, r2, bg = _lists(case, seed)
    if case.get("dup"):  # lists that differ in their ids come with the caller's population size
        return dto.Job.with_population(ids1, r1, ids2, r2, _population(case))
    job = dto.Job.from_lists(ids1, r1, ids2, r2, background=bg, drop_outside_background=bg is not None)
    if case.get("step"):
        thr = _step_thresholds(case)
        job.set_thresholds(thr, thr)
    return job


def _step_thresholds(case):
    return np.arange(case["step"], case["n"] + 1, case["step"], dtype=np.uint32)


def _host_perm(length, seed):
    return np.random.default_rng(seed).permutation(length).astype(np.uint32)


def _device_perms(perms, length, seed):
    """perms seeded permutations of [0, length) on the GPU; row 0 is the identity (task 0 of
    a run is the unpermuted one)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    out = torch.empty((perms, length), dtype=torch.int32, device="cuda")
    step = max(1, (64 << 20) // length)
    for p0 in range(0, perms, step):
        p1 = min(perms, p0 + step)
        out[p0:p1] = torch.argsort(torch.rand(p1 - p0, length, device="cuda", generator=gen), dim=1)
    out[0] = torch.arange(length, dtype=torch.int32, device="cuda")
    return out


def _device_records(count):
    """A buffer of `count` records: its words, and its p-values as a view of them."""
    words = torch.zeros((count, RECORD_WORDS), dtype=torch.int64, device="cuda")
    return words, words.view(torch.float64)[:, P_WORD]


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind, "case": case, "seed": seed}
    if kind == "batch":
        specs = W.batch_jobs(n_jobs=case["jobs"], seed=seed, n_min=case["n_min"], n_max=case["n_max"])
        jobs = [dto.Job.from_lists(a, b, c, d) for a, b, c, d, _ in specs]
        state["batch"] = dto.Batch(jobs, [case["perms"]] * len(jobs), seed=seed)
        return state
    job = state["job"] = _job(case, seed)
    if kind == "optimize":
        state["idx"] = (_host_perm(job.len1, seed + 1), _host_perm(job.len2, seed + 2)) if case["permuted"] else (None, None)
    elif kind == "device":
        state["mode"] = case.get("mode", "screened")
        if case["explicit"]:
            state["tasks"] = case["perms"] + 1
            state["idx"] = (_device_perms(state["tasks"], job.len1, seed + 1),
                            _device_perms(state["tasks"], job.len2, seed + 2))
        else:
            state["tasks"] = case["perms"]
        state["out"], state["pvalue"] = _device_records(state["tasks"])
    elif kind == "grid":
        state["out"], state["pvalue"] = _device_records(job.n_thresholds1 * job.n_thresholds2)
        state["idx"] = ()
        if case["permuted"]:
            state["idx"] = tuple(torch.from_numpy(_host_perm(n, seed + s).astype(np.int32)).cuda()
                                 for s, n in ((1, job.len1), (2, job.len2)))
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _result(res):
    """A run's result: its words, then p-value, empirical p-value and FDR as floats."""
    return {"words": np.frombuffer(res, dtype=np.int64), "pvalue": res.unpermuted.pvalue,
            "empirical_pvalue": res.empirical_pvalue, "fdr": res.fdr}


def run(state):
    kind = state["kind"]
    if kind == "run":
        res, perm = state["job"].run(state["case"]["perms"], seed=state["seed"])
        words = perm.view(np.int64).reshape(-1, RECORD_WORDS)
        return {"result": _result(res), "records": words, "pvalue": perm["pvalue"]}
    if kind == "optimize":
        r = state["job"].optimize(*state["idx"])
        return {"record": np.frombuffer(r.tobytes(), dtype=np.int64), "pvalue": float(r["pvalue"])}
    if kind == "batch":
        state["batch"].launch()
        results = state["batch"].results()
        return {"words": np.stack([np.frombuffer(r, dtype=np.int64) for r in results]),
                "pvalue": np.array([r.unpermuted.pvalue for r in results]),
                "empirical_pvalue": np.array([r.empirical_pvalue for r in results])}
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "grid":
        d1, d2 = (t.data_ptr() for t in state["idx"]) if state["idx"] else (None, None)
        _lib.check(_lib.lib().dto_process_threshold_pairs_noalloc(state["job"].handle, d1, d2, state["out"].data_ptr(),
                                                                  None, stream))
        return {"records": state["out"], "pvalue": state["pvalue"]}
    d1, d2 = (t.data_ptr() for t in state["idx"]) if "idx" in state else (None, None)
    state["job"].run_device(state["tasks"], state["out"].data_ptr(), seed=state["seed"], d_idx1=d1, d_idx2=d2,
                            mode=state["mode"], stream=stream)
    return {"records": state["out"], "pvalue": state["pvalue"]}


# ---------------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------------
def _n_thresholds(max_rank):
    t, count = 1, 0
    while t <= max_rank:
        count += 1
        t = int(math.floor(t * 1.01 + 1.0))
    return count


def _tasks_work(n, cells, tasks, explicit, every_cell_exact):
    """Per cell: two adds of the 2-D prefix count and one comparison with the best cell so
    far.  Where every cell's p-value is an output or the mode's definition, its tail as
    well: about 20 terms of 20 operations.  The job's tables (two bins of 2 bytes and a
    4-byte join an entry) are read once, index arrays once, a record written per task."""
    ops = cells * (403 if every_cell_exact else 3)
    return {"bytes": 8 * n + tasks * (RECORD_BYTES + (8 * n if explicit else 0)), "flops": tasks * ops}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        mean = math.exp(0.5 * (math.log(case["n_min"]) + math.log(case["n_max"])))
        one = _tasks_work(int(mean), _n_thresholds(int(mean)) ** 2, case["perms"] + 1, False, False)
        return {k: v * case["jobs"] for k, v in one.items()}
    n = case["n"]
    t = len(_step_thresholds(case)) if case.get("step") else _n_thresholds(n + case["extras"])
    if kind == "grid":
        one = _tasks_work(n, t * t, 1, case["permuted"], True)
        one["bytes"] += (t * t - 1) * RECORD_BYTES
        return one
    if kind == "optimize":
        return _tasks_work(n, t * t, 1, case["permuted"], False)
    explicit = case.get("explicit", False)
    tasks = case["perms"] + (1 if kind == "run" or explicit else 0)
    return _tasks_work(n, t * t, tasks, explicit, case.get("mode") == "plain")


# ---------------------------------------------------------------------------
# the same p-values in 64 bits
# ---------------------------------------------------------------------------
class _Reference:
    """Overlap grids and hypergeometric tails of one list pair, in float64 torch."""

    def __init__(self, case, seed):
        ids1, r1, ids2, r2, bg = _lists(case, seed)
        keep = set(bg) if bg is not None else None
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.N = _population(case)
        lists = []
        for ids, ranks in ((ids1, r1), (ids2, r2)):
            pairs = [(r, f) for f, r in zip(ids, ranks) if keep is None or f in keep]
            pairs.sort(key=lambda x: x[0])
            lists.append(pairs)
        bins = []
        for pairs in lists:
            ranks = np.array([r for r, _ in pairs])
            if case.get("step"):
                thr = _step_thresholds(case)
            else:
                thr, t = [], 1
                while t <= ranks[-1]:
                    thr.append(t)
                    t = int(math.floor(t * 1.01 + 1.0))
            bins.append((len(thr), torch.from_numpy(np.searchsorted(thr, ranks)).to(self.dev)))
        (self.T1, self.bin1), (self.T2, self.bin2) = bins
        where = {f: m for m, (_, f) in enumerate(lists[0])}
        self.join = torch.tensor([where.get(f, -1) for _, f in lists[1]], device=self.dev)
        size = [torch.bincount(b, minlength=t + 1)[:t].cumsum(0) for b, t in ((self.bin1, self.T1), (self.bin2, self.T2))]
        self.K, self.n = size[0][:, None].expand(self.T1, self.T2), size[1][None, :].expand(self.T1, self.T2)
        x = torch.arange(self.N + 1, dtype=torch.float64, device=self.dev)
        self.lf = torch.lgamma(x + 1.0)

    def overlaps(self, idx1, idx2):
        a = torch.empty_like(self.bin1)
        a[idx1] = self.bin1
        m = self.join[idx2]
        ok = m >= 0
        cell = a[m[ok]] * (self.T2 + 1) + self.bin2[ok]
        h = torch.bincount(cell, minlength=(self.T1 + 1) * (self.T2 + 1)).reshape(self.T1 + 1, self.T2 + 1)
        return h[:self.T1, :self.T2].cumsum(0).cumsum(1)

    def _log_term(self, K, n, k):
        lf, N = self.lf, self.N
        return (lf[K] - lf[k] - lf[K - k] + lf[N - K] - lf[n - k] - lf[N - K - n + k] - lf[N] + lf[n] + lf[N - n])

    def pvalues(self, K, n, k):
        """P(X >= k) of each (K, n, k): terms added upwards until none changes the sum."""
        lo, hi = (K + n - self.N).clamp(min=0), torch.minimum(K, n)
        p = torch.ones(k.shape, dtype=torch.float64, device=self.dev)
        p[k > hi] = 0.0
        at = torch.nonzero((k > lo) & (k <= hi))[:, 0]
        K, n, x, hi = K[at], n[at], k[at].clone(), hi[at]
        first = self._log_term(K, n, x)
        term, total = torch.ones_like(first), torch.ones_like(first)
        live = torch.arange(len(at), device=self.dev)
        Kf, nf, xf, hif = K.double(), n.double(), x.double(), hi.double()
        while len(live):
            for _ in range(32):
                r = (Kf - xf) * (nf - xf) / ((xf + 1) * (self.N - Kf - nf + xf + 1))
                term = term * r.clamp(min=0.0)
                total[live] += term
                xf = xf + 1
            on = (xf < hif) & ((term > total[live] * 1e-18) | (r >= 1.0))
            live, term, Kf, nf, xf, hif = live[on], term[on], Kf[on], nf[on], xf[on], hif[on]
        p[at] = (first + total.log()).exp().clamp(max=1.0)
        return p

    def minimum(self, idx1, idx2):
        """min over the grid: cells whose first term, a lower bound of the tail, lies above
        the smallest value the first bound's best cells reach are left out."""
        K, n, k = self.K.reshape(-1), self.n.reshape(-1), self.overlaps(idx1, idx2).reshape(-1)
        mean = K.double() * n.double() / self.N
        lo = (K + n - self.N).clamp(min=0)
        cand = torch.nonzero((k > lo) & (k <= torch.minimum(K, n)) & (k.double() > mean))[:, 0]
        if not len(cand):
            return float(self.pvalues(K, n, k).min())
        first = self._log_term(K[cand], n[cand], k[cand])
        best = cand[torch.topk(first, min(64, len(cand)), largest=False).indices]
        bound = self.pvalues(K[best], n[best], k[best]).min()
        cand = cand[first <= bound.log() + 1e-6]
        low = self.pvalues(K[cand], n[cand], k[cand]).min() if len(cand) else bound
        return float(torch.minimum(low, bound))


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch" or case.get("dup"):
        return None
    if kind == "device" and (not case["explicit"] or case["perms"] > 500):
        return None  # permutations drawn by the framework, or too many
    ref = _Reference(case, seed)
    len1, len2 = len(ref.bin1), len(ref.bin2)
    identity = (torch.arange(len1, device=ref.dev), torch.arange(len2, device=ref.dev))
    if kind == "run":
        return {"result": {"words": None, "pvalue": ref.minimum(*identity), "empirical_pvalue": None, "fdr": None},
                "records": None, "pvalue": None}
    if kind in ("optimize", "grid"):
        idx = identity
        if case["permuted"]:
            idx = tuple(torch.from_numpy(_host_perm(n, seed + s).astype(np.int64)).to(ref.dev)
                        for s, n in ((1, len1), (2, len2)))
        if kind == "optimize":
            return {"record": None, "pvalue": ref.minimum(*idx)}
        k = ref.overlaps(*idx)
        return {"records": None, "pvalue": ref.pvalues(ref.K.reshape(-1), ref.n.reshape(-1), k.reshape(-1))}
    i1, i2 = (_device_perms(case["perms"] + 1, n, seed + s).long() for s, n in ((1, len1), (2, len2)))
    p = [ref.minimum(i1[t], i2[t]) for t in range(case["perms"] + 1)]
    return {"records": None, "pvalue": torch.tensor(p, dtype=torch.float64)}
