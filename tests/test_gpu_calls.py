"""Calls at the limits of what a job keeps for them, and calls side by side."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REC = 72


def _lists(n, seed):
    rng = np.random.default_rng(seed)
    ids = ["g%d" % i for i in range(n)]
    r = np.arange(1, n + 1, dtype=np.uint32)
    return ids, r, [ids[o] for o in rng.permutation(n)], r.copy()


def _device(torch, job, perms, seed, mode):
    out = torch.zeros(perms * REC, dtype=torch.uint8, device="cuda:0")
    job.run_device(perms, out.data_ptr(), seed=seed, mode=mode)
    torch.cuda.synchronize()
    return out.cpu().numpy().tobytes()


@pytest.mark.parametrize("mode", ["screened", "plain"])
@pytest.mark.parametrize("perms", [1, 1024, 1025, 1026])
def test_records_around_the_call_room(dto, gpu, perms, mode):
    """A job's call room holds 1,025 records: a run of 1,024 permutations."""
    import torch
    job = dto.Job.from_lists(*_lists(400, 2))
    _, rec = job.run(perms, seed=11, mode=mode)
    assert rec.tobytes() == _device(torch, job, perms, 11, mode)
    job.close()


@pytest.mark.parametrize("tasks", [1, 2, 63, 64, 65, 255, 256, 257, 513])
def test_plain_tasks_around_the_split(dto, gpu, tasks):
    """Plain launches of up to 256 tasks split each over several workgroups."""
    import torch
    job = dto.Job.from_lists(*_lists(700, 3))
    assert _device(torch, job, tasks, 4, "plain") == _device(torch, job, tasks, 4, "screened")
    job.close()


@pytest.mark.parametrize("t1", [1, 8, 9, 4000])
def test_plain_rows_around_the_split(dto, gpu, t1):
    """Fewer rows than one workgroup's waves, one more, and many times the parts."""
    import torch
    job = dto.Job.from_lists(*_lists(4000, 3))
    job.set_thresholds(np.arange(1, t1 + 1, dtype=np.uint32), np.arange(1, 41, dtype=np.uint32) * 100)
    for tasks in (1, 40):
        assert _device(torch, job, tasks, 4, "plain") == _device(torch, job, tasks, 4, "screened")
    job.close()


@pytest.mark.parametrize("mode", ["screened", "plain"])
def test_threads_on_one_job(dto, gpu, mode):
    """Calls of several threads on one job: one takes its call room, the others
    allocate their own.  The first ones also race for the job's first launch."""
    n, threads, calls = 900, 6, 12
    rng = np.random.default_rng(5)
    idx = [tuple(rng.permutation(n).astype(np.uint32) for _ in range(2)) for _ in range(threads)]
    ref = dto.Job.from_lists(*_lists(n, 6))
    one = [ref.optimize(*idx[t], mode=mode) for t in range(threads)]
    run = [ref.run(20, seed=t, mode=mode) for t in range(threads)]
    job, bad = dto.Job.from_lists(*_lists(n, 6)), []
    start = threading.Barrier(threads)

    def work(t):
        try:
            start.wait()
            for c in range(calls):
                if (t + c) % 2:
                    ok = job.optimize(*idx[t], mode=mode) == one[t]
                else:
                    a, b = job.run(20, seed=t, mode=mode)
                    ok = bytes(a) == bytes(run[t][0]) and b.tobytes() == run[t][1].tobytes()
                if not ok:
                    bad.append((t, c))
        except Exception as e:
            bad.append((t, repr(e)))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    job.close()
    ref.close()


@pytest.mark.parametrize("n,dup", [(300, 0), (800, 40), (14000, 0), (20000, 0), (33000, 0)])
def test_batch_of_mixed_builds(dto, gpu, n, dup):
    """A batch runs all its jobs in one shape, that of the most demanding one:
    the others' results do not depend on it, and the first job's are those of
    a run of its own (the same permutations)."""
    first = [dto.Job.from_lists(*_lists(m, m)) for m in (1500, 60)]
    ids1, r1, ids2, r2 = _lists(n, 8)
    for q in range(dup):  # a feature that list 1 repeats and list 2 names: no registers for its pairs
        ids1[2 * q + 1] = ids1[2 * q]
    jobs = first + [dto.Job.with_population(ids1, r1, ids2, r2, n)]
    alone = dto.Batch(first, [30, 25], seed=9)
    mixed = dto.Batch(jobs, [30, 25, 4], seed=9)
    for b in (alone, mixed):
        b.launch()
    a, m = [bytes(r) for r in alone.results()], [bytes(r) for r in mixed.results()]
    assert m[:2] == a
    assert m[0] == bytes(first[0].run(30, seed=9)[0])
    for b in (alone, mixed):
        b.close()
    for j in jobs:
        j.close()


@pytest.mark.parametrize("population", [(1 << 24) - 1, (1 << 24) + 1, (1 << 25) + 12345])
def test_populations_beyond_float_counts(dto, gpu, population):
    """Counts of the population that a float does not hold exactly."""
    n = 3000
    ids1, r1, ids2, r2 = _lists(n, 12)
    ids2 = ids2[: n // 2] + ["x%d" % i for i in range(n - n // 2)]
    job = dto.Job.with_population(ids1, r1, ids2, r2, population)
    got, gp = job.run(4, seed=2)
    want, wp = job.run(4, seed=2, mode="plain")
    assert bytes(got) == bytes(want) and gp.tobytes() == wp.tobytes()
    job.close()
