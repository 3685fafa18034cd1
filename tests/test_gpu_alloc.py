"""Device allocations that fail, and calls after them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lists(n, seed=1):
    rng = np.random.default_rng(seed)
    ids = ["g%d" % i for i in range(n)]
    r = np.arange(1, n + 1, dtype=np.uint32)
    return ids, r, [ids[o] for o in rng.permutation(n)], r.copy()


def _fail_alloc(dto, job, n):
    dto._lib.check(dto._lib.lib().dto_internal_fail_alloc(job.handle, n))


@pytest.mark.parametrize("nth", [1, 2])
def test_upload_fails_then_succeeds(dto, gpu, nth):
    """N = 36,000: an upload allocates the pair staging and the tables.  Where
    either fails the call fails, and the next one uploads again (a job taken
    for resident without its staging would write through a null pointer)."""
    want = dto.Job.from_lists(*_lists(36000))
    job = dto.Job.from_lists(*_lists(36000), defer_upload=True)
    _fail_alloc(dto, job, nth)
    with pytest.raises(dto._lib.DtoError):
        job.optimize()
    assert job.optimize() == want.optimize()
    assert job.optimize(mode="plain") == want.optimize(mode="plain")
    job.close()
    want.close()


def _same(a, b):
    return bytes(a[0]) == bytes(b[0]) and a[1].tobytes() == b[1].tobytes()


@pytest.mark.parametrize("n", [50, 3000, 24000])
def test_no_memory_for_cut_tables(dto, gpu, n):
    """Screened calls of a job whose cut tables found no memory: the same
    records, and tables again once there is memory."""
    want = dto.Job.from_lists(*_lists(n))
    P = 4
    rng = np.random.default_rng(n)
    idx = dict(idx1=np.stack([rng.permutation(n) for _ in range(P)]), idx2=np.stack([rng.permutation(n) for _ in range(P)]))
    for call in (lambda j: j.run(P, seed=7), lambda j: j.run(P, **idx)):
        job = dto.Job.from_lists(*_lists(n))
        _fail_alloc(dto, job, 1)
        assert _same(call(job), call(want))
        assert _same(call(job), call(want))
        job.close()
    job = dto.Job.from_lists(*_lists(n))
    _fail_alloc(dto, job, 1)
    assert job.optimize() == want.optimize()
    job.close()
    want.close()


# the first-term kernels' shapes: table and bins in LDS, table in LDS, table
# global with the pairs in LDS, all global
@pytest.mark.parametrize("n", [1500, 22000, 27000, 36000])
def test_batch_without_cut_tables(dto, gpu, n):
    """A batch with one job whose cut tables found no memory."""
    sizes, perms = [300, n, 40], [5, 3, 9]
    res = []
    for nth in (0, 1):
        jobs = [dto.Job.from_lists(*_lists(m)) for m in sizes]
        _fail_alloc(dto, jobs[1], nth)
        b = dto.Batch(jobs, perms, seed=6)
        for rep in range(2):
            b.launch()
            res.append([bytes(r) for r in b.results()])
            if nth:
                b.autotune()
        b.close()
        for j in jobs:
            j.close()
    assert all(r == res[0] for r in res)


@pytest.mark.parametrize("nth", [2, 3])
def test_creation_needs_no_cut_tables(dto, gpu, nth):
    """An upload at this size makes one allocation.  The next are, from the
    first screened call on, the cut tables and, from the first asynchronous
    plain launch on, the partial results: calls that can do without them do."""
    import torch
    job = dto.Job.from_lists(*_lists(3000), defer_upload=True)
    _fail_alloc(dto, job, nth)
    want = dto.Job.from_lists(*_lists(3000))
    assert job.optimize(mode="plain") == want.optimize(mode="plain")
    assert job.process_threshold_pairs().tobytes() == want.process_threshold_pairs().tobytes()
    assert job.optimize() == want.optimize()
    rec = torch.zeros(2, 5 * 72, dtype=torch.uint8, device="cuda:0")
    for j, r in zip((job, want), rec):
        j.run_device(5, r.data_ptr(), seed=2, mode="plain")
    torch.cuda.synchronize()
    assert torch.equal(rec[0], rec[1])
    job.close()
    want.close()


def test_plain_call_allocates_nothing(dto, gpu):
    """A plain call that fits the job's call room needs no memory of its own."""
    job = dto.Job.from_lists(*_lists(200))
    held = job.device_bytes
    job.optimize(mode="plain")
    job.run(20, seed=1, mode="plain")
    assert job.device_bytes == held
    job.close()


@pytest.mark.parametrize("n", [900, 20000])
def test_first_launches_on_two_streams(dto, gpu, n):
    """The first screened launch builds the tables on its stream; one right
    after it on another stream waits for them."""
    import torch
    P = 6
    want = dto.Job.from_lists(*_lists(n))
    w = torch.zeros(P * 72, dtype=torch.uint8, device="cuda:0")
    want.run_device(P, w.data_ptr(), seed=3)
    torch.cuda.synchronize()
    for _ in range(3):
        job = dto.Job.from_lists(*_lists(n))
        outs, streams = [torch.zeros_like(w) for _ in range(3)], [torch.cuda.Stream() for _ in range(3)]
        torch.cuda.synchronize()
        for o, st in zip(outs, streams):
            job.run_device(P, o.data_ptr(), seed=3, stream=st.cuda_stream)
        torch.cuda.synchronize()
        assert all(torch.equal(o, w) for o in outs)
        job.close()
    want.close()


def test_device_bytes_counts_every_allocation(dto, gpu):
    """The footprint a job reports: the tables alone before the upload, then
    what the upload and the first launch of each mode allocate."""
    import torch
    n = 36000
    job = dto.Job.from_lists(*_lists(n), defer_upload=True)
    deferred = job.device_bytes
    seen = [deferred]
    out = torch.zeros(72, dtype=torch.uint8, device="cuda:0")
    for call in (lambda: job.process_threshold_pairs(), lambda: job.run_device(1, out.data_ptr(), mode="plain"),
                 lambda: job.optimize()):
        call()
        seen.append(job.device_bytes)
    torch.cuda.synchronize()
    assert seen == sorted(seen) and seen[1] > deferred + 2 * n * 1024  # staging: 1,024 slots of 16-bit rows
    assert seen[2] > seen[1]
    t1, t2 = job.n_thresholds1, job.n_thresholds2
    assert seen[3] - seen[2] > 14 * t1 * t2 * 2  # 14 levels of 16-bit counts
    job.set_thresholds(np.arange(1, 40), np.arange(1, 40))
    assert job.device_bytes < seen[2]
    job.close()
    assert job.device_bytes > 0
