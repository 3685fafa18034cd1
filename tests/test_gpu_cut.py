"""The cut-table kernels (screened mode) against the plain kernel, which
evaluates every cell: records equal in every field, p-value bits and tie
counts included, at the edges of the column segments, of the workgroup shapes
and builds, and on lists whose minimum is weak (several passes), tiny
(underflow) or tied."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lists(n, kind, seed):
    rng = np.random.default_rng(seed)
    ids = ["g%d" % i for i in range(n)]
    r = np.arange(1, n + 1, dtype=np.uint32)
    if kind == "reversed":  # every cell at or below its mean: no small p at all
        order = np.arange(n)[::-1]
    elif kind == "same":
        order = np.arange(n)
    else:
        order = rng.permutation(n)
    return ids, r, [ids[o] for o in order], r.copy()


def _compare(job, perms, seed, explicit):
    idx = (None, None)
    if explicit:
        rng = np.random.default_rng(seed)
        idx = tuple(np.stack([rng.permutation(m) for _ in range(perms)]).astype(np.uint32)
                    for m in (job.len1, job.len2))
    got, gp = job.run(perms, seed=seed, idx1=idx[0], idx2=idx[1])
    want, wp = job.run(perms, seed=seed, idx1=idx[0], idx2=idx[1], mode="plain")
    assert bytes(got) == bytes(want)
    assert gp.tobytes() == wp.tobytes()


@pytest.mark.parametrize("t2", [1, 2, 11, 12, 13, 767, 768, 769, 1537])
@pytest.mark.parametrize("kind", ["random", "reversed", "same"])
def test_column_segments(dto, gpu, t2, kind):
    n = 3200
    job = dto.Job.from_lists(*_lists(n, kind, t2))
    job.set_thresholds(np.arange(1, 34, dtype=np.uint32) * (n // 33), np.arange(1, t2 + 1, dtype=np.uint32) * (n // t2))
    _compare(job, 5, 3, explicit=False)
    job.close()


# with the 60 thresholds set here: 512 threads with pairs in registers to 15,248
# entries, in LDS to 19,280, 1,024 with pairs in registers to 31,136, in LDS to
# 39,264, in global memory above (the edges themselves: test_gpu_shapes.py)
@pytest.mark.parametrize("n", [1, 2, 5, 63, 65, 13500, 13900, 16300, 16500, 20900, 23500, 32700, 33100, 41000])
@pytest.mark.parametrize("explicit", [False, True])
def test_shapes(dto, gpu, n, explicit):
    job = dto.Job.from_lists(*_lists(n, "random", n))
    if n > 100:
        thr = np.unique(np.geomspace(1, n, 60).astype(np.uint32))
        job.set_thresholds(thr, thr)
    _compare(job, 3, 5, explicit)
    job.close()


def test_repeated_ids(dto, gpu):
    ids1, r1, ids2, r2 = _lists(5000, "random", 9)
    for q in range(0, 400, 2):
        ids2[q + 1] = ids2[q]
        ids1[3 * q + 1] = ids1[3 * q]
    job = dto.Job.with_population(ids1, r1, ids2, r2, 5200)
    _compare(job, 6, 2, explicit=True)
    job.close()
