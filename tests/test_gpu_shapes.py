"""The screened kernels' workgroup shapes (threads, and how pairs are built), each
on both sides of the sizes where the next one takes over, against the plain
kernel."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GLOBAL, LDS, REGS = 0, 1, 2


def _lists(n, seed):
    rng = np.random.default_rng(seed)
    ids = ["g%d" % i for i in range(n)]
    r = np.arange(1, n + 1, dtype=np.uint32)
    return ids, r, [ids[o] for o in rng.permutation(n)], r.copy()


def _shape(dto, job):
    nt, build = ctypes.c_int32(), ctypes.c_int32()
    dto._lib.check(dto._lib.lib().dto_internal_cut_shape(job.handle, ctypes.byref(nt), ctypes.byref(build)))
    return nt.value, build.value


def _compare(job, perms, seed):
    rng = np.random.default_rng(seed)
    idx = [np.stack([rng.permutation(m) for _ in range(perms)]).astype(np.uint32) for m in (job.len1, job.len2)]
    for kw in (dict(), dict(idx1=idx[0], idx2=idx[1])):
        got, gp = job.run(perms, seed=seed, **kw)
        want, wp = job.run(perms, seed=seed, mode="plain", **kw)
        assert bytes(got) == bytes(want)
        assert gp.tobytes() == wp.tobytes()


@pytest.mark.parametrize("n,nt,build", [
    (12344, 512, REGS), (12345, 512, LDS), (15728, 512, LDS), (15729, 1024, REGS), (25576, 1024, REGS), (25577, 1024, LDS),
    (32888, 1024, LDS), (32889, 1024, GLOBAL), (49800, 1024, GLOBAL), (49801, 512, GLOBAL), (60000, 512, GLOBAL)])
def test_reference_thresholds(dto, gpu, n, nt, build):
    job = dto.Job.from_lists(*_lists(n, n))
    assert _shape(dto, job) == (nt, build)
    _compare(job, 2, 5)
    job.close()


@pytest.mark.parametrize("t,nt,build", [(1600, 512, REGS), (1601, 512, LDS), (1956, 512, LDS), (1957, 1024, REGS),
                                        (2572, 1024, REGS), (2573, 1024, LDS), (2872, 1024, LDS), (2873, 512, LDS),
                                        (3700, 512, LDS)])
def test_custom_grids(dto, gpu, t, nt, build):
    n = 6000
    job = dto.Job.from_lists(*_lists(n, t))
    thr = np.arange(1, t + 1, dtype=np.uint32)
    job.set_thresholds(thr, thr)
    assert _shape(dto, job) == (nt, build)
    _compare(job, 2, 6)
    job.close()
