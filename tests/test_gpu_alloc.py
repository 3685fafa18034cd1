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
