"""Launches beside and inside stream captures."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REC = 72


def _job(dto, n, seed=1):
    rng = np.random.default_rng(seed)
    ids = ["g%d" % i for i in range(n)]
    r = np.arange(1, n + 1, dtype=np.uint32)
    return dto.Job.from_lists(ids, r, [ids[o] for o in rng.permutation(n)], r.copy())


def _records(torch, perms):
    return torch.zeros(perms * REC, dtype=torch.uint8, device="cuda:0")


@pytest.mark.parametrize("mode", ["screened", "plain"])
@pytest.mark.parametrize("inside", [False, True])
def test_first_launch_during_a_global_capture(dto, gpu, mode, inside):
    """A job's first launch of a mode may allocate.  Made while a stream is
    captured in global mode, on that stream or on another one, it leaves the
    capture whole, and its records are those of an ordinary launch."""
    import torch
    P, n = 7, 900
    ref = _job(dto, n)  # loads the kernels
    want = _records(torch, P)
    ref.run_device(P, want.data_ptr(), seed=3, mode=mode)
    job, got, x = _job(dto, n), _records(torch, P), torch.zeros(1000, device="cuda:0")
    other, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, capture_error_mode="global"):
        x += 1
        st = torch.cuda.current_stream() if inside else other
        job.run_device(P, got.data_ptr(), seed=3, mode=mode, stream=st.cuda_stream)
        x += 1
    for rep in range(1, 4):
        if inside:
            got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want), rep
        assert bool((x == 2 * rep).all()), rep
        ref.run_device(P, want.data_ptr(), seed=3, mode=mode)  # eager work between replays
        torch.cuda.synchronize()
    job.close()
    ref.close()


@pytest.mark.parametrize("mode", ["screened", "plain"])
def test_replay_among_many_ordinary_launches(dto, gpu, mode):
    """A captured launch replayed while ordinary launches of the same job, more
    than the ring of counters has slots, run on another stream."""
    import torch
    P, n = 100, 2000
    job = _job(dto, n)
    want, got = _records(torch, P), _records(torch, P)
    one_want, one = _records(torch, 1), _records(torch, 300)
    job.run_device(P, want.data_ptr(), seed=3, mode=mode)
    job.run_device(1, one_want.data_ptr(), seed=9, mode=mode)
    other, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        job.run_device(P, got.data_ptr(), seed=3, mode=mode, stream=torch.cuda.current_stream().cuda_stream)
    for _ in range(2):
        got.zero_()
        one.zero_()
        torch.cuda.synchronize()
        for q in range(300):
            if q % 30 == 0:
                graph.replay()
            job.run_device(1, one.data_ptr() + q * REC, seed=9, mode=mode, stream=other.cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        assert torch.equal(one.view(300, REC), one_want.expand(300, REC))
    job.close()
