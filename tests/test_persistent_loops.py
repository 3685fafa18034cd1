"""The persistent kernels' loops, read from their source.  In a loop whose
iteration ends with a block that only thread 0 runs and begins with another
one, the compiler may join the two, and the other lanes of thread 0's wave then
pass the barrier after the claim ahead of it.  A barrier between the blocks, for
the wave or the workgroup, keeps them apart, so every such kernel needs one
after its record is written."""
import os
import re

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "dual_threshold_optimization_amd", "csrc")


def _kernels():
    """(name, body) of every kernel that claims work from a counter and writes records."""
    out = []
    for f in sorted(os.listdir(CSRC)):
        if not f.endswith((".h", ".hip")):
            continue
        text = re.sub(r"/\*.*?\*/", "", open(os.path.join(CSRC, f)).read(), flags=re.S)
        for m in re.finditer(r"__global__[^;{]*?\b(k_\w+)\([^{]*\{", text):
            depth, i = 1, m.end()
            while depth:
                depth += {"{": 1, "}": -1}.get(text[i], 0)
                i += 1
            body = text[m.end():i]
            if "write_record(" in body and re.search(r"atomicAdd\(counter\b|&s_next\b|\bcounter, &", body):
                out.append((m.group(1), body))
    return out


def test_every_persistent_kernel_is_found():
    assert {n for n, _ in _kernels()} == {"k_cut", "k_batch_cut", "k_batch", "k_plain"}


@pytest.mark.parametrize("name,body", _kernels(), ids=lambda v: v if isinstance(v, str) and v.isidentifier() else "")
def test_barrier_after_thread_0_record(name, body):
    after = body[body.rindex("write_record("):]
    end = after.index(";") + 1
    # what follows in the iteration: up to the closing braces of the loops
    assert re.match(r"\s*\}?\s*(wave_sync|__syncthreads)\(\)", after[end:]), (name, after[end:end + 60])
