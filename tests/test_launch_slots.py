"""Which launches of a job may share a work counter and partial results."""
import ctypes

import numpy as np


def _slots(dto, captured):
    c = np.ascontiguousarray(captured, dtype=np.int32)
    out = np.zeros(len(c), dtype=np.uint32)
    dto._lib.check(dto._lib.lib().dto_internal_launch_slots(c.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)), len(c),
                                                            dto._lib.u32p(out)))
    return out


def test_captured_launches_keep_their_slots_to_themselves(dto):
    captured = np.zeros(2000, dtype=np.int32)
    captured[::50] = 1  # 40 captures among ordinary launches that wrap their ring several times
    s = _slots(dto, captured)
    assert not set(s[captured == 1]) & set(s[captured == 0])
    assert len(set(s[captured == 1])) == 40
    ordinary = s[captured == 0]
    for k in range(0, len(ordinary) - 256, 97):  # any 256 in flight are apart
        assert len(set(ordinary[k:k + 256])) == 256
    assert s.max() < 256 + 64
