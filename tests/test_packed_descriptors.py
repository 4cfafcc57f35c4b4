"""The packed descriptors (one buffer per call) hold what the ctypes
structures hold, for every form of tensor a caller may pass."""

from __future__ import annotations

import pytest
import torch


@pytest.mark.parametrize("make", [
    lambda: torch.zeros(3), lambda: torch.zeros(()), lambda: torch.zeros(0, 4, dtype=torch.bfloat16),
    lambda: torch.zeros(2, 3, 4, 5, dtype=torch.float16), lambda: torch.zeros(1, 2, 3, 4, 5),
    lambda: torch.zeros(4, 6).t()[1:], lambda: torch.zeros(2, dtype=torch.int64), lambda: torch.zeros(8, dtype=torch.int32)[3:],
])
def test_packed_descriptors_match_structures(make):
    from nanovllm_amd import _lib

    t = make()
    buf, at = _lib.pack(t, None, t)
    assert at[1] is None and at[2] - at[0] == 2 * _lib._ITEM_BYTES
    for address in (at[0], at[2]):
        got, want = _lib.NvdsaTensor.from_address(address), _lib.describe(t)
        for field, _ in _lib.NvdsaTensor._fields_:
            a, b = getattr(got, field), getattr(want, field)
            assert (list(a) == list(b)) if field == "shape" else a == b, field
    with pytest.raises(IndexError):
        _lib.pack(*[t] * (_lib._MAX_PACKED + 1))
    del buf
