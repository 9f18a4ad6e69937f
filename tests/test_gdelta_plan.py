"""Workspace of the chunked gated delta rule: bounded however many segments a pass holds (the library's host code)."""
from __future__ import annotations

import ctypes

import pytest


@pytest.fixture(scope="module")
def size():
    from vinf_3080ti_amd import _lib

    lib = _lib.load()

    def f(rows, key_heads=16, value_heads=48, kd=128, vd=128):
        flat = [v for i, n in enumerate(rows) for v in (i, 0, n, 0)]
        return lib.vq_gated_delta_seg_workspace_bytes((ctypes.c_int32 * len(flat))(*flat), len(rows), key_heads,
                                                      value_heads, kd, vd)

    return f


@pytest.mark.parametrize("vh,vd", [(48, 128), (32, 128), (4, 64), (64, 32)])
@pytest.mark.parametrize("n", [1, 2, 4, 5, 9, 16, 33, 64])
@pytest.mark.parametrize("rows", [24, 64, 512, 8192])
def test_workspace_is_bounded(size, vh, vd, n, rows):
    """32 MiB of chunk operands and, where a segment takes several launches, the group's fp32 states beside them."""
    slot, chunks = vh * 2304 * 4, -(-rows // 32)
    need = size([rows] * n, 4, vh, 128, vd)
    assert slot * min(chunks, 16) <= need <= (32 << 20) + (16 << 20)
    assert need <= n * (slot * min(chunks, 16) + vh * 128 * vd * 4)


def test_workspace_follows_the_long_segments(size):
    assert size([23] * 64) == 0 and size([1, 8, 23]) == 0
    assert size([24]) == size([23, 24, 5]) > 0
    assert size([40, 600, 24]) == size([600, 40, 24]) >= size([600])
    assert size([512], kd=64) == size([512], vd=48) == size([512], vd=160) == 0
