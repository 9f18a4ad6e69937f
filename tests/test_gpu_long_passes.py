"""Prompt-length passes of the sequence ops: the kernels that split a long segment's rows over workgroups, at the edges
of their spans and chunks, against the float64 restatements in oracle/oracle.py."""
from __future__ import annotations

import numpy as np
import pytest

from vinf_3080ti_amd import GGUFTensorType as T

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vinf_3080ti_amd.runtime import HipWeightRuntime

    return HipWeightRuntime()


def put(rt, name: str, a, elem: int = 4) -> None:
    a = np.ascontiguousarray(a, np.float32 if elem == 4 else np.float16).reshape(-1)
    rt.alloc(name, a.size, elem)
    rt.write(name, a.tobytes())


def get(rt, name: str, shape) -> np.ndarray:
    return np.array(rt.read_floats(name), np.float64).reshape(shape)


def put_weight(rt, name: str, a) -> None:
    a = np.ascontiguousarray(a, np.float32).reshape(-1)
    rt.upload_raw(name, a.tobytes(), T.F32, a.size, 1)


def segments(rt, rows, slots):
    """A pass of len(rows) segments in slots taken backwards, the first row of the second one moved away from the end
    of the first (explicit row0). Returns (table, total buffer rows)."""
    rt.alloc("pt", 64)
    rt.set_paging("pt", 64, 64 // slots, slots)
    segs, row0 = [], 0
    for i, n in enumerate(rows):
        row0 += 3 if i == 1 else 0
        segs.append((slots - 1 - i, 0, n, row0))
        row0 += n
    return segs, rt.set_segments(segs)


# A span of the conv is 8 rows: one row, one span, a span and a row, several spans with a remainder, together.
@pytest.mark.parametrize("K,rows", [(1, (9,)), (4, (8, 1)), (4, (7, 17, 1)), (8, (9, 64)), (3, (33, 2))])
@pytest.mark.parametrize("in_place", [False, True])
def test_conv_update_spans(rt, oracle_mod, K, rows, in_place):
    """Spans of a segment read the K rows before them from x, only the first one the state; out == x walks each
    channel's rows in order. Outputs within fp32 rounding of K products (rel 1e-5 as the existing conv tests), the
    state exact (it is copied inputs)."""
    rng = np.random.default_rng(100 * K + sum(rows))
    ch, slots = 300, 4
    segs, n = segments(rt, rows, slots)
    x = rng.standard_normal((n, ch)).astype(np.float32)
    cs0 = rng.standard_normal((slots, ch, K)).astype(np.float32)
    w = (rng.standard_normal((ch, K)) * 0.5).astype(np.float32)
    put_weight(rt, "cw", w)
    for write in (0, 1):
        put(rt, "cx", x)
        put(rt, "cs", cs0)
        put(rt, "co", x)
        rt.conv_update_seg("cx", "cs", "cw", "cx" if in_place else "co", ch, K, None, write)
        got, st = get(rt, "cx" if in_place else "co", (n, ch)), get(rt, "cs", (slots, ch, K))
        expect, states = x.astype(np.float64), cs0.astype(np.float64)
        for slot, _, m, r0 in segs:
            expect[r0:r0 + m], fin, _ = oracle_mod.conv_update(x[r0:r0 + m], cs0[slot], w)
            if write:
                states[slot] = fin
        assert np.allclose(got, expect, rtol=1e-5, atol=1e-6)
        assert np.array_equal(st, states)
    if len(rows) == 1:
        return
    segs, n = segments(rt, rows[-1:], slots)  # snapshots of the last segment's rows
    put(rt, "cs", cs0)
    put(rt, "csn", np.zeros((max(n - 1, 1), ch, K)))
    rt.conv_update_seg("cx" if not in_place else "co", "cs", "cw", "co", ch, K, "csn", 0)
    snaps = oracle_mod.conv_update(x[:n], cs0[segs[0][0]], w)[2]
    assert np.array_equal(get(rt, "csn", (-1, ch, K))[:n - 1], snaps)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 129, 200, 256, 257])
def test_rmsnorm_short_groups(rt, n):
    """Groups of up to 256 values take one wave each (64, 128 or 256 values per wave), longer ones a workgroup: against
    float64, in place and gated, 9 groups (a workgroup holds four). Bound: the fp32 sum of n squares and five
    roundings, under 4e-7 relative for n <= 257; expf in silu adds under 2e-7."""
    rng = np.random.default_rng(n)
    groups, eps = 9, 1e-6
    x, z = rng.standard_normal((2, groups, n)).astype(np.float32)
    w = rng.standard_normal(n).astype(np.float32)
    put_weight(rt, "nw", w)
    put(rt, "nz", z)
    expect = x.astype(np.float64) / np.sqrt((x.astype(np.float64) ** 2).mean(-1, keepdims=True) + eps) * w
    for gated in (False, True):
        put(rt, "nx", x)
        if gated:
            rt.gated_rmsnorm("nx", "nw", "nz", "nx", n, eps, groups)
            expect = expect * z / (1.0 + np.exp(-z.astype(np.float64)))
        else:
            rt.rmsnorm("nx", "nw", "nx", n, eps, groups)
        assert np.allclose(get(rt, "nx", (groups, n)), expect, rtol=6e-7, atol=1e-12)
