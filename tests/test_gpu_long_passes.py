"""Prompt-length passes of the sequence ops: the kernels that split a long segment's rows over workgroups, at the edges
of their spans and chunks, against the float64 restatements in oracle/oracle.py."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2
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


# Two, four and eight rows at once, shorter segments beside them; three hundred channels leave a part of a workgroup.
@pytest.mark.parametrize("K", [1, 3, 4, 8])
@pytest.mark.parametrize("rows", [(2,), (3,), (4,), (5,), (8,), (1, 2), (4, 1, 2, 3), (8, 5, 1, 7)])
def test_conv_update_short_segments(rt, oracle_mod, K, rows):
    """Decode and verify passes of several sequences, state and snapshots; bounds as above."""
    rng = np.random.default_rng(10 * K + sum(rows))
    ch, slots = 300, 4
    segs, n = segments(rt, rows, slots)
    x = rng.standard_normal((n, ch)).astype(np.float32)
    cs0 = rng.standard_normal((slots, ch, K)).astype(np.float32)
    w = (rng.standard_normal((ch, K)) * 0.5).astype(np.float32)
    put_weight(rt, "cw", w)
    put(rt, "cx", x)
    for write in (0, 1):
        put(rt, "cs", cs0)
        put(rt, "co", x)
        put(rt, "csn", np.zeros((max(n - 1, 1), ch, K)))
        snap = "csn" if len(rows) == 1 and n > 1 else None
        rt.conv_update_seg("cx", "cs", "cw", "co", ch, K, snap, write)
        expect, states = x.astype(np.float64), cs0.astype(np.float64)
        for slot, _, m, r0 in segs:
            expect[r0:r0 + m], fin, snaps = oracle_mod.conv_update(x[r0:r0 + m], cs0[slot], w)
            if write:
                states[slot] = fin
        assert np.allclose(get(rt, "co", (n, ch)), expect, rtol=1e-5, atol=1e-6)
        assert np.array_equal(get(rt, "cs", (slots, ch, K)), states)
        if snap:
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


def gated_delta_rows(oracle_mod, inp, segs, states, kh, vh, kd, vd, order):
    """The float64 restatement per segment: outputs [rows][vh][vd] at the segments' rows, states after the pass."""
    n = inp["conv"].shape[0]
    out, fin = np.zeros((n, vh, vd)), states.astype(np.float64)
    for slot, _, m, r0 in segs:
        rows = slice(r0, r0 + m)
        out[rows], fin[slot], _ = oracle_mod.gated_delta(inp["conv"][rows], inp["b"][rows], inp["a"][rows], inp["ssm_a"],
                                                         inp["dt"], states[slot], kh, vh, kd, vd, 1e-6, order)
    return out, fin


def gated_delta_inputs(rng, n, kh, vh, kd, vd, slots):
    return dict(conv=rng.standard_normal((n, 2 * kh * kd + vh * vd)).astype(np.float32),
                b=rng.standard_normal((n, vh)).astype(np.float32), a=rng.standard_normal((n, vh)).astype(np.float32),
                ssm_a=-rng.uniform(0.02, 2.0, vh).astype(np.float32), dt=rng.standard_normal(vh).astype(np.float32),
                state=(0.1 * rng.standard_normal((slots, vh, kd, vd))).astype(np.float32))


def run_gated_delta(rt, inp, segs, shape, elem, order, write, eps=1e-6):
    kh, vh, kd, vd = shape
    n = inp["conv"].shape[0]
    for name in ("ssm_a", "dt"):
        put_weight(rt, "g." + name, inp[name])
    for name in ("conv", "b", "a"):
        put(rt, "g." + name, inp[name])
    put(rt, "g.s", inp["state"], elem)
    put(rt, "g.o", np.zeros((n, vh, vd)))
    rt.set_segments(segs)
    rt.gated_delta_seg("g.conv", "g.b", "g.a", "g.ssm_a", "g.dt", "g.s", "g.o", kh, vh, kd, vd, eps, order, None, write)
    return get(rt, "g.o", (n, vh, vd)), get(rt, "g.s", inp["state"].shape)


# Chunks of 32 tokens from 24 rows on, 16 chunks (less with several segments) per launch pair: below and at the
# threshold, one chunk, a chunk and a row, two launch pairs, and long segments beside short ones; ragged head counts
# against the XCD grouping of 8 heads, narrow states, both head orders, fp16 state.
@pytest.mark.parametrize("rows,shape,order,elem", [
    ((23,), (1, 2, 128, 128), 0, 4), ((24,), (1, 2, 128, 128), 1, 4), ((32,), (2, 6, 128, 64), 0, 4),
    ((33, 1, 70), (3, 9, 128, 32), 1, 4), ((530,), (1, 1, 128, 96), 0, 4), ((65, 300, 5), (2, 10, 128, 128), 1, 2),
    ((520,), (1, 2, 128, 32), 0, 2)])
def test_gated_delta_chunks(rt, oracle_mod, rows, shape, order, elem):
    """The chunked kernels against the float64 restatement, relative to the largest value: fp32 sums over 128 state rows
    and 32 tokens per chunk, the same as the per-token kernel's error (3e-7 measured for both), so 2e-6; an fp16 state
    rounds once (2^-11). write_state = 0 leaves the state as it was."""
    kh, vh, kd, vd = shape
    rng = np.random.default_rng(sum(rows) + vh + vd)
    slots = 4
    rt.alloc("pt", 64)
    rt.set_paging("pt", 1024, 64 // slots, slots)
    segs, r0 = [], 0
    for i, m in enumerate(rows):
        segs.append((slots - 1 - i, 0, m, r0))
        r0 += m + (2 if i == 0 else 0)
    inp = gated_delta_inputs(rng, r0, kh, vh, kd, vd, slots)
    if elem == 2:
        inp["state"] = inp["state"].astype(np.float16).astype(np.float32)
    expect, fin = gated_delta_rows(oracle_mod, inp, segs, inp["state"], kh, vh, kd, vd, order)
    for write in (0, 1):
        out, st = run_gated_delta(rt, inp, segs, shape, elem, order, write)
        assert np.abs(out - expect).max() <= 2e-6 * np.abs(expect).max()
        want, tol = (fin, 2e-6 if elem == 4 else 5e-4) if write else (inp["state"], 0.0)
        assert np.abs(st - want).max() <= tol * np.abs(want).max()


@pytest.mark.parametrize("what", ["v", "k", "beta", "decay above one"])
def test_gated_delta_chunks_keep_causality(rt, oracle_mod, what):
    """A value that is not finite reaches its own token and the ones after it, never an earlier token of its chunk (nor,
    in v, another column), as the per-token kernel has it; decays above one whose products leave the fp32 range while
    the state does not are computed too."""
    shape = kh, vh, kd, vd = 1, 2, 128, 64
    rng = np.random.default_rng(5)
    n, bad = 80, 45
    rt.alloc("pt", 64)
    rt.set_paging("pt", 64, 16, 1)
    inp = gated_delta_inputs(rng, n, kh, vh, kd, vd, 1)
    segs = [(0, 0, n, 0)]
    if what == "decay above one":  # e^15 a token over a zero state and zero values, then decays near one
        inp["ssm_a"][:], inp["dt"][:], inp["a"][:32], inp["a"][32:] = 1.0, 0.0, 15.0, -12.0
        inp["state"][:] = inp["conv"][:32, 2 * kh * kd:] = 0.0
        expect, fin = gated_delta_rows(oracle_mod, inp, segs, inp["state"], kh, vh, kd, vd, 0)
        out, st = run_gated_delta(rt, inp, segs, shape, 4, 0, 1)
        assert np.abs(out - expect).max() <= 2e-6 * np.abs(expect).max()
        assert np.abs(st - fin).max() <= 2e-6 * np.abs(fin).max()
        return
    clean, _ = gated_delta_rows(oracle_mod, inp, segs, inp["state"], kh, vh, kd, vd, 0)
    cols = slice(None)
    if what == "v":
        inp["conv"][bad, 2 * kh * kd + 3] = np.inf  # head 0, column 3
        cols = 3
    elif what == "k":
        inp["conv"][bad, kh * kd + 7] = np.nan
    else:
        inp["b"][bad, 0] = np.nan
    out, st = run_gated_delta(rt, inp, segs, shape, 4, 0, 1)
    assert np.abs(out[:bad] - clean[:bad]).max() <= 2e-6 * np.abs(clean).max()
    assert not np.isfinite(out[bad:, 0, cols]).any() and not np.isfinite(st[0, 0, :, cols]).any()
    if what == "v":
        rest = np.arange(vd) != 3
        assert np.abs(out[:, 0, rest] - clean[:, 0, rest]).max() <= 2e-6 * np.abs(clean).max()


@pytest.mark.parametrize("elem", [4, 2])
def test_gated_delta_many_long_segments(rt, oracle_mod, elem):
    """A pass of twenty segments of 7 to 1100 rows: several groups of long ones, some of them over several launches, and
    short ones. Every segment's bits are those of a pass of its own; the longest and the shortest long one are right."""
    shape = kh, vh, kd, vd = 4, 48, 128, 32
    rng = np.random.default_rng(9)
    rows = [24, 1100, 40, 7, 513, 24, 90, 31, 32, 33, 64, 300, 24, 65, 25, 520, 128, 23, 48, 1]
    slots = len(rows)
    rt.alloc("pt", slots)
    rt.set_paging("pt", 2048, 1, slots)
    starts = np.cumsum([0] + rows)
    inp = gated_delta_inputs(rng, int(starts[-1]), kh, vh, kd, vd, slots)
    if elem == 2:
        inp["state"] = inp["state"].astype(np.float16).astype(np.float32)
    segs = [(slots - 1 - i, 0, n, int(starts[i])) for i, n in enumerate(rows)]
    out, st = run_gated_delta(rt, inp, segs, shape, elem, 0, 1)
    for i, n in enumerate(rows):
        part = dict(inp, **{k: inp[k][starts[i]:starts[i + 1]] for k in ("conv", "b", "a")})
        alone, fin = run_gated_delta(rt, part, [(slots - 1 - i, 0, n, 0)], shape, elem, 0, 1)
        assert np.array_equal(alone, out[starts[i]:starts[i + 1]]), n
        assert np.array_equal(fin[slots - 1 - i], st[slots - 1 - i]), n
    head = dict(inp, conv=np.concatenate([inp["conv"][:, :kd], inp["conv"][:, kh * kd:(kh + 1) * kd],
                                          inp["conv"][:, 2 * kh * kd:2 * kh * kd + vd]], 1), b=inp["b"][:, :1],
                a=inp["a"][:, :1], ssm_a=inp["ssm_a"][:1], dt=inp["dt"][:1])  # head 0 by itself
    for i in (0, 1):
        expect, fin = gated_delta_rows(oracle_mod, head, segs[i:i + 1], inp["state"][:, :1], 1, 1, kd, vd, 0)
        at = slice(starts[i], starts[i + 1])
        assert np.abs(out[at, :1] - expect[at]).max() <= 2e-6 * np.abs(expect).max()
        slot = segs[i][0]
        assert np.abs(st[slot, :1] - fin[slot]).max() <= (2e-6 if elem == 4 else 5e-4) * np.abs(fin[slot]).max()


def test_gated_delta_batch_invariant_cuts(rt):
    """In batch-invariant mode a prompt's bits do not depend on where it is cut into passes: 70 rows at once, as 40 + 30, and
    as 40 rows beside another sequence's and 30 alone; outside the mode the first of them runs in chunks."""
    shape = kh, vh, kd, vd = 1, 2, 128, 64
    rng = np.random.default_rng(13)
    rt.alloc("pt", 64)
    rt.set_paging("pt", 128, 16, 4)
    inp = gated_delta_inputs(rng, 110, kh, vh, kd, vd, 4)

    def part(lo, hi, state=inp["state"]):
        return dict(inp, state=state, **{k: inp[k][lo:hi] for k in ("conv", "b", "a")})

    chunked, _ = run_gated_delta(rt, part(0, 70), [(1, 0, 70, 0)], shape, 4, 0, 1)
    rt.set_batch_invariant(True)
    whole, fin = run_gated_delta(rt, part(0, 70), [(1, 0, 70, 0)], shape, 4, 0, 1)
    first, mid = run_gated_delta(rt, part(0, 40), [(1, 0, 40, 0)], shape, 4, 0, 1)
    beside, st = run_gated_delta(rt, inp, [(2, 0, 40, 70), (1, 0, 40, 0)], shape, 4, 0, 1)
    assert np.array_equal(first, whole[:40]) and np.array_equal(beside[:40], whole[:40])
    assert np.array_equal(st[1], mid[1])
    rest, end = run_gated_delta(rt, part(40, 70, mid), [(1, 40, 30, 0)], shape, 4, 0, 1)
    assert np.array_equal(rest, whole[40:]) and np.array_equal(end[1], fin[1])
    rt.set_batch_invariant(False)
    assert not np.array_equal(chunked, whole)
    assert np.abs(chunked - whole).max() <= 4e-6 * np.abs(whole).max()


@pytest.mark.parametrize("bad", [5, 511, 512, 600, 699])
def test_gated_delta_chunks_flagged_in_any_launch(rt, oracle_mod, bad):
    """One infinite value in a pass of 22 chunks over two launch pairs, in each of them and at their edge: its column from its
    token on, and nothing else (bound as above)."""
    shape = kh, vh, kd, vd = 1, 2, 128, 64
    rng = np.random.default_rng(14)
    n = 700
    rt.alloc("pt", 64)
    rt.set_paging("pt", 1024, 16, 1)
    inp = gated_delta_inputs(rng, n, kh, vh, kd, vd, 1)
    segs = [(0, 0, n, 0)]
    expect, fin = gated_delta_rows(oracle_mod, inp, segs, inp["state"], kh, vh, kd, vd, 0)
    inp["conv"][bad, 2 * kh * kd + vd + 37] = -np.inf  # head 1, column 37
    out, st = run_gated_delta(rt, inp, segs, shape, 4, 0, 1)
    touched = np.zeros((n, vh, vd), bool)
    touched[bad:, 1, 37] = True
    assert np.array_equal(~np.isfinite(out), touched)
    assert np.abs(np.where(touched, 0, out - expect)).max() <= 2e-6 * np.abs(expect).max()
    assert not np.isfinite(st[0, 1, :, 37]).any()
    st[0, 1, :, 37] = fin[0, 1, :, 37] = 0.0
    assert np.abs(st - fin).max() <= 2e-6 * np.abs(fin).max()


# Largest error of the outputs and of the state, as a multiple of the per-token kernel's (measured: independent keys 0.85
# and 0.8-1.1, correlated ones 1.1 and 1.1, equal ones 1.3-1.6 and 1.4-1.8).
@pytest.mark.parametrize("keys,out_bound,state_bound", [("independent", 1.0, 1.25), ("correlated", 1.3, 1.3),
                                                        ("equal", 2.0, 2.0)])
def test_gated_delta_chunks_rounding(rt, oracle_mod, keys, out_bound, state_bound):
    """Rel-L2 error against float64 beside the per-token kernel's on the same inputs, 512 rows: keys as a model's
    normalised ones, and keys that share a direction with beta near one and slow decays, where the triangular inverse has
    large entries off its diagonal and the sums cancel (token by token each update corrects the one before it)."""
    shape = kh, vh, kd, vd = 2, 4, 128, 128
    rt.alloc("pt", 64)
    rt.set_paging("pt", 512, 16, 1)
    err = np.zeros((2, 2))
    for seed in range(3):
        rng = np.random.default_rng(20 + seed)
        inp = gated_delta_inputs(rng, 512, kh, vh, kd, vd, 1)
        if keys != "independent":
            k = inp["conv"][:, kh * kd:2 * kh * kd]
            k[:] = (0.0 if keys == "equal" else 0.1) * k + 0.9 * rng.standard_normal(kh * kd)
            inp["b"] += 5.0
            inp["ssm_a"][:] = -rng.uniform(0.001, 0.05, vh)
        segs = [(0, 0, 512, 0)]
        expect, fin = gated_delta_rows(oracle_mod, inp, segs, inp["state"], kh, vh, kd, vd, 0)
        for i, invariant in enumerate((False, True)):
            rt.set_batch_invariant(invariant)
            out, st = run_gated_delta(rt, inp, segs, shape, 4, 0, 1)
            err[i] += rel_l2(out, expect) ** 2, rel_l2(st, fin) ** 2
        rt.set_batch_invariant(False)
    ratio = np.sqrt(err[0] / err[1])
    print(f"{keys}: outputs {ratio[0]:.2f}, state {ratio[1]:.2f}")
    assert ratio[0] <= out_bound and ratio[1] <= state_bound


@pytest.mark.parametrize("g", [1.001, 1.1, 1.3])
def test_gated_delta_chunks_decay_above_one(rt, oracle_mod, g):
    """Equal keys, each token replacing what the one before wrote: token by token nothing grows, while the products of a
    chunk's decays reach 1.3^32 = 4400. Bound as above, 2e-6 of the largest value."""
    shape = kh, vh, kd, vd = 1, 2, 128, 64
    rng = np.random.default_rng(8)
    rt.alloc("pt", 64)
    rt.set_paging("pt", 64, 16, 1)
    inp = gated_delta_inputs(rng, 64, kh, vh, kd, vd, 1)
    inp["conv"][:, :2 * kh * kd] = np.tile(rng.standard_normal(kd), 2)
    inp["a"][:], inp["dt"][:], inp["b"][:], inp["state"][:] = 0.0, 0.0, 6.0, 0.0
    inp["ssm_a"][:] = np.log(g) / np.log(2.0)
    segs = [(0, 0, 64, 0)]
    expect, _ = gated_delta_rows(oracle_mod, inp, segs, inp["state"], kh, vh, kd, vd, 0)
    out, _ = run_gated_delta(rt, inp, segs, shape, 4, 0, 1)
    assert np.abs(out - expect).max() <= 2e-6 * np.abs(expect).max()


@pytest.mark.parametrize("what", ["keys", "keys and queries", "keys, eps 0", "state", "values"])
def test_gated_delta_chunks_fp32_range(rt, oracle_mod, what):
    """Finite inputs whose norms, products with the state or sums leave the fp32 range behave as token by token: a key
    whose squares overflow has weight zero, and a state or value at the edge of the range reaches no earlier token of its
    chunk. Same finite elements as the per-token kernel's, those within 5e-6 of the column's largest: the state of that
    kernel is rounded once per token, 80 halves of 2^-23."""
    shape = kh, vh, kd, vd = 1, 2, 128, 64
    rng = np.random.default_rng(6)
    n, k0, eps = 80, kh * kd, 0.0 if what == "keys, eps 0" else 1e-6
    rt.alloc("pt", 64)
    rt.set_paging("pt", 64, 16, 1)
    inp = gated_delta_inputs(rng, n, kh, vh, kd, vd, 1)
    segs = [(0, 0, n, 0)]
    if what.startswith("keys"):  # sum of squares 1e42, with eps 0 1e-34
        inp["conv"][[20, 25], k0:k0 + kd] *= np.float32(1e20 if eps else 1e-18)
        if what == "keys and queries":
            inp["conv"][[20, 25], :kd] *= np.float32(1e20)
    elif what == "state":  # S^T k overflows at token 20 in column 3 of head 0, and nowhere before
        inp["ssm_a"][:], inp["b"][:] = -1e-6, -20.0
        inp["state"][0, 0, 5, 3] = 2.5e38
        inp["conv"][:, [5, k0 + 5]] = 0.01
        inp["conv"][20, k0 + 5] = 4.0
    else:  # d overflows at token 26 in column 3 of head 0
        inp["b"][:] = 20.0
        inp["conv"][26, k0:k0 + kd] = -inp["conv"][25, k0:k0 + kd]
        inp["conv"][[25, 26], 2 * kh * kd + 3] = 3e38
        inp["conv"][[25, 26], :kd] *= np.float32(0.01)  # (S^T q of the token before does not)
    out, st = run_gated_delta(rt, inp, segs, shape, 4, 0, 1, eps)
    rt.set_batch_invariant(True)
    want, fin = run_gated_delta(rt, inp, segs, shape, 4, 0, 1, eps)
    rt.set_batch_invariant(False)
    assert np.isfinite(want[:20]).all() and np.isfinite(want[:, 1]).all()
    for got, ref in ((out, want), (st[0], fin[0])):
        ok = np.isfinite(ref)
        assert np.array_equal(np.isfinite(got), ok)
        diff, size = np.where(ok, np.abs(np.where(ok, got, 0) - np.where(ok, ref, 0)), 0), np.where(ok, np.abs(ref), 0)
        if ref is want:
            assert (diff[:20].max((0, 1)) <= 5e-6 * size[:20].max((0, 1))).all()  # before the large value
        assert (diff.max((0, 1)) <= 5e-6 * size.max((0, 1))).all()


# Key blocks of 32 in two parities, 16-row tiles, two to four heads of a kv head per workgroup.
@pytest.mark.parametrize("heads,kvh,hd", [(6, 1, 256), (5, 1, 64), (6, 2, 128), (9, 1, 64), (2, 2, 256)])
@pytest.mark.parametrize("ntok,seq_len,window", [(9, 1, 0), (9, 24, 0), (16, 49, 0), (17, 48, 0), (33, 1, 5),
                                                 (20, 97, 40), (18, 64, 32)])
def test_prompt_attention_f16_blocks(rt, oracle_mod, heads, kvh, hd, ntok, seq_len, window):
    """The last key just before, on and after a block's and a step's edge, one parity without a key, windows that
    begin inside a block. Bar: that of the prompt attention tests (fp32 products and sums; splitting the keys in two
    shortens each chain of sums). A row's bits do not depend on the rows before it in the pass."""
    rng = np.random.default_rng(1000 * heads + hd + ntok + seq_len)
    max_seq = seq_len + ntok
    q = rng.standard_normal((ntok, heads, hd)).astype(np.float32)
    kc = (rng.standard_normal((kvh, max_seq, hd)) * 0.3).astype(np.float16)
    vc = rng.standard_normal((kvh, max_seq, hd)).astype(np.float16)
    put(rt, "pq", q)
    put(rt, "po", np.full(q.size, np.nan))
    put(rt, "pkc", kc, 2)
    put(rt, "pvc", vc, 2)
    rt.attention("pq", "pkc", "pvc", "po", heads, kvh, hd, max_seq, seq_len, ntok, 0, window)
    got = get(rt, "po", q.shape)
    ref = oracle_mod.attention(q, kc, vc, heads, kvh, seq_len, False, window)
    assert np.allclose(got, ref, rtol=2e-5, atol=2e-5)
    skip = ntok - 9
    put(rt, "pq", q[skip:])
    rt.attention("pq", "pkc", "pvc", "po", heads, kvh, hd, max_seq, seq_len + skip, 9, 0, window)
    assert np.array_equal(get(rt, "po", q.shape)[:9], got[skip:])


# More workgroups than CUs over long contexts: a head's two parities in one wave. Passes of a few rows: in two waves.
@pytest.mark.parametrize("G,hd", [(3, 64), (4, 128), (7, 64), (5, 128)])
@pytest.mark.parametrize("window,bidirectional", [(0, 0), (33, 0), (300, 0), (0, 1)])
def test_prompt_attention_f16_whole_heads(rt, oracle_mod, G, hd, window, bidirectional):
    """Both forms give the same bits: a pass of 530 rows against passes of 64 rows of it, and rows at the tiles' edges
    against the oracle (bar of the prompt attention tests)."""
    rng = np.random.default_rng(hd + G + window)
    kvh, ntok, before = 8, 530, 1200
    heads, keys = G * kvh, before + ntok
    print(f"whole heads G {G} hd {hd} window {window} bidirectional {bidirectional}", flush=True)
    q = rng.standard_normal((ntok, heads, hd)).astype(np.float32)
    kc = (rng.standard_normal((kvh, keys, hd)) * 0.3).astype(np.float16)
    vc = rng.standard_normal((kvh, keys, hd)).astype(np.float16)
    put(rt, "wk", kc, 2)
    put(rt, "wv", vc, 2)
    put(rt, "wq", q)
    put(rt, "wo", np.full(q.size, np.nan))
    rt.set_gemm_min_rows(9)
    rt.attention("wq", "wk", "wv", "wo", heads, kvh, hd, keys, before + 1, ntok, bidirectional, window)
    got = get(rt, "wo", q.shape)
    if not bidirectional:
        for r in (0, 64, ntok - 64):
            put(rt, "wq", q[r:r + 64])
            put(rt, "wo", np.full(q[:64].size, np.nan))
            rt.attention("wq", "wk", "wv", "wo", heads, kvh, hd, keys, before + 1 + r, 64, 0, window)
            assert np.array_equal(get(rt, "wo", q[:64].shape), got[r:r + 64]), r
    rt.set_gemm_min_rows(0)
    for r in (0, 15, 16, 511, ntok - 1):
        seq = keys if bidirectional else before + 1 + r
        ref = oracle_mod.attention(q[r:r + 1], kc, vc, heads, kvh, seq, False, window)
        assert np.allclose(got[r:r + 1], ref, rtol=2e-5, atol=2e-5), r


def test_prompt_attention_f16_whole_heads_paged(rt, oracle_mod):
    """The same over pages: more than 256 workgroups in a pass of 48 sequences, each sequence's rows as in a
    pass of its own."""
    rng = np.random.default_rng(12)
    heads, kvh, hd, page, pps, slots = 24, 8, 128, 64, 20, 48
    pages = rng.permutation(pps * slots).astype(np.int32)
    rt.alloc("wpt", pages.size)
    rt.write("wpt", pages.tobytes())
    rt.set_paging("wpt", page, pps, slots)
    pool = (rng.standard_normal((pps * slots, kvh, page, hd)) * 0.3).astype(np.float16)
    put(rt, "wk", pool, 2)
    put(rt, "wv", pool[::-1], 2)
    rows = [1 + 5 * (i % 4) for i in range(slots)]
    starts = np.cumsum([0] + rows)
    q = rng.standard_normal((int(starts[-1]), heads, hd)).astype(np.float32)
    put(rt, "wq", q)
    put(rt, "wo", np.full(q.size, np.nan))
    rt.set_batch_invariant(True)
    segs = [(slots - 1 - i, 1264 - 20 * i, n, int(starts[i])) for i, n in enumerate(rows)]
    rt.set_segments(segs)
    rt.attention_seg("wq", "wk", "wv", "wo", heads, kvh, hd)
    got = get(rt, "wo", q.shape)
    for i in (0, 1, 23, 47):
        part = q[starts[i]:starts[i + 1]]
        put(rt, "wq", part)
        put(rt, "wo", np.full(part.size, np.nan))
        rt.set_segments([segs[i][:3] + (0,)])
        rt.attention_seg("wq", "wk", "wv", "wo", heads, kvh, hd)
        assert np.array_equal(get(rt, "wo", part.shape), got[starts[i]:starts[i + 1]]), i
    rt.set_batch_invariant(False)
