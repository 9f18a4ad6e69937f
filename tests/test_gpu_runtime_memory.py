"""The runtime's device memory between its callers: tensors handed out or taken in, streams, threads and graphs."""
from __future__ import annotations

import numpy as np
import pytest

from vinf_3080ti_amd import GGUFTensorType as T

pytestmark = pytest.mark.gpu


@pytest.fixture
def rt():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vinf_3080ti_amd.runtime import HipWeightRuntime

    return HipWeightRuntime()


def test_exchanged_storage_is_followed(rt):
    """A buffer's tensor from buffer_tensor and a tensor given to upload_device stay the caller's to exchange or resize:
    later calls read and write what they hold then, and a size that no longer fits is refused."""
    import torch

    rng = np.random.default_rng(1)
    n = 256
    a, b, c = (torch.from_numpy(rng.standard_normal(n).astype(np.float32)).cuda() for _ in range(3))
    for name in ("a", "b", "o"):
        rt.alloc(name, n)
    ta, to = rt.buffer_tensor("a"), rt.buffer_tensor("o")
    ta.copy_(a)
    rt.buffer_tensor("b").copy_(b)
    rt.add("a", "b", "o", n)
    assert torch.equal(to, a + b)
    ta.set_(c)  # another storage
    rt.add("a", "b", "o", n)
    assert torch.equal(to, c + b)
    to.resize_(4096).zero_()  # a larger storage
    rt.add("a", "b", "o", n)
    assert torch.equal(to[:n], c + b) and not to[n:].any()
    assert rt.buffer_ptr("o") == (to.data_ptr(), 4096)
    ta.set_(torch.zeros(16, device="cuda"))
    with pytest.raises(ValueError):
        rt.add("a", "b", "o", n)
    w = torch.zeros(n * 4 + 256, dtype=torch.uint8, device="cuda")
    w[: n * 4].view(torch.float32).copy_(a)
    rt.upload_device("w", w, T.F32, n, 1)
    other = torch.zeros_like(w)
    other[: n * 4].view(torch.float32).copy_(c)
    for weight in (a, c):
        rt.alloc("x", n)
        rt.buffer_tensor("x").copy_(b)
        rt.rmsnorm("x", "w", "x", n, 1e-6)
        x = b.double()
        want = x / torch.sqrt((x * x).mean() + 1e-6) * weight.double()
        assert torch.allclose(rt.buffer_tensor("x").double(), want, rtol=1e-6, atol=1e-12)
        w.set_(other)


def test_exchanged_page_table_is_followed(rt):
    import torch

    page, kvh, hd = 16, 2, 64
    rt.alloc("pt", 4)
    rt.set_paging("pt", page, 4, 1)
    rt.set_segments([(0, 0, 40)])
    x = torch.randn(40, kvh, hd, device="cuda")
    for name in ("k", "v"):
        rt.alloc(name, x.numel())
        rt.buffer_tensor(name).copy_(x.reshape(-1))
        rt.alloc(name + "c", 4 * kvh * page * hd)
    rt.buffer_tensor("pt").set_(torch.tensor([2, 0, 3, 1], dtype=torch.int32, device="cuda").view(torch.float32))
    rt.kv_append_seg("k", "v", "kc", "vc", kvh, hd)
    pool = rt.buffer_tensor("kc").view(4, kvh, page, hd)
    assert torch.equal(pool[2].transpose(0, 1), x[:16]) and torch.equal(pool[0].transpose(0, 1), x[16:32])


KH, VH, KD, VD = 2, 4, 128, 64


def gated_delta_case(rt, rng, rows: int, tag: str) -> dict:
    """Buffers of one gated-delta pass (long enough for the chunked kernels) under names that end in tag."""
    import torch

    sizes = {"conv": rows * (2 * KH * KD + VH * VD), "b": rows * VH, "a": rows * VH, "s": VH * KD * VD, "o": rows * VH * VD}
    held = {}
    for name, n in sizes.items():
        rt.alloc(name + tag, n)
        held[name] = rt.buffer_tensor(name + tag)
        if name != "o":
            held[name].copy_(torch.from_numpy(rng.standard_normal(n).astype(np.float32)))
    for name, v in (("sa", -rng.uniform(0.02, 1.0, VH)), ("dt", rng.standard_normal(VH))):
        rt.upload_raw(name + tag, v.astype(np.float32).tobytes(), T.F32, VH, 1)
    held["rows"], held["tag"] = rows, tag
    return held


def gated_delta(rt, c: dict, write_state: int = 0) -> None:
    t = c["tag"]
    rt.gated_delta("conv" + t, "b" + t, "a" + t, "sa" + t, "dt" + t, "s" + t, "o" + t, KH, VH, KD, VD, 1e-6, 0, c["rows"],
                   None, write_state)


def test_threads_on_one_stream_take_turns(rt):
    """Calls that share a stream's workspace do not overlap between threads, from the look at it to the last launch (the
    launches of a call are stood in for by a wait on the host)."""
    import threading
    import time

    inside, most, seen = 0, 0, []

    class Stub:
        def __getattr__(self, name):
            return getattr(lib, name)

        def vq_gated_delta_seg_ws(self, *args):
            nonlocal inside, most
            inside += 1
            most = max(most, inside)
            seen.append(args[-3:-1])
            time.sleep(0.02)
            inside -= 1
            return 0

    lib = rt._rt._lib
    cases = [gated_delta_case(rt, np.random.default_rng(i), 40 + 100 * i, str(i)) for i in range(2)]
    rt._rt._lib = Stub()
    threads = [threading.Thread(target=lambda c=c: [gated_delta(rt, c) for _ in range(4)]) for c in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    rt._rt._lib = lib
    assert len(seen) == 8 and all(ws for ws, _ in seen) and most == 1


def test_streams_have_scratch_of_their_own(rt):
    """Two threads on two streams, calls of different sizes side by side: the results of each alone. The argmax ids too."""
    import threading

    import torch

    cases = [gated_delta_case(rt, np.random.default_rng(5 + i), 64 + 300 * i, str(i)) for i in range(2)]
    want = []
    for c in cases:
        gated_delta(rt, c)
        want.append(c["o"].clone())
    n, rows = 5000, 64
    for i in range(2):
        rt.alloc(f"l{i}", n * rows)
        x = torch.randn(rows, n, device="cuda")
        rt.buffer_tensor(f"l{i}").copy_(x.reshape(-1))
        want.append(x.argmax(1).tolist())
    torch.cuda.synchronize()
    failed = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                cases[i]["o"].zero_()
                gated_delta(rt, cases[i])
                ids = rt.argmax_rows(f"l{i}", n, rows)
                if not torch.equal(cases[i]["o"], want[i]) or ids != want[2 + i]:
                    failed.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    assert rt.vram_bytes() > rt.buffer_bytes()


def test_graph_keeps_its_workspace(rt):
    """A captured gated-delta pass of several chunks, warmed up on another stream than the capture's: every replay gives the
    eager bits, with eager calls between, also after a larger call has made the capture stream's workspace grow and other
    tensors have taken what is free."""
    import torch

    c = gated_delta_case(rt, np.random.default_rng(9), 200, "g")
    big = gated_delta_case(rt, np.random.default_rng(10), 1200, "b")
    state = c["s"].clone()
    gated_delta(rt, c, 1)
    want, after = c["o"].clone(), c["s"].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        gated_delta(rt, c, 1)
    for rep in range(5):
        if rep == 2:
            with torch.cuda.stream(side):
                gated_delta(rt, big)
            torch.cuda.synchronize()
            hold = [torch.full((1 << 18,), float("nan"), device="cuda") for _ in range(64)]
        c["o"].fill_(float("nan"))
        c["s"].copy_(state)
        gated_delta(rt, big)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c["o"], want) and torch.equal(c["s"], after), rep
    del hold


def test_gated_delta_workspace_contract(rt):
    """vq_gated_delta_seg_ws: too small or misaligned a workspace is refused before any launch, none is the per-token route,
    and a pass without long segments needs none."""
    import ctypes

    import torch

    from vinf_3080ti_amd import _lib

    lib = rt._rt._lib
    c = gated_delta_case(rt, np.random.default_rng(3), 64, "w")
    sa, dt = (rt.tensor_info(k + "w")[0] for k in ("sa", "dt"))
    seg = (ctypes.c_int32 * 4)(0, 0, 64, 0)
    need = lib.vq_gated_delta_seg_workspace_bytes(seg, 1, KH, VH, KD, VD)
    ws = torch.empty(need + 16, dtype=torch.uint8, device="cuda")

    def call(at, nbytes, table=seg):
        c["o"].zero_()
        st = lib.vq_gated_delta_seg_ws(c["conv"].data_ptr(), c["b"].data_ptr(), c["a"].data_ptr(), sa, dt, c["s"].data_ptr(), 4,
                                       c["o"].data_ptr(), KH, VH, KD, VD, 1e-6, 0, table, 1, None, 0, at, nbytes, None)
        torch.cuda.synchronize()
        return st, c["o"].clone()

    assert need > 0
    for at, nbytes in ((ws.data_ptr(), need - 1), (ws.data_ptr(), 0), (ws.data_ptr() + 4, need)):
        st, out = call(at, nbytes)
        assert st == _lib.VQ_ERR_WORKSPACE and not out.any()
    st, chunked = call(ws.data_ptr(), need)
    assert st == 0 and chunked.any()
    st, token = call(None, 0)
    assert st == 0 and torch.allclose(chunked, token, rtol=0, atol=2e-6 * float(token.abs().max()))
    short = (ctypes.c_int32 * 4)(0, 0, 23, 0)
    assert lib.vq_gated_delta_seg_workspace_bytes(short, 1, KH, VH, KD, VD) == 0
    assert call(ws.data_ptr(), 0, short)[0] == 0
