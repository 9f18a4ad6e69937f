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
