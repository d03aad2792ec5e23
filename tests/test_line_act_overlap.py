"""One token with its input operation, written in place of its input (a residual stream x = x + rs * linear(op(x))): the
fused launch, whose workgroups all read x while others store, is not taken (CPU; the bits on a GPU)."""
import ctypes
from types import SimpleNamespace

import pytest
import torch

from wgpkernels_amd import int8 as wq


@pytest.mark.parametrize("n,start,act,fused", [
    (64, None, "rms_norm", True), (64, 0, "rms_norm", False), (64, 64, "rms_norm", True), (16, 56, "gelu", False), (32, 64, "swiglu", False),
    (32, 96, "swiglu", False), (32, 128, "swiglu", True),
])
def test_route(monkeypatch, n, start, act, fused):
    calls = []
    lib = SimpleNamespace(has=lambda name: True, call=lambda name, *args: calls.append(name))
    monkeypatch.setattr(wq, "library", lambda: lib)
    monkeypatch.setattr(wq, "_lib", lib)
    monkeypatch.setattr(wq._native, "gpu", lambda t: SimpleNamespace(stream=lambda: None))
    memory = torch.zeros(256, dtype=torch.bfloat16)
    width = 128 if act == "swiglu" else 64
    out = None if start is None else memory[start:start + n].view(1, n)
    y = wq.linear(memory[:width].view(1, width), torch.zeros(n, 64, dtype=torch.int8), torch.ones(n), mode="lines", act=act, out=out)
    assert y.shape == (1, n)
    assert calls == (["wq8_gemv_line_act"] if fused else ["wq8_transform_rows", "wq8_gemv_lines"])


@pytest.mark.parametrize("act,y", [(1, 0x10000), (1, 0x10000 + 126), (1, 0x10000 - 30), (2, 0x10000 + 254)])
def test_entry_point_refuses_an_overlap(act, y):
    path = wq.default_library_path()
    if not path.exists():
        pytest.skip("library not built")
    lib = wq._native.Library(path)
    p = ctypes.c_void_p
    # refused before any pointer is used
    assert lib.wq8_gemv_line_act(p(0x10000), act, None, 1e-6, p(0x20000), p(0x30000), None, None, None, p(y), 16, 64, 1, None) == -2


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["rms_norm", "gelu"])
def test_in_place_of_the_input(act):
    k = 2048
    g = torch.Generator().manual_seed(3)
    x = torch.randn(1, k, generator=g).bfloat16().cuda()
    w = torch.randint(-127, 128, (k, k), generator=g, dtype=torch.int8).cuda()
    s = ((torch.rand(k, generator=g) + 0.5) / 127 / k ** 0.5).cuda()
    rs = torch.rand(k, generator=g).bfloat16().cuda()
    want = wq.linear(x, w, s, mode="lines", act=act, eps=1e-6, residual=x, residual_scale=rs)
    y = wq.linear(x, w, s, mode="lines", act=act, eps=1e-6, residual=x, residual_scale=rs, out=x)
    torch.cuda.synchronize()
    assert y is x and torch.equal(y, want)
