"""One token with its input operation in the GEMV's launch (wq8_gemv_line_act): the bits of transform_rows + gemv_lines at
the edges of its K range (one partial line, whole and ragged lines, more than one chunk a thread, 16 lines), N on both
sides of two rows a wave, with and without the optional operands; and where linear() takes it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", ["rms_norm", "swiglu", "gelu"])
@pytest.mark.parametrize("k,n", [(16, 3), (1024, 17), (1040, 700), (2064, 8193), (5120, 520), (8192, 8200), (8208, 33), (16384, 40)])
def test_line_act_equals_two_launches(wq, k, n, act, dtype):
    from wgpkernels_amd.int8 import _native
    g = torch.Generator().manual_seed(k + n)
    x = (3 * torch.randn(1, 2 * k if act == "swiglu" else k, generator=g)).to(dtype).cuda()
    aw = (1 + 0.1 * torch.randn(k, generator=g)).to(dtype).cuda()
    w = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8).cuda()
    s = ((torch.rand(n, generator=g) + 0.5) / 127).cuda()
    bias, res, rs = (torch.randn(*shape, generator=g).to(dtype).cuda() for shape in ((n,), (1, n), (n,)))
    p = lambda t: None if t is None else t.data_ptr()
    for weight, b, r, scale in ((aw, bias, res, rs), (None, None, None, None)):
        print(f"line act={act} k={k} n={n} {dtype} operands={b is not None}", flush=True)
        want = wq.gemv_lines(wq.transform_rows(x, 0, act, weight, 1e-6), w, s, b, r, scale)
        y = torch.empty(1, n, dtype=dtype, device="cuda")
        wq.library().call("wq8_gemv_line_act", x.data_ptr(), wq.ACTS[act], p(weight), 1e-6, w.data_ptr(), s.data_ptr(), p(b), p(r), p(scale),
                          y.data_ptr(), n, k, wq.DTYPES[dtype], _native.gpu(x).stream())
        torch.cuda.synchronize()
        assert torch.equal(y, want)


def test_line_act_route(wq, monkeypatch):
    """linear() takes the fused launch for one unrotated token and small weights, and refuses what it refused."""
    calls = []
    lib = wq.library()
    call = lib.call
    monkeypatch.setattr(lib, "call", lambda name, *args: (calls.append(name), call(name, *args))[1])
    x = torch.randn(2, 512, device="cuda").bfloat16()
    w = torch.randint(-127, 128, (64, 512), dtype=torch.int8, device="cuda")
    s = torch.rand(64, device="cuda") / 127
    run = lambda **kw: (calls.clear(), wq.linear(kw.pop("x", x[:1]), w, kw.pop("s", s), mode="lines", **kw), list(calls))[2]
    assert run(act="gelu") == ["wq8_gemv_line_act"]
    assert run(x=x, act="gelu") == ["wq8_transform_rows", "wq8_gemv_lines"]
    assert run(act="gelu", group=16) == ["wq8_transform_rows", "wq8_gemv_lines"]
    assert run() == ["wq8_gemv_lines"]
    odd = torch.randn(1, 520, device="cuda").bfloat16()[:, 4:516]  # not 16-byte aligned
    with pytest.raises(ValueError):
        run(x=odd, act="gelu")
    with pytest.raises(ValueError):
        run(s=torch.rand(64, 4, device="cuda"), act="gelu")
    with pytest.raises(RuntimeError):
        run(x=x[:1].float(), act="gelu")
