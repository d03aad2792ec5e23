"""3-4 tokens with K a multiple of 4 but not of 16 on the persistent matrix-core kernel (gemv_quads, TAIL): 1, 2 and 3 words
left over per row, K just past and just short of whole chunks of 256 and of the longest rows, one partial quad of rows and
more quad groups than workgroups, the row pitch of a wider tensor (odd pitches too), the optional operands. Norm-relative
error against the FP64 oracle rounded to the output dtype within 1e-3, as every few-token kernel."""
import pytest
import torch

from conftest import DT, bits, from_bits, rel_err

pytestmark = pytest.mark.gpu

SHAPES = [(20, 3), (28, 64), (44, 5), (252, 37), (260, 1000), (1028, 8200), (2044, 9), (4108, 4097), (5124, 700), (8188, 66), (8204, 1026),
          (13828, 130), (16380, 50)]


@pytest.mark.parametrize("m", (3, 4))
@pytest.mark.parametrize("k,n", SHAPES)
def test_quads_tail(wq, oracle, k, n, m):
    for i, dtype in enumerate((torch.bfloat16, torch.float16)):
        g = torch.Generator().manual_seed(k + n + m + i)
        pitch = k + (0, 6, 1)[(k // 4 + m + i) % 3]
        wide = torch.randn(m, pitch, generator=g).to(dtype)
        wide[:, k:] = float("nan")  # values past K must not reach the products
        w = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8)
        s = (torch.rand(n, generator=g) + 0.5) / 127
        full = i == 0
        bias, res, rs = (torch.randn(*shape, generator=g).to(dtype) if full else None for shape in ((n,), (m, n), (n,)))
        print(f"quads tail m={m} n={n} k={k} pitch={pitch} {dtype}", flush=True)
        cu = lambda t: None if t is None else t.cuda()
        y = wq.gemv_lines(wide.cuda()[:, :k], w.cuda(), s.cuda(), cu(bias), cu(res), cu(rs))
        torch.cuda.synchronize()
        b = lambda t: None if t is None else bits(t)
        ref = oracle.linear_f64(bits(wide[:, :k].contiguous()), DT[dtype], w.numpy(), s.numpy(), b(bias), b(res), b(rs))
        want = torch.from_numpy(ref).to(dtype).float()
        assert rel_err(y.cpu().float(), want) <= 1e-3
        for t in range(m):
            assert rel_err(y[t].cpu().float(), want[t]) <= 1e-3
