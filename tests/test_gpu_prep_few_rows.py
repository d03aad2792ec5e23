"""Preparation of few rows (prep_parts, prep_wide: a row spread over several workgroups, or over up to 1024 threads)
against the CPU oracle and against the one-row-per-workgroup form, bit for bit: row counts on both sides of the lines where
the form changes, K on both sides of each part count (2048 elements a part; up to 8 parts), every input operation and
ConvRot group, odd row pitches, BF16, FP16 and (without an operation) FP32."""
import numpy as np
import pytest
import torch

from conftest import DT, bits

pytestmark = pytest.mark.gpu

KS = (2048, 2064, 4096, 5120, 6160, 8192, 8208, 13824, 16384, 16392)


def inputs(m, k, dtype, act, seed, pad=0):
    g = torch.Generator().manual_seed(seed)
    width = 2 * k if act == "swiglu" else k
    x = torch.randn(m, width + pad, generator=g).to(dtype)
    x[:, : width : 37] *= 30
    return x[:, :width], (1 + 0.1 * torch.randn(k, generator=g)).to(dtype) if act == "rms_norm" else None


@pytest.mark.parametrize("k", KS)
@pytest.mark.parametrize("act", [None, "rms_norm", "swiglu", "gelu"])
def test_few_rows_match_oracle(wq, oracle, k, act):
    for i, (m, dtype) in enumerate(((1, torch.bfloat16), (3, torch.float16), (5, torch.float32))):
        if dtype == torch.float32 and act:
            continue
        x, aw = inputs(m, k, dtype, act, 10 * k + i, pad=16 * i)
        group = next((g for g in ((256, 64, 16)[i:] + (0,)) if g == 0 or k % g == 0), 0)
        for rot in {0, group}:
            print(f"few rows m={m} k={k} {dtype} act={act} group={rot}", flush=True)
            xc = x.cuda() if i == 0 else torch.empty(m, x.shape[1] + 16 * i, dtype=dtype, device="cuda")[:, : x.shape[1]].copy_(x)
            awc = None if aw is None else aw.cuda()
            args = (DT[dtype], rot, act, None if aw is None else bits(aw), 1e-6)
            q, sa = wq.quantize_blocks(xc, rot, act, awc, 1e-6)
            qo, so = oracle.quantize_blocks(bits(x), *args)
            np.testing.assert_array_equal(q.cpu().numpy(), qo)
            np.testing.assert_array_equal(sa.cpu().numpy(), so)
            hi, lo, s = wq.quantize(xc, rot, True, act, awc, 1e-6)
            ho, loo, so = oracle.quantize(bits(x), DT[dtype], rot, True, act, None if aw is None else bits(aw), 1e-6)
            np.testing.assert_array_equal(hi.cpu().numpy(), ho)
            np.testing.assert_array_equal(lo.cpu().numpy(), loo)
            np.testing.assert_array_equal(s.cpu().numpy(), so)
            if dtype != torch.float32 and (act or rot):
                t = wq.transform_rows(xc, rot, act, awc, 1e-6)
                np.testing.assert_array_equal(bits(t), oracle.transform_rows(bits(x), *args))


@pytest.mark.parametrize("k,lines", [(4096, (512,)), (5120, (256, 341, 512, 768)), (13824, (146, 256, 512, 1024))])
@pytest.mark.parametrize("act", ["rms_norm", "gelu"])
def test_spread_rows_equal_whole_rows(wq, k, lines, act):
    """One row more or less changes the form, not a row's bits: the rows at each line against the same rows in a call of 2048
    (beyond every line)."""
    x, aw = inputs(2048, k, torch.bfloat16, act, k)
    x, aw = x.cuda(), None if aw is None else aw.cuda()
    q, sa = wq.quantize_blocks(x, 0, act, aw, 1e-6)
    hi, lo, s = wq.quantize(x, 0, True, act, aw, 1e-6)
    t = wq.transform_rows(x, 0, act, aw, 1e-6)
    for line in lines:
        for m in (line, line + 1):
            part = x[:m]
            assert all(torch.equal(a, b[:m]) for a, b in zip(wq.quantize_blocks(part, 0, act, aw, 1e-6), (q, sa)))
            assert all(torch.equal(a, b[:m]) for a, b in zip(wq.quantize(part, 0, True, act, aw, 1e-6), (hi, lo, s)))
            assert torch.equal(wq.transform_rows(part, 0, act, aw, 1e-6), t[:m])
