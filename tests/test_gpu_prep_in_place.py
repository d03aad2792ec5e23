"""transform_rows written over its own input (out == x, rows k values apart): the bits of a separate output, for RMSNorm rows
of one part, several parts and past the parts' range, on both sides of the row count where the parts begin."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k", [2048, 2064, 5120, 13824, 16384, 16512])
@pytest.mark.parametrize("m", [1, 3, 146, 600])
def test_transform_rows_in_place(wq, m, k, dtype):
    from wgpkernels_amd.int8 import _native
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(m, k, generator=g).to(dtype).cuda()
    aw = (1 + 0.1 * torch.randn(k, generator=g)).to(dtype).cuda()
    for act, group in (("rms_norm", 0), ("rms_norm", 16), ("gelu", 0)):
        print(f"in place m={m} k={k} {dtype} act={act} group={group}", flush=True)
        weight = aw if act == "rms_norm" else None
        want = wq.transform_rows(x, group, act, weight, 1e-6)
        y = x.clone()
        wq.library().call("wq8_transform_rows", y.data_ptr(), y.data_ptr(), m, k, k, wq.DTYPES[dtype], group, wq.ACTS[act],
                          None if weight is None else weight.data_ptr(), 1e-6, _native.gpu(x).stream())
        torch.cuda.synchronize()
        assert torch.equal(y, want)
