"""A GEMM-path linear() fills the first rows of an output that has more of them (a buffer kept for the largest call)."""
from types import SimpleNamespace

import pytest
import torch

from wgpkernels_amd import int8 as wq


@pytest.mark.parametrize("path", ["exact", "block", "row"])
@pytest.mark.parametrize("scratch", [wq.SCRATCH_BYTES, 1])  # one chunk, chunks of CHUNK_ROW_MULTIPLE rows
def test_output_with_more_rows(monkeypatch, path, scratch):
    def call(name, *args):
        if name == "wq8_gemm":
            written.append((args[8], args[9], args[10]))  # y, m, n

    written = []
    lib = SimpleNamespace(call=call, wq8_gemm_workspace=lambda *args: None)
    monkeypatch.setattr(wq, "library", lambda: lib)
    monkeypatch.setattr(wq._native, "gpu", lambda t: SimpleNamespace(stream=lambda: 0, cus=256, name="none"))
    monkeypatch.setattr(wq, "_tile_plan", lambda *args: (0, 0, 0, 0))
    monkeypatch.setattr(wq, "SCRATCH_BYTES", scratch)
    m, n, k = 300, 24, 128
    out = torch.zeros(m + 5, n, dtype=torch.bfloat16)
    y = wq.linear(torch.zeros(m, k, dtype=torch.bfloat16), torch.zeros(n, k, dtype=torch.int8), torch.ones(n), mode=path, out=out)
    assert y is out and written[0][0] == out.data_ptr()
    assert sum(rows for _, rows, _ in written) == m and all(w[2] == n for w in written)
    with pytest.raises(ValueError):
        wq.linear(torch.zeros(m, k, dtype=torch.bfloat16), torch.zeros(n, k, dtype=torch.int8), torch.ones(n), mode=path, out=out[:m - 1])
