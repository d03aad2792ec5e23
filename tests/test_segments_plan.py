"""linear_prepared_segments(): its tile is timed on the segment launches themselves, apart from a plain GEMM of the joined
shape (CPU, with a recording library and given timings)."""
from types import SimpleNamespace

import pytest
import torch

from wgpkernels_amd import int8 as wq

M, K, ROWS, COUNT = 40, 256, 24, 3


@pytest.fixture
def fake(monkeypatch, tmp_path):
    f = SimpleNamespace(calls=[], microseconds={}, capturing=False)
    variant = lambda name, args: args[12] if name == "wq8_gemm_segments" else args[13]
    f.variants = lambda: [variant(*c) for c in f.calls]
    lib = SimpleNamespace(call=lambda name, *args: f.calls.append((name, args)), wq8_gemm_workspace=lambda *args: None,
                          wq8_gemm_select=lambda *args: 0, has=lambda name: True)

    def time_cold(library, runs, device):
        for r in runs.values():
            r()
        f.timed = [n for n, _ in f.calls], f.variants()
        return {r: f.microseconds[r] for r in runs}

    monkeypatch.setattr(wq, "_lib", lib)
    monkeypatch.setattr(wq, "library", lambda: lib)
    monkeypatch.setattr(wq._native, "gpu", lambda t: SimpleNamespace(stream=lambda: 0, cus=256, name="none"))
    monkeypatch.setattr(wq._tuning, "store", wq._tuning.Store(tmp_path / "store.json"))
    monkeypatch.setattr(wq._tuning, "time_cold", time_cold)
    monkeypatch.setattr(wq._tuning, "is_capturing", lambda: f.capturing)
    monkeypatch.setattr(wq, "_plans", {("block", M, COUNT * ROWS, K, None): (18, 1, 0, 0)})  # a plain GEMM of the joined shape
    monkeypatch.setattr(wq, "_segment_plans", {}, raising=False)
    f.weights = [torch.zeros(ROWS, K, dtype=torch.int8) for _ in range(COUNT)]
    f.scales = [torch.ones(ROWS) for _ in range(COUNT)]
    f.outputs = [torch.zeros(M, ROWS, dtype=torch.bfloat16) for _ in range(COUNT)]
    f.prepared = {"block": wq.Prepared("block", torch.zeros(M, K, dtype=torch.int8), None, torch.ones(M, 2), torch.bfloat16),
                  "exact": wq.Prepared("exact", torch.zeros(M, K, dtype=torch.int8), torch.zeros(M, K, dtype=torch.int8), torch.ones(M), torch.bfloat16)}
    f.run = lambda path="block": wq.linear_prepared_segments(f.prepared[path], f.weights, f.scales, [None] * COUNT, f.outputs)
    return f


@pytest.mark.parametrize("path,tiles,fastest", [("block", [10, 15, 18], 10), ("block", [10, 15, 18], 15), ("exact", [1, 7, 17], 17)])
def test_times_its_own_launches(fake, path, tiles, fastest):
    fake.microseconds = {v: 50.0 - 10 * (v == fastest) for v in tiles}
    assert fake.run(path) is fake.outputs
    assert fake.timed == (["wq8_gemm_segments"] * 3, tiles)
    assert fake.variants()[-1] == fastest and all(args[14] == 0 for _, args in fake.calls)  # split 0, as they run
    fake.calls.clear()
    fake.run(path)  # decided
    assert [n for n, _ in fake.calls] == ["wq8_gemm_segments"] and fake.variants() == [fastest]
    wq._segment_plans.clear()  # and stored
    fake.calls.clear()
    fake.run(path)
    assert fake.variants() == [fastest]


def test_under_capture_nothing_is_timed_or_kept(fake):
    fake.capturing = True
    fake.run()
    assert fake.variants() == [10] and not wq._segment_plans and not wq._tuning.store.entries()


def test_refuses_other_shapes(fake):
    fake.weights[1] = torch.zeros(ROWS + 8, K, dtype=torch.int8)
    with pytest.raises(ValueError):
        fake.run()
    fake.weights[1] = torch.zeros(ROWS, K, dtype=torch.int8)
    fake.scales[2] = torch.ones(ROWS - 1)
    with pytest.raises(ValueError):
        fake.run()
    fake.scales[2] = torch.ones(ROWS)
    fake.prepared["block"].scale = torch.ones(M)
    with pytest.raises(ValueError):
        fake.run()
