"""choose_path(): faster GEMM tiles never move a call to a coarser path than the one that the decision rule picks on the
long and short tiles (CPU, with given timings)."""
from types import SimpleNamespace

import pytest
import torch

from wgpkernels_amd import int8 as wq

# path timings on the best tile; exact and block on the long and short tiles; weight groups; precise; the path
CASES = [
    (100, dict(exact=44.7, block=35.9), dict(exact=54.4, block=50.3), False, False, "exact"),       # not 'block'
    (13, dict(small=37.4, exact=35.8, block=36.9), dict(exact=39.7, block=42.2), False, False, "small"),  # not 'exact'
    (13, dict(small=38.4, exact=35.8, block=38.0), dict(exact=37.0, block=39.0), False, False, "small"),  # exact 4% faster
    (13, dict(small=45.0, exact=35.8, block=38.0), dict(exact=37.0, block=39.0), False, False, "exact"),  # exact 20% faster
    (13, dict(small=37.4, exact=35.8), dict(exact=39.7), False, True, "small"),
    (32, dict(small=28.4, exact=30.0, block=20.0), dict(exact=33.0, block=35.0), False, False, "small"),  # not 'block'
    (333, dict(exact=42.1, block=37.2), dict(exact=48.3, block=46.0), True, False, "exact"),
    (256, dict(exact=48.0, block=41.0), dict(exact=59.0, block=45.0), False, False, "block"),       # 'block' on both
    (256, dict(exact=59.0, block=45.4), dict(exact=62.0, block=55.9), False, False, "exact"),       # just past the line
    (256, dict(exact=62.0, block=45.4), dict(exact=62.0, block=55.9), False, False, "block"),       # near, but 11% slower
    (512, dict(exact=27.0, block=24.0), dict(exact=32.7, block=26.2), False, False, "block"),       # well past it and slower
    (16, dict(exact=41.3, block=47.4), dict(exact=68.6, block=51.2), True, False, "exact"),         # finer and no slower
    (100, dict(exact=44.7), dict(exact=54.4), False, True, "exact"),
    (13, dict(small=36.0, exact=20.0), dict(exact=33.0), False, True, "exact"),   # near on the drawn tiles, far on the best
    (13, dict(small=36.0, exact=20.0, block=34.0), dict(exact=33.0, block=34.0), False, False, "exact"),
    (100, dict(exact=50.0, block=25.0), dict(exact=54.0, block=50.0), False, False, "exact"),  # finer on the drawn tiles: stays
    (333, dict(exact=50.0, block=42.0), dict(exact=56.0, block=50.0), False, False, "exact"),  # 'block' before, as fast now
    (333, dict(exact=54.0, block=42.0), dict(exact=59.0, block=50.0), False, False, "block"),  # 18% over it, and slower
    (100, dict(exact=44.7, block=35.5), dict(exact=47.4, block=40.9), False, False, "exact"),  # a faster preparation: 1.08 to 1.16
]


@pytest.mark.parametrize("m,best,drawn,groups,precise,expected", CASES)
def test_no_coarser_than_on_the_drawn_tiles(monkeypatch, tmp_path, m, best, drawn, groups, precise, expected):
    seen = []

    def time_cold(library, runs, device):
        seen.extend(runs)
        # the long and short tiles differ from one another; the fastest of a path stands for it
        return {r: best[r] if isinstance(r, str) else drawn[r[0]] + 3.0 * (r[1] not in (1, 10, 12, 14)) + r[2] for r in runs}

    monkeypatch.setattr(wq._native, "gpu", lambda t: SimpleNamespace(name="none"))
    monkeypatch.setattr(wq, "library", lambda: None)
    monkeypatch.setattr(wq, "_has_weight_groups", lambda scale: scale.dim() == 2)
    monkeypatch.setattr(wq._tuning, "store", wq._tuning.Store(tmp_path / "store.json"))
    monkeypatch.setattr(wq._tuning, "is_capturing", lambda: False)
    monkeypatch.setattr(wq._tuning, "time_cold", time_cold)
    monkeypatch.setattr(wq, "_decided_paths", {})
    w = torch.zeros(64, 256, dtype=torch.int8)
    s = torch.ones(64, 2) if groups else torch.ones(64)
    assert wq.choose_path(torch.zeros(m, 256, dtype=torch.bfloat16), w, s, precise=precise) == expected
    # no tile of the mid kernel is among the drawn ones
    assert not [r for r in seen if not isinstance(r, str) and r[1] in wq.MID_TILES.values()]
