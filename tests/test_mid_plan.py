"""The tiles that the mid-tile parity tests run, from the library's own choice (CPU): every tile shape of every mode, and both
tiles of segments."""
import pytest

from test_gpu_mid import CASES, SEGMENTS, mid_plan

WIDE = {(128, 160), (128, 192)}
SHAPES = {(64, 32), (64, 64), (128, 64), (128, 128)}
TILES = {16: SHAPES | WIDE | {(256, 128)}, 17: SHAPES | {(64, 128)}, 18: SHAPES | WIDE | {(256, 128)}, 19: SHAPES | WIDE, 20: SHAPES | {(64, 128)}}


@pytest.fixture(autouse=True)
def test_library():
    from wgpkernels_amd import build
    if not build.library_file("int8_test").exists():
        pytest.skip("test library not built")


@pytest.mark.parametrize("variant", TILES)
def test_every_tile_is_run(variant):
    plans = {mid_plan(m, n, k, v, cus, split) for v, m, n, k, cus, split in CASES if v == variant}
    assert {p[:2] for p in plans} == TILES[variant]
    assert {p[2] > 1 for p in plans} == {True, False}  # whole K and pieces


def test_segments_run_both_tiles():
    for m, rows, k, cus, tile, _ in SEGMENTS:
        for variant in (16, 17, 18):
            assert mid_plan(m, 3 * rows, k, variant, cus, 0, rows) == (tile, tile, 1)
    assert {s[4] for s in SEGMENTS} == {64, 128}
