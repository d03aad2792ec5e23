"""GPU parity of the mid tiles (variants 16-20, gemm_mid.h) through the C-ABI, against the CPU oracle: every tile shape of
every mode at ragged sizes (tokens, channels and K past whole tiles and k-blocks, odd and even k-block counts), whole K and
split into pieces. The CU count that a call passes steers the shape. row, exact, block and block+g bit for bit in the
oracle's (piece) order; exact+g, whose scaling order the oracle does not have, within a bound from its arithmetic."""
import ctypes

import numpy as np
import pytest
import torch

from conftest import DT, bits, from_bits, gemm_exact64
from test_gpu_gemm import operands

pytestmark = pytest.mark.gpu

MODES = {16: "row", 17: "exact", 18: "block", 19: "block+g", 20: "exact+g"}
# (variant, m, n, k, CUs counted, split): the comment is the tile that this asks for
CASES = [
    (16, 69, 38, 800, 16, 1), (16, 84, 67, 784, 4, 1),        # 64 x 32, 64 x 64
    (16, 135, 68, 800, 4, 0), (16, 130, 166, 784, 4, 1),      # 128 x 64, 128 x 128
    (16, 131, 270, 800, 2, 1), (16, 131, 322, 784, 2, 0),     # 128 x 160, 128 x 192
    (16, 273, 195, 800, 4, 1), (16, 148, 247, 2080, 6, 1),    # 256 x 128; 3 pieces
    (17, 87, 33, 864, 32, 1), (17, 85, 68, 816, 4, 0),        # 64 x 32, 64 x 64
    (17, 141, 195, 864, 3, 1), (17, 166, 65, 800, 4, 0),      # 64 x 128, 128 x 64
    (17, 135, 138, 816, 1, 1),                                # 128 x 128
    (18, 65, 45, 784, 4, 1), (18, 74, 67, 848, 4, 1),         # 64 x 32, 64 x 64
    (18, 146, 68, 784, 4, 0), (18, 139, 149, 848, 4, 1),      # 128 x 64, 128 x 128
    (18, 132, 277, 784, 4, 1), (18, 134, 324, 800, 4, 1),     # 128 x 160, 128 x 192
    (18, 274, 196, 784, 4, 1), (18, 130, 214, 1856, 6, 1),    # 256 x 128; 3 pieces
    (19, 73, 35, 816, 8, 0), (19, 70, 44, 2064, 16, 1),       # 64 x 32; 4 pieces
    (19, 65, 75, 1072, 4, 0), (19, 162, 69, 2080, 32, 1),     # 64 x 64; 4 pieces
    (19, 159, 67, 784, 4, 1), (19, 140, 141, 800, 4, 0),      # 128 x 64, 128 x 128
    (19, 129, 257, 880, 2, 0), (19, 136, 269, 1808, 8, 1),    # 128 x 160; 2 pieces
    (19, 132, 349, 800, 1, 1), (19, 1, 509, 2080, 6, 1),      # 128 x 192; 2 pieces
    (20, 66, 35, 800, 32, 0), (20, 83, 76, 2064, 32, 1),      # 64 x 32; 4 pieces
    (20, 81, 65, 816, 4, 1), (20, 84, 124, 2080, 16, 1),      # 64 x 64; 4 pieces
    (20, 67, 134, 816, 4, 0), (20, 213, 140, 800, 3, 1),      # 64 x 128, 128 x 64
    (20, 132, 131, 848, 1, 1),                                # 128 x 128
    (16, 3, 5, 16, 256, 1), (17, 40, 9, 128, 256, 1), (18, 1, 1, 64, 256, 1), (19, 33, 17, 144, 256, 0), (20, 2, 40, 256, 256, 1),
    (17, 70, 130, 8 * 1024, 256, 1), (18, 97, 260, 12 * 1024, 256, 1),  # 8 pieces
]
# segments: (m, rows of each of three weights, k, CUs counted, side of the square tile, dtype)
SEGMENTS = [(100, 264, 640, 256, 64, torch.bfloat16), (200, 1000, 640, 256, 64, torch.bfloat16), (130, 200, 784, 4, 128, torch.bfloat16),
            (200, 264, 640, 4, 128, torch.float16), (150, 104, 912, 2, 128, torch.float16), (99, 136, 784, 64, 64, torch.float16)]


def mid_plan(m, n, k, variant, cus, split, seg_rows=0):
    """(tokens, channels, K pieces) of the tile that the library gives a mid launch (host only)."""
    from wgpkernels_amd.int8 import _native
    plan = (ctypes.c_int * 3)()
    assert _native.load_test_library().wq8_debug_mid_plan(m, n, k, variant, cus, split, seg_rows, plan) == 0
    return tuple(plan)


def p(t):
    return None if t is None else t.data_ptr()


def run(wq, variant, cu, dtype, cus, split):
    """(outputs, pieces) of one call on the CUDA operands of test_gpu_gemm.operands()."""
    a, a_lo, sa, b, sb, bias, res, rs = cu
    lib = wq.library()
    (m, k), n = a.shape, b.shape[0]
    sizes = (ctypes.c_int64 * 2)()
    lib.wq8_gemm_workspace(m, n, k, variant, cus, split, sizes)
    assert sizes[1] == 0  # no counters: pieces are added by a second launch
    words = 2 if MODES[variant] == "exact" else 1
    pieces = max(1, sizes[0] // (4 * words * m * n)) if sizes[0] else 1
    ws = torch.empty(max(16, sizes[0]), dtype=torch.uint8, device="cuda")
    y = res.clone() if res is not None else torch.empty(m, n, dtype=dtype, device="cuda")
    rc = lib.wq8_gemm(p(a), p(a_lo), p(sa), p(b), p(sb), p(bias), p(y if res is not None else None), p(rs), p(y), m, n, k, DT[dtype], variant,
                      cus, split, p(ws), None, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    return y, pieces


@pytest.mark.parametrize("index", range(len(CASES)), ids=["-".join(map(str, c)) for c in CASES])
def test_mid_tiles_match_oracle(wq, oracle, index):
    variant, m, n, k, cus, split = CASES[index]
    mode = MODES[variant]
    base, groups = mode.removesuffix("+g"), mode.endswith("+g")
    dtype = (torch.bfloat16, torch.float16)[index % 2]
    ops = operands(m, n, k, 300 + index, groups, base == "exact", base == "block", dtype, residual=index % 3 == 0)
    print(f"mid variant={variant} m={m} n={n} k={k} cus={cus} split={split} {dtype}", flush=True)
    y, pieces = run(wq, variant, [None if t is None else t.cuda() for t in ops], dtype, cus, split)
    if not split:
        assert pieces == 1
    a, a_lo, sa, b, sb, bias, res, rs = ops
    np_ = lambda t: None if t is None else t.numpy()
    as_bits = lambda t: None if t is None else bits(t)
    if mode != "exact+g":
        order = "block_biased" if mode == "block" else base
        want = oracle.gemm(np_(a), np_(a_lo), np_(sa), np_(b), np_(sb), as_bits(bias), DT[dtype], order, as_bits(res), as_bits(rs), pieces=pieces)
        np.testing.assert_array_equal(bits(y), want)
        return
    # exact+g: FP32 sums of k-blocks / 128 + pieces terms and five more roundings, each within 2^-24 of the magnitudes
    # added, then one rounding of the output (2^-9 in BF16, 2^-12 in FP16 for results that are not denormal)
    args = (as_bits(bias), dtype, "exact")
    ref = gemm_exact64(np_(a), np_(a_lo), np_(sa), np_(b), np_(sb), *args, as_bits(res), as_bits(rs))
    size = gemm_exact64(np.abs(np_(a)), np.abs(np_(a_lo)), np_(sa), np.abs(np_(b)), np_(sb), None, dtype, "exact")
    if res is not None:
        size = size * np.abs(rs.double().numpy())[None, :] + np.abs(res.double().numpy())
    if bias is not None:
        size = size + np.abs(bias.double().numpy())[None, :]
    bound = 2.0 ** -24 * (-(-k // 128) + pieces + 5) * size + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * np.abs(ref) + 1e-7
    assert (np.abs(from_bits(bits(y), dtype).double().numpy() - ref) <= bound).all()


@pytest.mark.parametrize("path", ["row", "exact", "block"])
@pytest.mark.parametrize("m,rows,k,cus,tile,dtype", SEGMENTS, ids=str)
def test_mid_segments_equal_separate_linears(wq, monkeypatch, path, m, rows, k, cus, tile, dtype):
    """Segments on the mid tiles (64 x 64 and 128 x 128; tiles that straddle two segments): the same bits as one linear per
    weight over whole K, on the mid tile of that shape and on the long tile."""
    assert mid_plan(m, 3 * rows, k, wq.MID_TILES[path], cus, 0, rows) == (tile, tile, 1)
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, k, generator=g).to(dtype).cuda()
    weights = [torch.randint(-127, 128, (rows, k), generator=g, dtype=torch.int8).cuda() for _ in range(3)]
    scales = [((torch.rand(rows, generator=g) + 0.5) / 127).cuda() for _ in range(3)]
    biases = [torch.randn(rows, generator=g).to(dtype).cuda(), None, torch.randn(rows, generator=g).to(dtype).cuda()]
    prepared = wq.prepare(x, 0, path)
    wants = [[wq.gemm(prepared.x, prepared.lo, prepared.scale, w, s, bias, dtype, 0, v) for w, s, bias in zip(weights, scales, biases)]
             for v in (wq.MID_TILES[path], wq.TILES[path][0])]
    monkeypatch.setattr(wq, "_segment_plans", {(path, m, rows, 3, k, 0): (wq.MID_TILES[path], 0)})
    monkeypatch.setattr(wq._native.gpu(x), "cus", cus)
    outputs = [torch.empty(m, rows, dtype=dtype, device="cuda") for _ in range(3)]
    print(f"mid segments {path} m={m} rows={rows} k={k} cus={cus} {dtype}", flush=True)
    wq.linear_prepared_segments(prepared, weights, scales, biases, outputs)
    torch.cuda.synchronize()
    for want in wants:
        assert all(torch.equal(y, w) for y, w in zip(outputs, want))


def test_mid_pieces_replay_in_a_graph(wq):
    """A captured mid launch in pieces (two kernels) replays to the eager bits with new activations."""
    m, n, k = 97, 260, 12 * 1024
    g = torch.Generator(device="cuda").manual_seed(1)
    w = torch.randint(-127, 128, (n, k), device="cuda", generator=g, dtype=torch.int8)
    s = torch.rand(n, device="cuda", generator=g) / 127
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    prepared = wq.prepare(x, 0, "block")
    call = lambda: wq.gemm(prepared.x, None, prepared.scale, w, s, None, torch.bfloat16, 1, wq.MID_TILES["block"])
    call()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            y = call()
    torch.cuda.current_stream().wait_stream(stream)
    for step in range(4):
        fresh = wq.prepare(torch.randn(m, k, device="cuda", generator=g).bfloat16(), 0, "block")
        prepared.x.copy_(fresh.x)
        prepared.scale.copy_(fresh.scale)
        want = call()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), step
