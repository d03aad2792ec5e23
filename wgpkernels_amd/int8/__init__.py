"""INT8 weight linears on AMD Instinct MI355X (gfx950):

    Y = op(X) @ (W * scales).T + bias            or, with a residual,   Y = R + residual_scale * (...)

W is a checkpoint's INT8 (N, K) matrix, used as stored (never dequantized or copied). scales are FP32 per channel (N,)
or per channel and 128-element K block (N, ceil(K / 128)). op is None, 'rms_norm', 'swiglu' or 'gelu', applied in FP32
while the activation is prepared.

A drop-in for the reference's `wgpkernels.int8` (wgpkernels/int8/__init__.py): the same public functions, arguments,
paths, fusions, errors and autotune behaviour. `from wgpkernels import int8` resolves to this module. The kernels are
hand-written HIP for gfx950 in libwgp_int8.so (built by `python -m wgpkernels_amd.build`), reached through its C-ABI
with ctypes. PyTorch supplies tensors and the current stream. Without the library every call raises: there is no CPU
fallback.

Paths:
- 'lines' (1-4 tokens): HBM-streaming GEMV with the activations unquantized.
- 'small' (up to 32 tokens): the INT8 weights converted exactly to BF16/FP16 on matrix cores.
- 'exact': INT8 matrix cores on x = s * (hi + lo / 254), two passes.
- 'block': one INT8 pass, one FP32 scale per token and 128-element K block.
- 'row': one scale per token (W8A8), on request only.
linear() picks a path per GPU, shape and token-count bucket by timing the candidates once (see choose_path()).
"""
import ctypes
import functools
import time
from contextvars import ContextVar
from pathlib import Path

import torch

from . import _native, _policy, _tuning
from ._native import ptr as _ptr
from ._policy import (DECIDE_MAX_ROWS, EXACT_ROWS, EXACT_TOLERANCE, LINE_MAX_ROWS, LINE_ROWS, SMALL_MAX_ROWS,  # noqa: F401
                      SMALL_ROWS, LinearShape)

# Quantized activations of the GEMM paths are made in row chunks of at most this many bytes. The reference allows
# 16 MiB (wgpkernels/int8/__init__.py:38); MI355X has 288 GB of HBM, so one chunk covers a 32760-token latent at
# K = 5120 and a long linear is one quantize launch and one GEMM launch.
SCRATCH_BYTES = 512 * 1024 * 1024
ACTS = {None: 0, "rms_norm": 1, "swiglu": 2, "gelu": 3}
DTYPES = {torch.float16: 0, torch.bfloat16: 1, torch.float32: 2}
HIP_ARCHS = _native.HIP_ARCHS
# Rows of a chunk are a multiple of the long GEMM tile's token height.
CHUNK_ROW_MULTIPLE = 256

_lib = None
_sizes = (ctypes.c_int64 * 2)()
_tuning_quietly = ContextVar("wgpkernels_amd_int8_tuning_quietly", default=False)


# ---- library --------------------------------------------------------------------------------------------------------
def default_library_path():
    return Path(__file__).with_name("libwgp_int8.so")


def load_library(path=None):
    """Loads libwgp_int8.so (default: the one built next to this file), checks its ABI, binds its entry points,
    allocates each supported GPU's split counters and resolves its allocation-free GEMM array (so that nothing is
    allocated or looked up later under graph capture)."""
    global _lib
    lib = _native.Library(path or default_library_path())
    sizes = (ctypes.c_int64 * 2)()
    for index in _native.supported_gpus():
        _native.gpu(torch.device("cuda", index)).counters
        with torch.cuda.device(index):
            # a workspace query resolves the device's allocation-free GEMM array (no symbol lookup under capture later)
            lib.wq8_gemm_workspace(256, 256, 128, 10, 1, 0, sizes)
    _lib = lib
    return lib


def library():
    """The loaded library, loading the default one on first use."""
    return _lib if _lib is not None else load_library()


def weight_groups_supported():
    """Whether the loaded library takes per-(channel, 128-element K block) weight scales (N, ceil(K / 128))."""
    return _lib is not None and bool(_lib.features & _native.FEATURE_WEIGHT_GROUPS)


def segments_supported():
    """Whether the loaded library runs several linears of one input in one GEMM (linear_prepared_segments)."""
    return _lib is not None and _lib.has("wq8_gemm_segments")


def prepare_stream(stream):
    """Gives `stream` split counters of its own, so that its GEMMs may run at the same time as those of the GPU's other
    streams (which share one set). Call it outside graph capture, before the stream's first call."""
    if stream.cuda_stream not in _native.stream_counters:
        counters = torch.zeros(_native.COUNTER_INTS, dtype=torch.int32, device=stream.device)
        torch.cuda.current_stream(stream.device).synchronize()
        _native.stream_counters[stream.cuda_stream] = counters


# ---- argument checks ----------------------------------------------------------------------------------------------
def _op_width(x, act):
    """K of the linear fed by x: SwiGLU rows hold [gate | value]."""
    return x.shape[1] // 2 if act == "swiglu" else x.shape[1]


def _check_activation(x, aligned=True):
    """2-D with unit column stride; with `aligned`, 16-byte aligned start and row pitch (the quantizers load 16 bytes
    per lane from plain pointers; the few-token kernels load through buffer descriptors and take any pitch)."""
    if x.dim() != 2 or (x.shape[1] > 1 and x.stride(1) != 1):
        raise ValueError("activations must be 2-D with unit column stride")
    if aligned and (x.data_ptr() % 16 or (x.shape[0] > 1 and (x.stride(0) * x.element_size()) % 16)):
        raise ValueError("activation rows must be 16-byte aligned")
    if x.dtype not in DTYPES:
        raise ValueError(f"activations must be FP16, BF16 or FP32, not {x.dtype}")


def _overlap(a, a_values, b, b_values):
    """Whether the first a_values of a and the first b_values of b, read as contiguous, share memory."""
    return (a.data_ptr() < b.data_ptr() + b_values * b.element_size()) and (b.data_ptr() < a.data_ptr() + a_values * a.element_size())


def _row_pitch(x):
    """Elements between rows as the kernels read them. A one-row input's stride is meaningless (PyTorch reports
    (K, 1).t() as contiguous with stride (1, 1)), so its pitch is its width."""
    return x.stride(0) if x.shape[0] > 1 else x.shape[1]


def _is_block_mode(mode, sa):
    return mode.startswith("block") if mode else sa.dim() == 2


def _check_gemm(a, a_lo, sa, b, sb, y, mode):
    """Shapes the GEMM kernels read. They trust their arguments, so a mismatch raises here rather than reading past a
    buffer."""
    (m, k), n = a.shape, b.shape[0]
    kblocks = (k + 127) // 128
    if b.dim() != 2 or b.shape[1] != k or (a_lo is not None and a_lo.shape != a.shape) or tuple(y.shape) != (m, n):
        raise ValueError("INT8 GEMM operand shapes do not match")
    want_sa = m * kblocks if _is_block_mode(mode, sa) else m
    if sa.numel() != want_sa or sb.numel() not in (n, n * kblocks):
        raise ValueError(f"INT8 GEMM scale shapes do not match mode {mode or 'inferred'}: sa {tuple(sa.shape)}, sb {tuple(sb.shape)}")
    if any(t is not None and not t.is_contiguous() for t in (a, a_lo, sa, b, sb, y)):
        raise ValueError("INT8 GEMM operands must be contiguous")


def _has_weight_groups(sb):
    """Whether sb is per (channel, 128-element K block) rather than per channel."""
    if sb.dim() != 2:
        return False
    library()
    if not weight_groups_supported():
        raise RuntimeError("This INT8 library does not take per-(channel, k-block) weight scales; rebuild it")
    return True


# ---- activation preparation (reference: wgpkernels/int8/__init__.py:143-176) ---------------------------------------
def quantize_blocks(x, group=0, act=None, act_weight=None, eps=0.0):
    """INT8 of op(x) (ConvRot-rotated when group > 0) with one FP32 scale per row and 128-element block:
    (q (M, K) int8, scales (M, ceil(K / 128)) float32)."""
    lib = library()
    _check_activation(x)
    m, k = x.shape[0], _op_width(x, act)
    q = x.new_empty((m, k), dtype=torch.int8)
    scale = x.new_empty((m, (k + 127) // 128), dtype=torch.float32)
    # RMSNorm over rows longer than the kernel keeps in registers computes the row norms first
    inv_rms = torch.empty(m, dtype=torch.float32, device=x.device) if act == "rms_norm" and k > 16384 else None
    lib.call("wq8_quantize_blocks", x.data_ptr(), q.data_ptr(), scale.data_ptr(), m, k, _row_pitch(x), DTYPES[x.dtype], group, ACTS[act],
             _ptr(act_weight), eps, _ptr(inv_rms), _native.gpu(x).stream())
    return q, scale


def quantize(x, group=0, hilo=False, act=None, act_weight=None, eps=0.0):
    """Row-wise symmetric INT8 of op(x) (ConvRot-rotated when group > 0): (hi, lo or None, FP32 row scales (M,))."""
    lib = library()
    _check_activation(x)
    m, k = x.shape[0], _op_width(x, act)
    hi = x.new_empty((m, k), dtype=torch.int8)
    lo = torch.empty_like(hi) if hilo else None
    scale = x.new_empty(m, dtype=torch.float32)
    lib.call("wq8_quantize", x.data_ptr(), hi.data_ptr(), _ptr(lo), scale.data_ptr(), m, k, _row_pitch(x), DTYPES[x.dtype], group, ACTS[act],
             _ptr(act_weight), eps, _native.gpu(x).stream())
    return hi, lo, scale


def transform_rows(x, group=0, act=None, act_weight=None, eps=0.0):
    """op(x), ConvRot-rotated, rounded once to x's dtype: the unquantized activation of the few-token paths."""
    lib = library()
    _check_activation(x)
    m, k = x.shape[0], _op_width(x, act)
    out = x.new_empty((m, k))
    lib.call("wq8_transform_rows", x.data_ptr(), out.data_ptr(), m, k, _row_pitch(x), DTYPES[x.dtype], group, ACTS[act], _ptr(act_weight), eps,
             _native.gpu(x).stream())
    return out


def rotate_groups(x, group):
    """ConvRot rotation (groups of 16, 64 or 256), rounded once to the input dtype."""
    lib = library()
    _check_activation(x)
    out = x.new_empty(x.shape)
    lib.call("wq8_rotate_groups", x.data_ptr(), out.data_ptr(), x.shape[0], x.shape[1], _row_pitch(x), DTYPES[x.dtype], group,
             _native.gpu(x).stream())
    return out


# ---- GEMM tiles (reference: wgpkernels/int8/__init__.py:179-329) ------------------------------------------------------
# Variant ids keep the reference's modes (its int8_gemm.cu:1417-1432); the tiles behind them are this library's.
# Per mode: (long-tile variant, short-tile variant or None). The timed choice compares both, whole tiles only (split 0)
# and with the split-K tail (split 1: the tiles of an incomplete last wave split along K), as the reference times its
# stream-K (wgpkernels/int8/__init__.py:180-183).
# The block mode's 10 and 15 are its tiles with the single-FMA biased fold (15, the short one, is an id the reference does
# not use); 11 is the short tile in the reference's fold order.
TILES = {"row": (0, 6), "exact": (1, 7), "block": (10, 15), "block+g": (12, 13), "exact+g": (14, None)}
# Per mode: the tiles for launches of about one tile per CU (ids the reference does not use). They were faster than the
# short tiles at every shape measured (M = 1-2000, K = 1536-13824, N = 1536-13824: by 3-100%) but four, which were within 1.5%
# (M = 1-128 row and exact), so the timed choice compares them with the long ones; the short tiles run when asked for by id,
# untimed, in the path choice (_drawn_runs) and in segments, which have two of the mid tiles only.
MID_TILES = {"row": 16, "exact": 17, "block": 18, "block+g": 19, "exact+g": 20}
VARIANT_MODES = {0: "row", 2: "row", 6: "row", 1: "exact", 7: "exact", 10: "block", 11: "block", 12: "block+g", 13: "block+g",
                 14: "exact+g", 15: "block", **{v: mode for mode, v in MID_TILES.items()}}


def tile_candidates(mode):
    """(variant, split) pairs the tile choice times for `mode`: the untimed default first."""
    return [(v, split) for v in (TILES[mode][0], MID_TILES[mode]) for split in (1, 0)]


def _timed_tiles(mode, m, n, cus):
    """tile_candidates(), without the mid tiles where the long tiles (about 256 x 192) fill the CUs twice over: from there
    on the long ones are faster (M = 2000, N = 13824: by 20-35% in every mode)."""
    long_only = m * n > 2 * cus * 256 * 192
    return [c for c in tile_candidates(mode) if not (long_only and c[0] == MID_TILES[mode])]


def _untimed_tile(mode, m, n, k, cus):
    """Tile of a shape nobody has timed yet (under capture): the library's wave-count estimate, with the split-K tail
    (as the reference's untimed choice, wgpkernels/int8/__init__.py:273-276)."""
    long_v, short_v = TILES[mode]
    base = "exact" if mode.startswith("exact") else "row"
    short = library().wq8_gemm_select(m, n, k, base == "exact", cus) in (6, 7)
    return (short_v if short and short_v is not None else long_v), 1


def _choose_tile(mode, timings, m, n, k, cus):
    """The fastest of the timed (variant, split) pairs; in the modes that fold in FP32 by _policy.decide_tile()."""
    if mode in ("row", "exact"):  # INT32 sums: the same bits in every tile and split
        return min(timings, key=timings.get)
    own, mid = None, (MID_TILES[mode], 1)
    if mode != "exact+g" and mid in timings:  # (the mid exact+g tile scales in an order of its own, split or not)
        library().wq8_gemm_workspace(m, n, k, mid[0], cus, 1, _sizes)
        own = mid if _sizes[0] else None  # planes of partial sums: K pieces of its own
    return _policy.decide_tile(timings, own)


# (mode, M, N, K, device) -> (variant, split, slot bytes, counter bytes) of decided shapes
_plans = {}


def _tile_plan(a, a_lo, sa, b, sb, bias, y, mode, output_is_residual):
    (m, k), n = a.shape, b.shape[0]
    shape = (mode, m, n, k, b.device.index)
    plan = _plans.get(shape)
    if plan is not None:
        return plan
    state = _native.gpu(b)
    key = f"{mode}|{_tuning.gemm_rows_bucket(m)}x{n}x{k}|{state.name}"
    choice = _tuning.store.get(key)
    decided = choice is not None
    if choice is None and _tuning.is_capturing():
        choice = _untimed_tile(mode, m, n, k, state.cus)
    elif choice is None:
        # the timing writes its outputs: never into an output that is also the residual
        scratch = torch.empty_like(y) if output_is_residual else y
        label = f"INT8 GEMM {mode} {m}x{n}x{k}"
        loud = not _tuning_quietly.get()
        if loud:
            print(f"[WGPKernels] Autotuning {label}...", flush=True)
        started = time.time()
        runs = {c: (lambda c: lambda: gemm(a, a_lo, sa, b, sb, bias, y.dtype, c[1], c[0], scratch))(c) for c in _timed_tiles(mode, m, n, state.cus)}
        timings = _tuning.time_cold(library(), runs, b.device)
        choice = _choose_tile(mode, timings, m, n, k, state.cus)
        _tuning.store.put(key, list(choice))
        decided = True
        if loud:
            print(f"[WGPKernels] Selected {label}: tiles {choice[0]}, split {choice[1]} ({timings[choice] * 1000:.1f} us; "
                  f"tuned in {time.time() - started:.2f} s).", flush=True)
    variant, split = choice
    library().wq8_gemm_workspace(m, n, k, variant, state.cus, split, _sizes)
    plan = (variant, split, _sizes[0], _sizes[1])
    if decided:
        _plans[shape] = plan
    return plan


def _workspace(device, slot_bytes, counter_bytes, raw_stream):
    slots = torch.empty(slot_bytes, dtype=torch.uint8, device=device) if slot_bytes else None
    counters = _native.counters_for(_native.gpu(device), raw_stream, counter_bytes).data_ptr() if counter_bytes else None
    return slots, counters


def gemm(a, a_lo, sa, b, sb, bias, out_dtype, split=None, variant=None, out=None, mode=None, residual=None, residual_scale=None):
    """Y = epilogue(A @ B.T) of prepared INT8 activations. mode 'row' (sa per row), 'exact' (a_lo given) or 'block' (sa
    per row and 128-element block), inferred when omitted; sb per channel (N) or per (channel, K block) with 'exact' /
    'block'. residual (M, N) and residual_scale (N) in out_dtype: Y = residual + residual_scale * (A @ B.T + bias); out
    may be the residual. variant forces a tile configuration (no tuning), with split 0 (whole tiles) or 1 (the tiles of an
    incomplete last wave split along K, their partial sums added by the last piece to finish)."""
    lib = library()
    m, k = a.shape
    n = b.shape[0]
    y = a.new_empty((m, n), dtype=out_dtype) if out is None else out
    forced = variant is not None
    if forced and variant not in VARIANT_MODES:
        raise ValueError(f"unknown INT8 GEMM variant {variant}")
    _check_gemm(a, a_lo, sa, b, sb, y, VARIANT_MODES[variant] if forced else mode)
    state = _native.gpu(a)
    if forced:
        split = split or 0
        lib.wq8_gemm_workspace(m, n, k, variant, state.cus, split, _sizes)
        slot_bytes, counter_bytes = _sizes[0], _sizes[1]
    else:
        mode = mode or ("exact" if a_lo is not None else "block" if sa.dim() == 2 else "row")
        if _has_weight_groups(sb):
            if mode == "row":
                raise ValueError("Weights with per-(n, k-block) scales run the 'block' or 'exact' path")
            mode += "+g"
        variant, split, slot_bytes, counter_bytes = _tile_plan(a, a_lo, sa, b, sb, bias, y, mode, residual is not None)
    stream = state.stream()
    slots, counters = _workspace(a.device, slot_bytes, counter_bytes, stream)
    lib.call("wq8_gemm", a.data_ptr(), _ptr(a_lo), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), _ptr(bias), _ptr(residual), _ptr(residual_scale),
             y.data_ptr(), m, n, k, DTYPES[out_dtype], variant, state.cus, split, _ptr(slots), counters, stream)
    return y


# ---- few-token paths (reference: wgpkernels/int8/__init__.py:332-353) --------------------------------------------------
def small(x, weight, scale, bias=None, residual=None, residual_scale=None, out=None):
    """Up to 32 tokens, unquantized activations: INT8 weights converted exactly to 16-bit on matrix cores, FP32
    accumulation. K a multiple of 64."""
    lib = library()
    _check_activation(x, aligned=False)
    m, k = x.shape
    n = weight.shape[0]
    state = _native.gpu(x)
    y = x.new_empty((m, n)) if out is None else out
    lib.wq8_small_workspace(m, n, k, state.cus, _sizes)
    stream = state.stream()
    slots, counters = _workspace(x.device, _sizes[0], _sizes[1], stream)
    lib.call("wq8_small", x.data_ptr(), _row_pitch(x), weight.data_ptr(), scale.data_ptr(), _ptr(bias), _ptr(residual), _ptr(residual_scale),
             y.data_ptr(), m, n, k, DTYPES[x.dtype], state.cus, _ptr(slots), counters, stream)
    return y


def gemv_lines(x, weight, scale, bias=None, residual=None, residual_scale=None, out=None):
    """One to four tokens, unquantized activations: FP32 GEMV streaming the weight rows. K a multiple of 4."""
    lib = _lib if _lib is not None else load_library()
    _check_activation(x, aligned=False)
    m, k = x.shape
    y = x.new_empty((m, weight.shape[0])) if out is None else out
    lib.call("wq8_gemv_lines", x.data_ptr(), _row_pitch(x), weight.data_ptr(), scale.data_ptr(), _ptr(bias), _ptr(residual),
             _ptr(residual_scale), y.data_ptr(), m, weight.shape[0], k, DTYPES[x.dtype], _native.gpu(x).stream())
    return y


# One token with an input operation: applied in the GEMV's own launch for weights of at most this many values and K at most
# this wide, where that is faster than preparing it apart (fewtoken.hip, gemv_line_act).
LINE_ACT_MAX_WEIGHTS, LINE_ACT_MAX_K = 5120 * 5120, 5120


def _line_act(x, weight, scale, bias, act, act_weight, eps, residual, residual_scale, out):
    """linear() of one token through wq8_gemv_line_act, or None where it does not apply (then transform_rows and gemv_lines
    run, with the same bits)."""
    n, k = weight.shape
    if (x.shape[0] != 1 or scale.dim() != 1 or k > LINE_ACT_MAX_K or n * k > LINE_ACT_MAX_WEIGHTS or k % 16 or x.dtype == torch.float32
            or _op_width(x, act) != k or not library().has("wq8_gemv_line_act")):
        return None
    # written in place of its input (a residual stream x = x + rs * linear(op(x))): every workgroup reads x while others store
    if out is not None and _overlap(x, x.shape[1], out, n):
        return None
    _check_activation(x)
    y = x.new_empty((1, n)) if out is None else out
    _lib.call("wq8_gemv_line_act", x.data_ptr(), ACTS[act], _ptr(act_weight), eps, weight.data_ptr(), scale.data_ptr(), _ptr(bias), _ptr(residual),
              _ptr(residual_scale), y.data_ptr(), n, k, DTYPES[x.dtype], _native.gpu(x).stream())
    return y


# ---- prepared activations (reference: wgpkernels/int8/__init__.py:367-430) ----------------------------------------------
class Prepared:
    """An activation prepared for one path: unquantized (transformed, rotated) rows for 'lines' / 'small', INT8 rows and
    scales for 'exact' / 'block' / 'row'. One preparation serves every weight of the same K; rows() is a view."""
    __slots__ = ("path", "x", "lo", "scale", "dtype")

    def __init__(self, path, x, lo, scale, dtype):
        self.path, self.x, self.lo, self.scale, self.dtype = path, x, lo, scale, dtype

    def rows(self, start, stop):
        return Prepared(self.path, self.x[start:stop], None if self.lo is None else self.lo[start:stop],
                        None if self.scale is None else self.scale[start:stop], self.dtype)


def prepare(x, group=0, path="block", act=None, act_weight=None, eps=0.0):
    """op(x) prepared once for `path` (see choose_path()); x 2-D BF16/FP16 with 16-byte aligned rows, act_weight in
    x's dtype."""
    if path in ("lines", "small"):
        # the few-token kernels read 16-bit activations as they are: op and rotation are applied once, rounded to x's dtype
        if act:
            values = transform_rows(x, group, act, act_weight, eps)
        else:
            values = rotate_groups(x, group) if group else x
        return Prepared(path, values, None, None, x.dtype)
    if path == "block":
        q, scale = quantize_blocks(x, group, act, act_weight, eps)
        return Prepared(path, q, None, scale, x.dtype)
    if path in ("exact", "row"):
        hi, lo, scale = quantize(x, group, path == "exact", act, act_weight, eps)
        return Prepared(path, hi, lo, scale, x.dtype)
    raise ValueError(f"unknown INT8 path {path!r}")


def linear_prepared(prepared, weight, scale, bias=None, residual=None, residual_scale=None, out=None):
    """Y = prepared @ (weight * scale).T + bias (or residual + residual_scale * (...)); weight an INT8 (N, K) matrix or a
    row range of one."""
    if prepared.path in ("lines", "small"):
        if scale.dim() == 2:
            raise ValueError("Weights with per-(n, k-block) scales run the 'block' or 'exact' path")
        kernel = gemv_lines if prepared.path == "lines" else small
        return kernel(prepared.x, weight, scale, bias, residual, residual_scale, out)
    return gemm(prepared.x, prepared.lo, prepared.scale, weight, scale, bias, prepared.dtype, out=out, mode=prepared.path, residual=residual,
                residual_scale=residual_scale)


# (mode, M, rows of a weight, weights, K, device) -> (variant, workspace bytes) of decided segment launches
_segment_plans = {}


def _segments_plan(prepared, weights, scales, launch):
    """The tile of a segments launch: its own launches timed (launch(variant, workspace bytes)), whole tiles only, as they
    run. A plain GEMM of the joined shape does not stand for them: it has every mid tile and K pieces, segments have the
    square mid tiles over whole K (us, block, 3 x 5120 channels, K = 5120, M = 333: long 51, mid 63, short 76; row, 3 x 1536,
    K = 1536, M = 200: short 13.0, mid 14.6, long 28.6: the short tiles are candidates here)."""
    mode, (m, k), count, rows = prepared.path, prepared.x.shape, len(weights), weights[0].shape[0]
    state = _native.gpu(prepared.x)
    kblocks, want = (k + 127) // 128, m * ((k + 127) // 128) if mode == "block" else m
    if (any(tuple(w.shape) != (rows, k) for w in weights) or any(s.numel() not in (rows, rows * kblocks) for s in scales)
            or prepared.scale.numel() != want):
        raise ValueError("INT8 GEMM segment shapes do not match")
    if not (prepared.x.is_contiguous() and prepared.scale.is_contiguous() and (prepared.lo is None or prepared.lo.is_contiguous())):
        raise ValueError("INT8 GEMM operands must be contiguous")

    def workspace_bytes(variant):
        library().wq8_gemm_workspace(m, count * rows, k, variant, state.cus, 0, _sizes)
        return _sizes[0]

    key = f"{mode}+seg{count}|{_tuning.gemm_rows_bucket(m)}x{count * rows}x{k}|{state.name}"
    variant = _tuning.store.get(key)
    decided = variant is not None
    if not decided and _tuning.is_capturing():
        variant = _untimed_tile(mode, m, count * rows, k, state.cus)[0]
    elif not decided:
        label = f"INT8 GEMM {mode} {m}x({count}x{rows})x{k}"
        loud = not _tuning_quietly.get()
        if loud:
            print(f"[WGPKernels] Autotuning {label}...", flush=True)
        started = time.time()
        candidates = [v for v in (*TILES[mode], MID_TILES[mode]) if v is not None]
        timings = _tuning.time_cold(library(), {v: functools.partial(launch, v, workspace_bytes(v)) for v in candidates}, prepared.x.device)
        variant = min(timings, key=timings.get)
        _tuning.store.put(key, variant)
        decided = True
        if loud:
            print(f"[WGPKernels] Selected {label}: tiles {variant} ({timings[variant] * 1000:.1f} us; tuned in {time.time() - started:.2f} s).",
                  flush=True)
    plan = (variant, workspace_bytes(variant))
    if decided:
        _segment_plans[(mode, m, rows, count, k, prepared.x.device.index)] = plan
    return plan


def linear_prepared_segments(prepared, weights, scales, biases, outputs):
    """outputs[s] = prepared @ (weights[s] * scales[s]).T + biases[s] for 1 to 4 linears in one GEMM launch ('exact',
    'block' or 'row' preparations, per-channel scales, equal row counts that are multiples of 8). The input is read once
    for all of them; the tile is timed on these launches once per shape."""
    lib = library()
    if not segments_supported():
        raise RuntimeError("the loaded INT8 library has no wq8_gemm_segments")
    a, count, rows = prepared.x, len(weights), weights[0].shape[0]
    m, k = a.shape
    state = _native.gpu(a)
    table = lambda tensors: (ctypes.c_void_p * 4)(*[_ptr(t) for t in tensors])
    tables = table(weights), table(scales), table(biases), table(outputs)

    def launch(variant, workspace_bytes):
        stream = state.stream()
        slots, _ = _workspace(a.device, workspace_bytes, 0, stream)
        lib.call("wq8_gemm_segments", a.data_ptr(), _ptr(prepared.lo), prepared.scale.data_ptr(), *tables, count, rows, m, k,
                 DTYPES[prepared.dtype], variant, state.cus, 0, _ptr(slots), None, stream)

    plan = _segment_plans.get((prepared.path, m, rows, count, k, a.device.index))
    launch(*(plan if plan is not None else _segments_plan(prepared, weights, scales, launch)))
    return outputs


# ---- linear (reference: wgpkernels/int8/__init__.py:433-520) ----------------------------------------------------------
def chunk_rows(mode, k):
    """Token rows per chunk of a GEMM path: the chunk's quantized activations stay within SCRATCH_BYTES."""
    kblocks = (k + 127) // 128
    row_bytes = {"exact": 2 * k + 4, "block": k + 4 * kblocks}.get(mode, k + 4)
    return max(CHUNK_ROW_MULTIPLE, SCRATCH_BYTES // row_bytes // CHUNK_ROW_MULTIPLE * CHUNK_ROW_MULTIPLE)


def _gemm_linear(path, x, weight, scale, bias, group, act, act_weight, eps, residual, residual_scale, out):
    m = x.shape[0]
    y = x.new_empty((m, weight.shape[0])) if out is None else out
    step = chunk_rows(path, weight.shape[1])
    if m <= step:  # one chunk: no row views (about a microsecond of host time each) but of an output with more rows
        if m:
            linear_prepared(prepare(x, group, path, act, act_weight, eps), weight, scale, bias, residual, residual_scale,
                            y if y.shape[0] == m else y[:m])
        return y
    for start in range(0, m, step):
        stop = min(m, start + step)
        prepared = prepare(x[start:stop], group, path, act, act_weight, eps)
        linear_prepared(prepared, weight, scale, bias, None if residual is None else residual[start:stop], residual_scale, y[start:stop])
    return y


def _run_path(path, x, weight, scale, bias, group, act=None, act_weight=None, eps=0.0, residual=None, residual_scale=None, out=None):
    if path in ("lines", "small"):
        if act and path == "lines" and not group:
            y = _line_act(x, weight, scale, bias, act, act_weight, eps, residual, residual_scale, out)
            if y is not None:
                return y
        return linear_prepared(prepare(x, group, path, act, act_weight, eps), weight, scale, bias, residual, residual_scale, out)
    return _gemm_linear(path, x, weight, scale, bias, group, act, act_weight, eps, residual, residual_scale, out)


def _drawn_runs(paths, x, weight, scale, bias, group, act, act_weight, eps):
    """(path, variant, split) -> a run of each GEMM path of `paths` on the fastest of its long and short tiles: what the path
    choice is decided on (_policy.decide_no_coarser). The tiles are timed on the bare GEMM first, as a tile choice does, so
    that as many whole linears are timed against each other as there are paths: each more among them makes the others'
    later launches start colder (up to 5% for a path of several launches)."""
    m, k = x.shape[0], weight.shape[1]
    suffix = "+g" if _has_weight_groups(scale) else ""

    def run(path, variant, split):
        step = chunk_rows(path, k)
        for start in range(0, m, step):
            p = prepare(x[start:start + step], group, path, act, act_weight, eps)
            gemm(p.x, p.lo, p.scale, weight, scale, bias, p.dtype, split, variant)

    def fastest(path):
        chunk = functools.cache(lambda: prepare(x[:chunk_rows(path, k)], group, path, act, act_weight, eps))
        tiles = [(path, v, split) for v in TILES[path + suffix] if v is not None for split in (1, 0)]

        def one(_, variant, split):
            p = chunk()  # prepared once, by the first untimed run
            gemm(p.x, p.lo, p.scale, weight, scale, bias, p.dtype, split, variant)

        timings = _tuning.time_cold(library(), {t: functools.partial(one, *t) for t in tiles}, x.device)
        return min(timings, key=timings.get)

    return {t: functools.partial(run, *t) for t in (fastest(p) for p in paths if p in ("exact", "block"))}


_decided_paths = {}  # (m, n, k, group, act, precise, weight groups, device index) -> path


def choose_path(x, weight, scale, bias=None, group=0, precise=False, act=None, act_weight=None, eps=0.0):
    """The path linear() takes: the fastest full-precision path while it costs at most EXACT_TOLERANCE more than 'block'
    (always a full-precision one with precise=True), decided with the GEMM paths on the long and short tiles, never a coarser
    one for a faster tile (_policy.decide_no_coarser). Timed once per GPU, shape, input operation and token-count bucket on
    this call's input, with cold caches, and cached; a fixed rule applies where nothing may be timed."""
    m, k, n = x.shape[0], weight.shape[1], weight.shape[0]
    if m > DECIDE_MAX_ROWS and not precise:
        return "block"
    weight_groups = _has_weight_groups(scale)
    # a plain tuple: a decided call returns here without building the shape object (host time of a decode step)
    memo = (m, n, k, group, act, precise, weight_groups, x.get_device())
    path = _decided_paths.get(memo)
    if path is not None:
        return path
    shape = LinearShape(m, n, k, group, act, precise, weight_groups)
    state = _native.gpu(x)
    key = shape.key(_tuning.path_rows_bucket(m), state.name)
    path = _tuning.store.get(key)
    if path is None:
        if _tuning.is_capturing():
            return shape.untimed()
        label = (f"INT8 path {m}x{n}x{k}{f' ConvRot {group}' if group else ''}{f' {act}' if act else ''}"
                 f"{' (precise)' if precise else ''}")
        print(f"[WGPKernels] Autotuning {label}...", flush=True)
        started = time.time()
        quiet = _tuning_quietly.set(True)
        try:
            runs = {p: (lambda p: lambda: _run_path(p, x, weight, scale, bias, group, act, act_weight, eps))(p) for p in shape.candidates()}
            timings = drawn = _tuning.time_cold(library(), runs, x.device)
            if len(runs) > 1:
                few = {p: run for p, run in runs.items() if p in ("lines", "small")}
                drawn = _tuning.time_cold(library(), {**few, **_drawn_runs(runs, x, weight, scale, bias, group, act, act_weight, eps)}, x.device)
                drawn = {r if isinstance(r, str) else r[0]: t for r, t in drawn.items()}
        finally:
            _tuning_quietly.reset(quiet)
        path = _policy.decide_no_coarser(timings, drawn, precise)
        _tuning.store.put(key, path)
        print(f"[WGPKernels] Selected {label}: {path} ({timings[path] * 1000:.1f} us; tuned in {time.time() - started:.2f} s).", flush=True)
    _decided_paths[memo] = path
    return path


def linear(x, weight, scale, bias=None, group=0, precise=False, mode=None, act=None, act_weight=None, eps=0.0, residual=None,
           residual_scale=None, out=None):
    """Y = op(X) @ (INT8 weight * FP32 scales).T + bias for 2-D BF16/FP16 X (16-byte aligned rows, unit column stride), or
    residual + residual_scale * (...) (X's dtype; out may be the residual). act: None, 'rms_norm' (act_weight: K values
    in X's dtype or None; eps), 'swiglu' (X rows [gate | value]) or 'gelu' (tanh approximation). mode forces a path
    ('lines', 'small', 'exact', 'block', 'row'); otherwise choose_path() decides."""
    path = mode or choose_path(x, weight, scale, bias, group, precise, act, act_weight, eps)
    return _run_path(path, x, weight, scale, bias, group, act, act_weight, eps, residual, residual_scale, out)


from ._selftest import reference_linear as _reference, reference_rotation as _reference_rotation, selftest  # noqa: E402,F401
