"""Workloads of the INT8 weight linear, as a program that uses the library calls it: decode steps, batched decode, text
contexts, and the long latents of a video model, through the public entry points of wgpkernels_amd.int8.

Three kinds of case:
- "linear": one linear() call;
- "mlp":    the two linears of a feed-forward block, hidden states between them in the model's 16-bit type; with "gated",
            the first one makes [gate | value] rows and the second applies SwiGLU, else it applies GELU;
- "qkv":    one prepare() that serves three weights of the same input: one launch for all of them on the GEMM paths
            (linear_prepared_segments), one linear_prepared() each on the few-token paths.

A case's fields: m tokens, k input and n output channels (of one weight; "mlp": f hidden channels instead of n), dtype,
act (the input operation), rotation (ConvRot group, 0: none), groups (weight scales per channel and 128-element K block
instead of per channel), residual (Y = R + rs * (...)), path (a path forced with mode=; "auto": the library chooses).
"""
import torch

from wgpkernels_amd import int8

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
EPS = 1e-6


def case(name, kind, m, k, n, dtype="bf16", path="auto", act="", rotation=0, groups=False, residual=False, gated=False):
    c = {"kind": kind, "m": m, "k": k, "n": n, "dtype": dtype, "path": path, "act": act, "rotation": rotation, "groups": groups,
         "residual": residual, "gated": gated}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest call: a time embedding or a one-token projection of a small model, all latency
        case("token1_square_1536", "linear", 1, 1536, 1536),
        # one decode step through a feed-forward block of Wan-14B width: the weights of both linears stream from HBM
        case("token1_mlp_5120", "mlp", 1, 5120, 13824, act="rms_norm", residual=True),
        # a few conditioning tokens, odd sizes (K a multiple of 4 only, N odd), FP16
        case("tokens3_ragged_fp16", "linear", 3, 5124, 4999, dtype="fp16", path="lines", residual=True),
        # batched decode through a gated feed-forward block
        case("tokens13_gated_mlp", "mlp", 13, 5120, 13824, gated=True, residual=True),
        # batched decode, one prepared input for the query, key and value projections
        case("tokens32_qkv_fp16", "qkv", 32, 5120, 5120, dtype="fp16", path="small", act="rms_norm"),
        # a short prompt in full precision, weights stored rotated (ConvRot)
        case("tokens100_exact_rotated", "linear", 100, 5120, 5120, dtype="fp16", path="exact", rotation=256),
        # a 512-token text context through a feed-forward block
        case("context512_mlp_block", "mlp", 512, 5120, 13824, path="block", act="rms_norm", residual=True),
        # a ragged context on a checkpoint with group-128 weight scales
        case("context333_group128", "linear", 333, 3072, 12288, path="block", act="swiglu", groups=True, residual=True),
        # per-token INT8 (W8A8), asked for by a program that trades accuracy; ragged in tokens and channels
        case("frames2000_row_rotated", "linear", 2000, 1536, 5000, path="row", rotation=64),
        # fused query, key and value projections of a 4096-token latent in full precision
        case("frames4096_exact_qkv", "qkv", 4096, 5120, 5120, path="exact", act="rms_norm"),
        # group-128 weight scales in full precision over a longer latent
        case("frames8192_group128_exact", "linear", 8192, 3072, 12288, path="exact", act="swiglu", groups=True, residual=True),
        # the largest: the feed-forward block of a 21 x 30 x 52 video latent (32760 tokens)
        case("latent32760_mlp", "mlp", 32760, 5120, 13824, act="rms_norm", residual=True),
    ]


def _log(rng, low, high):
    """An integer whose logarithm is uniform over [low, high]."""
    return max(low, min(high, round(low * (high / low) ** rng.random())))


def draw(rng):
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    span = rng.choice(["few", "few", "mid", "mid", "long"])
    if span == "few":  # decode and batched decode: the few-token kernels
        m = _log(rng, 1, 32)
        kind = rng.choice(["linear", "linear", "mlp", "qkv"])
        k = 64 * _log(rng, 8, 216)
        n = _log(rng, 512, 27648)
        if kind == "linear":
            if m <= 4 and rng.random() < 0.4:  # K a multiple of 4 only
                return case("", kind, m, 4 * _log(rng, 128, 3456), n, dtype, "lines", residual=rng.random() < 0.5)
            act = rng.choice(["", "rms_norm", "gelu", "swiglu"])
            rotation = rng.choice([0, 0, 16, 64])
            return case("", kind, m, k, n, dtype, act=act, rotation=rotation, residual=rng.random() < 0.5)
        if kind == "mlp":
            gated = rng.random() < 0.5
            return case("", kind, m, 64 * _log(rng, 16, 80), 64 * _log(rng, 32, 216), dtype, act=rng.choice(["", "rms_norm"]), residual=True,
                        gated=gated)
        return case("", kind, m, 64 * _log(rng, 16, 80), 8 * _log(rng, 64, 640), dtype, "lines" if m <= 2 else "small", act="rms_norm")
    # prompts, contexts and latents: the GEMM paths
    m = _log(rng, 33, 4096) if span == "mid" else _log(rng, 4097, 16384)
    kind = rng.choice(["linear", "linear", "mlp", "qkv"])
    path = rng.choice(["block", "block", "exact", "row"])
    if kind == "mlp":
        path = "exact" if path == "row" else path
        gated = rng.random() < 0.3
        return case("", kind, m, 64 * _log(rng, 16, 80), 64 * _log(rng, 32, 128), dtype, path, act=rng.choice(["", "rms_norm"]), residual=True,
                    gated=gated)
    if kind == "qkv":
        return case("", kind, m, 64 * _log(rng, 16, 80), 8 * _log(rng, 64, 640), dtype, path, act="rms_norm")
    k = 16 * _log(rng, 32, 864 if span == "mid" else 320)
    n = _log(rng, 512, 13824) if rng.random() < 0.3 else 8 * _log(rng, 64, 1728)
    groups = path != "row" and rng.random() < 0.3
    rotation = rng.choice([0, 16, 64, 256])
    rotation = rotation if rotation and k % rotation == 0 else 0
    return case("", kind, m, k, n, dtype, path, act=rng.choice(["", "rms_norm", "gelu", "swiglu"]), rotation=rotation, groups=groups,
                residual=rng.random() < 0.5)


class _Inputs:
    """Seeded inputs on the GPU: activations N(0, 1) with 1% of the channels 20 times larger where the model's input is
    drawn, weights uniform in [-127, 127], scales that give outputs of unit variance, bias 0.02 N(0, 1)."""

    def __init__(self, c, seed):
        self.c, self.dtype = c, DTYPES[c["dtype"]]
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, scale=1.0, offset=0.0):
        return (torch.randn(*shape, device="cuda", generator=self.gen, dtype=torch.float32 if shape[0] < 4096 else self.dtype) * scale
                + offset).to(self.dtype)

    def tokens(self, m, k):
        x = self.normal(m, k)
        loud = torch.randint(0, k, (max(1, k // 100),), device="cuda", generator=self.gen)
        x[:, loud] *= 20
        return x

    def weight(self, n, k):
        w = torch.randint(-127, 128, (n, k), device="cuda", generator=self.gen, dtype=torch.int8)
        shape = (n, (k + 127) // 128) if self.c["groups"] else (n,)
        s = (torch.rand(*shape, device="cuda", generator=self.gen) + 0.5) / 127 * (3.0 / k) ** 0.5
        return {"w": w, "s": s, "bias": self.normal(n, scale=0.02)}


def prepare(case, seed):
    c, make = case, _Inputs(case, seed)
    m, k, n = c["m"], c["k"], c["n"]
    state = {"case": c, "x": make.tokens(m, 2 * k if c["act"] == "swiglu" else k)}
    if c["act"] == "rms_norm":
        state["norm"] = make.normal(k, scale=0.1, offset=1.0)
    if c["kind"] == "linear":
        state["weights"] = [make.weight(n, k)]
        out = n
    elif c["kind"] == "mlp":
        state["weights"] = [make.weight(2 * n if c["gated"] else n, k), make.weight(k, n)]
        out = k
    else:
        state["weights"] = [make.weight(n, k) for _ in range(3)]
        out = n
    if c["residual"]:
        state["residual"] = make.normal(m, out)
        state["rs"] = make.normal(out, scale=0.1, offset=0.5)
    return state


def _linear(state, x, weight, act, residual):
    c = state["case"]
    return int8.linear(x, weight["w"], weight["s"], weight["bias"], group=c["rotation"], mode=None if c["path"] == "auto" else c["path"],
                       act=act or None, act_weight=state.get("norm") if act == "rms_norm" else None, eps=EPS,
                       residual=state.get("residual") if residual else None, residual_scale=state.get("rs") if residual else None)


def run(state):
    c, x, weights = state["case"], state["x"], state["weights"]
    if c["kind"] == "linear":
        return _linear(state, x, weights[0], c["act"], True)
    if c["kind"] == "mlp":
        hidden = _linear(state, x, weights[0], c["act"], False)
        return {"hidden": hidden, "y": _linear(state, hidden, weights[1], "swiglu" if c["gated"] else "gelu", True)}
    prepared = int8.prepare(x, c["rotation"], c["path"], c["act"] or None, state.get("norm"), EPS)
    if c["path"] in ("lines", "small"):
        return [int8.linear_prepared(prepared, w["w"], w["s"], w["bias"]) for w in weights]
    outputs = [torch.empty(c["m"], c["n"], dtype=x.dtype, device=x.device) for _ in weights]
    return int8.linear_prepared_segments(prepared, [w["w"] for w in weights], [w["s"] for w in weights], [w["bias"] for w in weights], outputs)


def _shapes(c):
    """(input width, K, N) of each linear of the case."""
    wide = 2 if c["act"] == "swiglu" else 1
    if c["kind"] == "linear":
        return [(wide * c["k"], c["k"], c["n"])]
    if c["kind"] == "qkv":
        return [(c["k"], c["k"], c["n"])] * 3
    up = 2 * c["n"] if c["gated"] else c["n"]
    return [(c["k"], c["k"], up), (up, c["n"], c["k"])]


def work(case):
    c, m = case, case["m"]
    shapes = _shapes(c)
    nbytes = flops = 0
    for i, (width, k, n) in enumerate(shapes):
        nbytes += n * k + 4 * n * ((k + 127) // 128 if c["groups"] else 1) + 2 * n + 2 * m * n
        if i == 0 or c["kind"] == "mlp":
            nbytes += 2 * m * width
        flops += 2 * m * n * k
    if c["residual"]:
        nbytes += 2 * m * shapes[-1][2] + 2 * shapes[-1][2]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Outputs are rounded once to 16 bits (relative step 2^-8 in BF16, 2^-11 in FP16). Another order of the FP32 sums flips
    # the last place of a few outputs; the input operation of the few-token paths is rounded to 16 bits too, and rounded
    # hidden states move the INT8 codes of a second linear.
    step = 1.0 if case["dtype"] == "bf16" else 0.125
    if case["kind"] == "mlp":
        return {"rel": 6e-3 if case["dtype"] == "bf16" else 2e-3}
    return {"rel": 4e-3 * step, "max": 0.04 * step}


# ---- the same in 64 bits, without the library --------------------------------------------------------------------------
def _rotate(v, group):
    """ConvRot: groups of `group` values times the Kronecker power of the 4 x 4 matrix of ones with a negated
    anti-diagonal, orthonormal."""
    h4 = torch.ones(4, 4, device=v.device, dtype=v.dtype)
    h4[torch.arange(4), 3 - torch.arange(4)] = -1.0
    h = h4
    while h.shape[0] < group:
        h = torch.kron(h, h4)
    return (v.reshape(-1, group) @ h).reshape(v.shape) / group ** 0.5


def _operation(x, act, norm):
    v = x.double()
    if act == "rms_norm":
        v = v / torch.sqrt(v.square().mean(dim=1, keepdim=True) + EPS)
        return v * norm.double() if norm is not None else v
    if act == "swiglu":
        half = v.shape[1] // 2
        return v[:, :half] * torch.sigmoid(v[:, :half]) * v[:, half:]
    if act == "gelu":
        return 0.5 * v * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (v + 0.044715 * v ** 3)))
    return v


def _codes(v, path):
    """The values that the INT8 codes of a path stand for: one scale per 128 elements (block) or per token (row); the
    full-precision paths keep the value itself."""
    if path not in ("block", "row"):
        return v
    m, k = v.shape
    if path == "block":
        padded = torch.nn.functional.pad(v, (0, -k % 128)).reshape(m, -1, 128)
    else:
        padded = v.reshape(m, 1, k)
    amax = padded.abs().amax(dim=2, keepdim=True)
    codes = torch.where(amax > 0, torch.round(padded * (127.0 / amax)), torch.zeros_like(padded))
    return (codes * (amax / 127.0)).reshape(m, -1)[:, :k]


def _exact_linear(state, x, weight, act, residual):
    c = state["case"]
    path = c["path"] if c["path"] != "auto" else "block" if c["m"] > 4096 else "full"
    v = _operation(x, act, state.get("norm"))
    if c["rotation"]:
        v = _rotate(v, c["rotation"])
    v = _codes(v, path)
    s = weight["s"].double()
    s = torch.repeat_interleave(s, 128, dim=1)[:, :v.shape[1]] if s.dim() == 2 else s[:, None]
    y = v @ (weight["w"].double() * s).t() + weight["bias"].double()
    if residual and "residual" in state:
        y = state["residual"].double() + state["rs"].double() * y
    return y


def exact(case, seed):
    state = prepare(case, seed)
    c, x, weights = case, state["x"], state["weights"]
    if c["kind"] == "linear":
        return _exact_linear(state, x, weights[0], c["act"], True)
    if c["kind"] == "qkv":
        return [_exact_linear(state, x, w, c["act"], False) for w in weights]
    hidden = _exact_linear(state, x, weights[0], c["act"], False)
    # the second linear takes the hidden states in the model's 16-bit type
    rounded = hidden.to(x.dtype)
    return {"hidden": hidden, "y": _exact_linear(state, rounded, weights[1], "swiglu" if c["gated"] else "gelu", True)}
