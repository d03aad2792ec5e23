"""Which path serves a linear: the timed choice between the full-precision paths and 'block', and the fixed rule used
where nothing may be timed (graph capture, compilation); and which of a mode's timed tiles a GEMM runs (decide_tile).

The rule is the reference's (wgpkernels/int8/__init__.py:453-509): take the fastest full-precision path ('lines',
'small', 'exact') while it costs at most EXACT_TOLERANCE more than 'block', else 'block'; precise=True never takes
'block'; above DECIDE_MAX_ROWS tokens 'block' is taken untimed. Per-(channel, k-block) weight scales leave 'exact' as
the only full-precision path. It is applied to the long and short tiles' times (decide_no_coarser): where a mid tile makes
'block' faster than that, a full-precision path can cost more than EXACT_TOLERANCE over the 'block' it leaves.

The fixed rule's thresholds are MI355X measurements, not the reference's RTX 5090 ones: with cold weights 'lines' is
the fastest path up to 4 tokens and 'small' up to 32 at the Wan widths (K, N in {5120, 13824}), where 'exact' (two
INT8 passes plus a quantize launch) was 20-45% slower.
"""
from dataclasses import dataclass

EXACT_TOLERANCE = 0.10
DRAWN_BAND = 0.06  # see decide_no_coarser()
WHOLE_MARGIN, ORDER_MARGIN = 0.02, 0.10  # see decide_tile()
# few-token kernel limits (their C-ABI bounds) and the alignment their loads need
LINE_MAX_ROWS, SMALL_MAX_ROWS = 4, 32
LINE_K_MULTIPLE, SMALL_K_MULTIPLE = 4, 64
# the untimed rule: lines up to LINE_ROWS tokens, small up to SMALL_ROWS, exact up to EXACT_ROWS, then block
LINE_ROWS, SMALL_ROWS, EXACT_ROWS = 4, 32, 64
DECIDE_MAX_ROWS = 4096


@dataclass(frozen=True)
class LinearShape:
    """What a path decision depends on besides the GPU."""
    m: int
    n: int
    k: int
    group: int = 0
    act: str = None
    precise: bool = False
    weight_groups: bool = False

    def few_token_ok(self, max_rows, k_multiple):
        return not self.weight_groups and self.m <= max_rows and self.k % k_multiple == 0

    def candidates(self):
        """Paths the timed choice compares, full-precision ones first."""
        paths = []
        if self.few_token_ok(LINE_MAX_ROWS, LINE_K_MULTIPLE):
            paths.append("lines")
        if self.few_token_ok(SMALL_MAX_ROWS, SMALL_K_MULTIPLE):
            paths.append("small")
        paths.append("exact")
        if not self.precise:
            paths.append("block")
        return paths

    def untimed(self):
        """The fixed rule."""
        if self.few_token_ok(LINE_ROWS, LINE_K_MULTIPLE):
            return "lines"
        if self.few_token_ok(SMALL_ROWS, SMALL_K_MULTIPLE):
            return "small"
        return "exact" if self.precise or self.m <= EXACT_ROWS else "block"

    def key(self, rows_bucket, device_name):
        """Cache key, in the reference's format (wgpkernels/int8/__init__.py:485-486)."""
        parts = [f"path{'+precise' if self.precise else ''}", f"{rows_bucket}x{self.n}x{self.k}", f"g{self.group}"]
        if self.act:
            parts.append(self.act)
        if self.weight_groups:
            parts.append("wgroups")
        parts.append(device_name)
        return "|".join(parts)


def decide(timings, precise):
    """The path of measured `timings` (path -> ms): the fastest full-precision path unless it costs more than
    (1 + EXACT_TOLERANCE) x 'block'."""
    full = {p: t for p, t in timings.items() if p != "block"}
    best = min(full, key=full.get)
    if not precise and "block" in timings and full[best] > (1 + EXACT_TOLERANCE) * timings["block"]:
        return "block"
    return best


def decide_no_coarser(timings, drawn, precise):
    """decide() on `drawn`, the timings with the GEMM paths on the long and short tiles, for which the line between the
    paths was drawn. Tiles that are faster for some sizes make a call faster but never coarser: decided on the best
    tiles (`timings`), 19 of 133 shapes (M = 64-2000, K 1536-13824, N 1536-27648) went from 'exact' to 'block' (M = 100,
    K = 13824, N = 5120: exact 54.4 and block 50.3 us on the drawn tiles, 44.7 and 35.9 on the best) and two from
    'small' to 'exact'. So the path taken may be slower than another one is now, but not than what ran on the drawn tiles:
    - 'block' gives way to a full-precision path whose best tile costs no more than the drawn 'block'. Near the line
      (DRAWN_BAND) one within EXACT_TOLERANCE of it will do: a faster preparation takes more of 'block' than of 'exact' and
      so moves their ratio past the line (M = 100, K = 13824, N = 5120, gelu: 54.4 / 50.3 us = 1.08 became 47.4 / 40.9 =
      1.16). Of 560 shapes timed three times, 11 of 1608 choices were coarser than before the faster preparations without a
      band, 4 with 0.03, 2 with 0.06 and 0.08; what the band of 0.06 adds measured at most 1% slower than before.
    - 'lines' and 'small' read the inputs as they are, where 'exact' makes hi/lo codes of them: it takes their place only
      when more than EXACT_TOLERANCE faster, on the drawn or on the best tiles (the two are within 3% at M = 8-32, K = 5120,
      N = 27648, and a faster preparation alone turned them: the error of a gated feed-forward block of 13 tokens went from
      2.2e-3 to 2.5e-3)."""
    path = decide(drawn, precise)
    if path == "exact":
        within = lambda p, times: times[p] <= (1 + EXACT_TOLERANCE) * times["exact"]
        near = {p: t for p, t in drawn.items() if p in ("lines", "small") and within(p, drawn) and within(p, timings)}
        return min(near, key=near.get, default=path)
    if path == "block":
        full = {p: t for p, t in timings.items() if p != "block"}
        best = min(full, key=full.get)
        drawn_full = min(t for p, t in drawn.items() if p != "block")
        near = drawn_full <= (1 + EXACT_TOLERANCE + DRAWN_BAND) * drawn["block"]
        if full[best] <= (1 + (EXACT_TOLERANCE if near else 0)) * drawn["block"]:
            return best
    return path


def decide_tile(timings, own_order=None):
    """The tile of measured `timings` ((variant, split) -> ms) of a mode that folds in FP32, where the order of the sums
    shows in the last bits: the fastest, but whole K (split 0, the same order in every tile) unless the same tile's split is
    more than WHOLE_MARGIN faster, and `own_order`, a candidate in K pieces that no other one has, only when it is more than
    ORDER_MARGIN faster than the rest. A tile whose split gains nothing then gives the same bits in every process: at M =
    32760, K = 13824, N = 5120 split 0 and 1 are 0.6-1.5% apart (1992 / 2003 us), and which one timing calls faster changes.
    At M = 512 there the mid tile's 3 pieces are 6% faster than the long tile's 4 (59 / 63 us, not taken), at M = 256 25%
    (41 / 51 us, taken)."""
    rest = {c: t for c, t in timings.items() if c != own_order}
    best = min(rest, key=rest.get)
    if own_order in timings and (1 + ORDER_MARGIN) * timings[own_order] < rest[best]:
        return own_order
    whole = (best[0], 0)
    return whole if rest.get(whole, float("inf")) <= (1 + WHOLE_MARGIN) * rest[best] else best
