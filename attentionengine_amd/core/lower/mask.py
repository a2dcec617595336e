"""mask_mod lowering and mask inference.

The reference traces ``mask_mod(b, h, q_idx, kv_idx)`` with ``torch.fx`` and prints one python
statement per node (attention_engine/core/codegen/common.py:124-152, vocabulary: python
``operator.*`` functions and ``torch.logical_and``), then materialises the block mask to choose
between the dense-causal and the block-sparse template (core/lower/lower.py:721-756).

Here the same fx graph becomes one C++ statement per node inside ``ae_mask_mod``; arithmetic is
done on ``int`` exactly as python does it (floor division and modulo keep python's sign rules),
so the device mask equals the host mask bit for bit.  Mask inference classifies every
(q-tile, kv-tile) pair as empty / partial / full so the kernel can skip empty tiles and skip the
elementwise test on full ones.
"""
from __future__ import annotations

import operator

import torch
import torch.fx as fx


# fx target -> C++ expression template.  Comparison results are bool, arithmetic is int.
_BINARY = {
    operator.ge: "({0} >= {1})", operator.gt: "({0} > {1})", operator.le: "({0} <= {1})",
    operator.lt: "({0} < {1})", operator.eq: "({0} == {1})", operator.ne: "({0} != {1})",
    operator.add: "({0} + {1})", operator.sub: "({0} - {1})", operator.mul: "({0} * {1})",
    operator.floordiv: "ae_floordiv({0}, {1})", operator.mod: "ae_pymod({0}, {1})",
    operator.and_: "({0} & {1})", operator.or_: "({0} | {1})", operator.xor: "({0} ^ {1})",
    torch.logical_and: "((bool)({0}) & (bool)({1}))", torch.logical_or: "((bool)({0}) | (bool)({1}))",
    torch.logical_xor: "((bool)({0}) ^ (bool)({1}))",
}
_UNARY = {
    operator.neg: "(-{0})", operator.not_: "(!{0})", operator.invert: "ae_invert({0})",
    operator.abs: "ae_iabs({0})", abs: "ae_iabs({0})", torch.logical_not: "(!(bool)({0}))",
    torch.abs: "ae_iabs({0})",
}

MASK_HELPERS = """
AE_DEV int ae_floordiv(int a, int b) { int q = a / b; return ((a % b != 0) && ((a < 0) != (b < 0))) ? q - 1 : q; }
AE_DEV int ae_pymod(int a, int b) { int r = a % b; return (r != 0 && ((r < 0) != (b < 0))) ? r + b : r; }
AE_DEV int ae_iabs(int a) { return a < 0 ? -a : a; }
AE_DEV bool ae_invert(bool a) { return !a; }
AE_DEV int ae_invert(int a) { return ~a; }
"""


def _arg(a):
    if isinstance(a, fx.Node):
        return "n_" + a.name   # prefixed: fx names such as "xor" / "and" are C++ tokens
    if isinstance(a, bool):
        return "true" if a else "false"
    if isinstance(a, int):
        return str(a)
    raise NotImplementedError(f"mask_mod: unsupported constant operand {a!r} (integers only)")


class LoweredMask:
    """Result of tracing a mask_mod."""

    def __init__(self, body: str, uses_b: bool, uses_h: bool, python_lines):
        self.body = body              # statements of ae_mask_mod, ending in a return
        self.uses_b = uses_b
        self.uses_h = uses_h
        self.python_lines = python_lines  # the traced graph, one line per node (debug aid)


def lower_mask_mod(mask_mod) -> LoweredMask:
    """fx-trace ``mask_mod`` and translate it to the body of
    ``bool ae_mask_mod(int b, int h, int q_idx, int kv_idx)``."""
    graph = fx.symbolic_trace(mask_mod).graph
    nodes = list(graph.nodes)
    placeholders = [n for n in nodes if n.op == "placeholder"]
    if len(placeholders) != 4:
        raise NotImplementedError("mask_mod must take exactly (b, h, q_idx, kv_idx)")
    canonical = ["b", "h", "q_idx", "kv_idx"]
    lines = [f"const int n_{ph.name} = {c}; (void)n_{ph.name};" for ph, c in zip(placeholders, canonical)]
    py = []
    ret = None
    for n in nodes:
        if n.op == "placeholder":
            continue
        if n.op == "output":
            ret = n.args[0]
            continue
        if n.op != "call_function":
            raise NotImplementedError(f"mask_mod: unsupported graph node {n.op} ({n.target})")
        if n.target in _BINARY and len(n.args) == 2:
            expr = _BINARY[n.target].format(_arg(n.args[0]), _arg(n.args[1]))
        elif n.target in _UNARY and len(n.args) == 1:
            expr = _UNARY[n.target].format(_arg(n.args[0]))
        else:
            raise NotImplementedError(f"mask_mod: unsupported operation {n.target}")
        lines.append(f"const auto n_{n.name} = {expr};")
        py.append(f"{n.name} = {getattr(n.target, '__name__', n.target)}({', '.join(_arg(a) for a in n.args)})")
    if ret is None:
        raise NotImplementedError("mask_mod returned nothing")
    lines.append(f"return (bool)({_arg(ret)});")
    used = {a.name for n in nodes for a in n.all_input_nodes}
    return LoweredMask("\n".join("  " + ln for ln in lines), placeholders[0].name in used,
                       placeholders[1].name in used, py)


class MaskPlan:
    """What the prefill kernel needs to know about a mask.

    mode 0: no mask; mode 1: exactly ``q_idx >= kv_idx`` (analytic tile skip + diagonal test);
    mode 2: tile-class table int8 [b|1, h|1, n_q_tiles, n_kv_tiles] with 0 = skip, 1 = visit and
    apply the elementwise mask, 2 = visit, fully visible.
    """

    def __init__(self, mode: int, table=None, block_m: int = 0, block_n: int = 0, elementwise: bool = False, band=None):
        self.mode = mode
        # (lo, hi) where the mask of mode 2 is exactly lo <= q_idx - kv_idx <= hi (hi None: no far edge at this size)
        self.band = band
        self.table = table
        self.block_m = block_m
        self.block_n = block_n
        self.elementwise = elementwise
        # late q tiles visit clearly more kv tiles than early ones (causal variants, long sliding windows): the
        # kernels then start the long q tiles first
        self.heavy_last = False
        if table is not None and table.shape[2] >= 4:
            work = (table > 0).sum(dim=-1).to(torch.float32).mean(dim=(0, 1))
            third = table.shape[2] // 3
            self.heavy_last = bool(work[-third:].mean() >= 1.25 * work[:third].mean())


class MaskSurvey:
    """A mask evaluated once over the whole [Sq, Skv] grid, in blocks of ``step_m`` x ``step_n`` positions that tables of
    any coarser tile are put together from (``table``)."""

    def __init__(self, classes, causal, band, Sq, Skv, step_m, step_n):
        self.classes = classes        # int8 [b|1, h|1, blocks, blocks]: 0 empty, 1 partly, 2 fully visible
        self.causal = causal          # exactly q_idx >= kv_idx, over equal lengths
        self.band = band              # see MaskPlan; None for masks that read b or h
        self.Sq, self.Skv, self.step_m, self.step_n = Sq, Skv, step_m, step_n

    def table(self, tile_m, tile_n):
        """int8 [b|1, h|1, n_q_tiles, n_kv_tiles] (see MaskPlan)."""
        c = self.classes
        rm, rn = tile_m // self.step_m, tile_n // self.step_n
        if (rm, rn) == (1, 1):
            return c
        some, every = (c > 0), (c == 2)
        for dim, r in ((3, rn), (2, rm)):
            some, every = _blocks(some, dim, r, torch.any), _blocks(every, dim, r, torch.all)
        return some.to(torch.int8) + every.to(torch.int8)


def survey_mask(mask_mod, lowered: LoweredMask, B: int, H: int, Sq: int, Skv: int, step_m: int = 32, step_n: int = 32,
                chunk_rows: int = 4096) -> MaskSurvey:
    """Evaluates the mask on the host: with batch/head extent 1 when the traced graph does not read b / h, and in row
    chunks so the full [Sq, Skv] grid is never resident at once."""
    mb = B if lowered.uses_b else 1
    mh = H if lowered.uses_h else 1
    parts = []
    causal, one = True, (mb, mh) == (1, 1)
    d_lo, d_hi, seen = Sq + Skv, -(Sq + Skv), 0       # extremes of q - kv over the visible positions, and their number
    chunk_rows = max(step_m, (chunk_rows // step_m) * step_m)
    kv = torch.arange(Skv).view(1, 1, 1, Skv)
    bb = torch.arange(mb).view(mb, 1, 1, 1)
    hh = torch.arange(mh).view(1, mh, 1, 1)
    for r0 in range(0, Sq, chunk_rows):
        r1 = min(Sq, r0 + chunk_rows)
        q = torch.arange(r0, r1).view(1, 1, r1 - r0, 1)
        m = mask_mod(bb, hh, q, kv)
        if not isinstance(m, torch.Tensor):
            m = torch.tensor(bool(m))
        m = m.to(torch.bool).expand(mb, mh, r1 - r0, Skv)
        here = (causal or one) and bool(torch.equal(m, (q >= kv).expand_as(m)))
        causal = causal and here
        if one and here:              # (the extremes and the number of a causal chunk are known)
            d_lo, d_hi = min(d_lo, max(0, r0 - Skv + 1)), max(d_hi, r1 - 1)
            seen += int(torch.arange(r0 + 1, r1 + 1).clamp(max=Skv).sum())
        elif one:
            rows = m[0, 0]
            any_row = rows.any(dim=1)
            if bool(any_row.any()):
                qr = torch.arange(r0, r1)[any_row]
                first = rows[any_row].to(torch.int8).argmax(dim=1)
                last = Skv - 1 - rows[any_row].flip(1).to(torch.int8).argmax(dim=1)
                d_lo, d_hi = min(d_lo, int((qr - last).min())), max(d_hi, int((qr - first).max()))
            seen += int(rows.sum())
        # a block cut by the sequence end is "full" when every in-range element is visible
        some = _blocks(_blocks(m, 3, step_n, torch.any), 2, step_m, torch.any)
        every = _blocks(_blocks(m, 3, step_n, torch.all), 2, step_m, torch.all)
        parts.append(some.to(torch.int8) + every.to(torch.int8))
    band = None
    if one and seen and seen == band_size(Sq, Skv, d_lo, d_hi):
        band = (d_lo, None if d_hi >= Sq - 1 else d_hi)
    return MaskSurvey(torch.cat(parts, dim=2), causal and Sq == Skv, band, Sq, Skv, step_m, step_n)


def plan_mask(mask_mod, lowered: LoweredMask, B: int, H: int, Sq: int, Skv: int, tile_m: int,
              tile_n: int, elementwise: bool = True, chunk_rows: int = 4096, survey=None) -> MaskPlan:
    """Classify the mask on the host for tiles of ``tile_m`` x ``tile_n`` positions, from a ``survey`` of the same mask
    and extents if there is one."""
    if mask_mod is None:
        return MaskPlan(0)
    if survey is None or tile_m % survey.step_m or tile_n % survey.step_n:
        survey = survey_mask(mask_mod, lowered, B, H, Sq, Skv, tile_m, tile_n, chunk_rows)
    if survey.causal and elementwise:
        return MaskPlan(1, None, tile_m, tile_n, True)
    table = survey.table(tile_m, tile_n)
    if not elementwise:
        # mask_value != "-inf": the forward only skips tiles (attn_tl.py:124-137 guards the
        # elementwise test with is_inf_mask); visited tiles are treated as fully visible.
        table = torch.where(table > 0, torch.full_like(table, 2), table)
    return MaskPlan(2, table.contiguous(), tile_m, tile_n, elementwise, survey.band if elementwise else None)


def band_size(Sq: int, Skv: int, lo: int, hi: int) -> int:
    """Number of positions of a [Sq, Skv] grid with lo <= q - kv <= hi.  A mask whose visible positions all lie in the
    band and are as many as the band has is the band."""
    q = torch.arange(Sq)
    return int(((q - lo).clamp(max=Skv - 1) - (q - hi).clamp(min=0) + 1).clamp(min=0).sum())


def _blocks(x: torch.Tensor, dim: int, n: int, reduce) -> torch.Tensor:
    """``reduce`` (torch.any / torch.all) over runs of n elements of dimension ``dim``; a last run that the end cuts is
    reduced over what it has."""
    if n == 1:
        return x
    whole = x.shape[dim] // n * n
    parts = []
    if whole:
        parts.append(reduce(x.narrow(dim, 0, whole).unflatten(dim, (whole // n, n)), dim=dim + 1))
    if whole < x.shape[dim]:
        parts.append(reduce(x.narrow(dim, whole, x.shape[dim] - whole), dim=dim, keepdim=True))
    return parts[0] if len(parts) == 1 else torch.cat(parts, dim=dim)
