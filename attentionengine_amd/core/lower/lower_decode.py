"""Decode lowering and operators: GQA split-KV decode and MLA (shared latent KV) decode.

Stands where the reference's decode lowerings fill their templates
(attention_engine/core/lower/lower_decode_gqa.py:348-408, lower_decode_mla.py:25-38, generic
``lower_combine`` in lower_decode.py:287-313) and where the generated ``_attention.forward``
allocates the split-KV work buffers and launches split + combine
(core/template/tl_template/attn/attn_gqa_decode_tl.py:338-349, mla_decode_tl.py:326-335).

Differences from the reference that are on purpose:
  * the reference's decode templates ignore score_mod / online_func and hard-code softmax with
    scale D^-0.5 (attn_gqa_decode_tl.py:38,52-67; mla_decode_tl.py:30); here the traced user
    functions are honoured, including ``OnlineFunc.combine``;
  * partial results are fp32 and the merged lse (natural log) is kept on ``final_rowscales``
    (the CuTe MLA convention, cute_template_kvshared/flash_api.cpp:180-181,204-209).
"""
from __future__ import annotations

import functools
import math
import os

import torch

from ..codegen.hip_gen import Emitter
from ..runtime import hip_rt as rt
from ..runtime import host
from ..transform.core import SymbolicColReduceArray
from ..transform.graph import Var
from . import lower as L


def lower_combine(online_func, final_rowscale_names):
    """Trace ``OnlineFunc.combine`` on [num_split, block_M] arrays and emit ``ae_combine``.

    Returns the function text.  ``w[k]`` is the o_scale of split k.  When o_scale has the form
    ``exp(x - y)`` with x one of the input rowscales and y free of the split axis (the log-domain
    merge of attn_script/gqa_inference.py:73-81), y is the merged value of that rowscale and is
    written to ``merged``; other rowscales have no defined merge and are set to NaN."""
    nrs = max(1, len(final_rowscale_names))
    syms = {n: SymbolicColReduceArray(n, Var(n), shape_idx=["num_split", "block_M"])
            for n in final_rowscale_names}
    leaves = {id(s): (f"rs[{i}]", True) for i, s in enumerate(syms.values())}
    o_scale = online_func.combine(syms)
    em = Emitter(leaves, {}, ["num_split"], n="AE_NSPLIT", prefix="cb", split_axis=True)
    val = em.value(o_scale)
    merged = {}
    if o_scale.code.type == "Exp" and o_scale.prev and o_scale.prev[0].code.type == "Sub":
        x, y = o_scale.prev[0].prev
        for i, s in enumerate(syms.values()):
            if x is s and "num_split" not in y.shape_idx:
                yv = em.value(y)
                if not yv[1]:
                    merged[i] = yv[0]
    body = [em.code()]
    src = f"{val[0]}[e]" if val[1] else val[0]
    body += ["#pragma unroll", f"  for (int e = 0; e < AE_NSPLIT; e++) w[e] = {src};"]
    undefined = '__builtin_nanf("")'
    for i in range(len(final_rowscale_names)):
        body.append(f"  merged[{i}] = {merged.get(i, undefined)};")
    text = "\n".join(body)
    # (a template over the number of partial results, whatever the configuration's macro of that name says)
    return f"""#pragma push_macro("AE_NSPLIT")
#undef AE_NSPLIT
template <int AE_NSPLIT>
AE_DEV void ae_combine(const float (&rs)[{nrs}][AE_NSPLIT], float (&w)[AE_NSPLIT],
                       float (&merged)[{nrs}]) {{
{text}
}}
#pragma pop_macro("AE_NSPLIT")
"""


def merges_in_any_order(online_func, final_rowscale_names) -> bool:
    """True when ``OnlineFunc.combine`` is the log-sum-exp merge of one row scale (attn_script/gqa_inference.py:73-81):
    o_scale = exp(lse - (log(sum(exp(lse - max(lse)))) + max(lse))).  Partial results may then be merged in groups first
    and the groups afterwards; another combine() sees all of them at once, as its author wrote it."""
    if len(final_rowscale_names) != 1:
        return False
    lse = SymbolicColReduceArray("lse", Var("lse"), shape_idx=["num_split", "block_M"])
    try:
        o = online_func.combine({final_rowscale_names[0]: lse})
        x, y = o.prev[0].prev
        a, b = y.prev
        log, mx = (a, b) if a.code.type == "Log" else (b, a)
        total = log.prev[0]
        term = total.prev[0]
        return (o.code.type == "Exp" and o.prev[0].code.type == "Sub" and x is lse and y.code.type == "Add"
                and log.code.type == "Log" and mx.code.type.endswith("ReduceMax") and mx.prev[0] is lse
                and total.code.type.endswith("ReduceSum") and term.code.type == "Exp"
                and term.prev[0].code.type == "Sub" and term.prev[0].prev[0] is lse and term.prev[0].prev[1] is mx)
    except (AttributeError, IndexError, TypeError, ValueError):
        return False


def combine_rows(threads, dv):
    """Output rows of a merge workgroup (AE_COMBINE_ROWS of csrc/kernels/ae_combine.hip): four value columns a thread."""
    return max(1, threads // (dv // 4))


def merge_capacity(n, any_order):
    """Partial results that a merge of ``n`` is built for.  The log-sum-exp merge gives places without a result no weight, so
    it is built for powers of two: a cache that grows by a token a call meets a new kernel only where it has doubled.  Up to
    16 places every count, beyond that 5, 6, 7 and 8 eighths of the places are constants of the build and cost what a build
    for the exact count does; others up to 0.1 us a call (B1 H64 Skv4009, 21 of 32 places: merge 3.92 us on both).  Another combine() is built for its exact count."""
    return 1 << (n - 1).bit_length() if any_order else n


def merge_config(dv, dtype, n_rowscales, capacity, threads, splits_per_partial=1):
    """ae_config.h of csrc/kernels/ae_combine.hip."""
    return "\n".join([
        "// generated by core/lower/lower_decode.py -- do not edit",
        f"#define AE_DV {dv}",
        f"#define AE_DTYPE_BF16 {1 if dtype == torch.bfloat16 else 0}",
        f"#define AE_N_ROWSCALES {n_rowscales}",
        f"#define AE_NSPLIT {capacity}",
        f"#define AE_SPLITS_PER_PARTIAL {splits_per_partial}",
        f"#define AE_COMBINE_THREADS {threads}",
        "",
    ])


class Merges:
    """The merge kernels of one operator (csrc/kernels/ae_combine.hip)."""

    def __init__(self, d, dv, dtype, n_rowscales, functor_src, any_order, threads, allow_spills=None):
        self._dims, self._dtype, self._n_rowscales, self._functor_src = (d, dv), dtype, n_rowscales, functor_src
        self.any_order, self._threads, self._allow_spills = any_order, threads, allow_spills
        self._modules = {}

    def config(self, n, splits_per_partial=1):
        return merge_config(self._dims[1], self._dtype, self._n_rowscales, merge_capacity(n, self.any_order), self._threads,
                            splits_per_partial)

    def cfg(self, n, splits_per_partial=1):
        """The launch configuration of a merge of ``n`` partial results a row."""
        return rt.TileCfg(block_m=combine_rows(self._threads, self._dims[1]),
                          block_n=merge_capacity(n, self.any_order) * splits_per_partial, threads=self._threads, lds_bytes=0,
                          head_dim=self._dims[0], head_dim_v=self._dims[1], elem_bytes=2, n_rowscales=self._n_rowscales,
                          mask_mode=0, merge_in_wg=int(self.any_order))

    def module(self, n, splits_per_partial=1):
        key = (merge_capacity(n, self.any_order), splits_per_partial)
        m = self._modules.get(key)
        if m is None:
            m = self._modules[key] = rt.compile_module(
                "ae_combine.hip", {"ae_config.h": self.config(n, splits_per_partial), "ae_functors.h": self._functor_src},
                allow_spills=self._allow_spills)
        return m


def render_decode_config(d, dv, dtype, n_waves, waves_per_eu, v_pad, n_rowscales, o_scale_one,
                         even_kv, n_split, merge_in_wg=False, merge_last=False, wg_first=False) -> str:
    return "\n".join([
        "// generated by core/lower/lower_decode.py -- do not edit",
        f"#define AE_D {d}",
        f"#define AE_DV {dv}",
        f"#define AE_NWAVES {n_waves}",
        f"#define AE_DTYPE_BF16 {1 if dtype == torch.bfloat16 else 0}",
        f"#define AE_N_ROWSCALES {n_rowscales}",
        f"#define AE_O_SCALE_ONE {1 if o_scale_one else 0}",
        f"#define AE_EVEN_KV {1 if even_kv else 0}",
        f"#define AE_WAVES_PER_EU {waves_per_eu}",
        f"#define AE_V_PAD {v_pad}",
        f"#define AE_NSPLIT {n_split}",
        f"#define AE_MERGE_IN_WG {1 if merge_in_wg else 0}",
        f"#define AE_MERGE_LAST {1 if merge_last else 0}",
        f"#define AE_WG_FIRST {1 if wg_first else 0}",
        "",
    ])


class _SplitTuning:
    """tune=True for the split-KV decode operators: their one measured choice is how many workgroups share
    the kv axis of a (batch, kv head).  The reference tunes ``num_split`` (1, 2, 4, 8) together with its tile
    sizes whenever it builds the MLA decode kernel (mla_decode_tl.py:13-24, 308-319).  Here the candidates are
    the planned count, its half and its multiples; they are measured on the caller's tensors at the first call
    of a shape -- with a paged cache that includes the actual sequence lengths, whose spread decides how many
    splits balance the chip -- and kept in ``tune_file`` as ``[splits]`` under the five problem keys
    (core/lower/tuner.py)."""

    @staticmethod
    def _balanced_splits(coeff, Skv):
        """Splits beyond which the merge costs more than the shorter stream saves.  A workgroup's time is about
        a * Skv / splits for its share of the kv axis plus b * splits for the partial results and their merge, least
        at sqrt(a * Skv / b); ``coeff`` = sqrt(a / b), measured per kernel, rounded to a power of two."""
        return 2 ** max(0, round(math.log2(max(1.0, coeff * math.sqrt(Skv)))))

    # attributes that plan_splits() reads at call time: a new value drops the plans made under the old one
    @property
    def target_workgroups(self):
        return self._target_workgroups

    @target_workgroups.setter
    def target_workgroups(self, n):
        self._target_workgroups = n
        self._host.clear()

    def _init_tuning(self, tune, tune_file):
        self._tune_file = tune_file if (tune and tune_file) else ""
        self._tuned = {}          # (B, Hq, Hkv, Skv) -> the count plan_splits() starts from
        self.tune_times = None

    def _tune_splits(self, key, candidates, run, usable=None):
        """Fills self._tuned[key] from tune_file or by measuring run() under every candidate.  ``usable(n)``: the plan can
        launch a count of the file, also one that is no candidate (the file was written under another plan)."""
        from . import tuner
        B, Hq, Hkv, Skv = key
        pk = {"batch": B, "heads": Hq, "seq_len": Skv, "dim": self.D, "dimv": self.DV}
        found = tuner.lookup(self._tune_file, pk)
        if (isinstance(found, list) and len(found) == 1 and
                (found[0] in candidates or (usable is not None and type(found[0]) is int and usable(found[0])))):
            self._tuned[key] = found[0]
            return
        log = print if os.environ.get("AE_TUNE_VERBOSE", "") == "1" else None

        def build(c):
            # (a plan of the native host path serves every later call of the shape: each candidate starts without one)
            self._tuned[key] = c
            self._host.clear()
            return c
        best, _, times = tuner.pick(candidates, build, lambda c: run(), log)
        build(best)
        self.tune_times = {candidates[i]: ms for i, ms in times.items()}
        tuner.store(self._tune_file, pk, [best])


class GQADecodeOp(_SplitTuning):
    """mod(q [B,1,Hq,D], k [B,Skv,Hkv,D], v [B,Skv,Hkv,DV]) -> o [B,1,Hq,DV]."""

    TILE = 32          # kv rows per wave tile (AE_TILE in csrc/kernels/ae_decode.hip)
    N_WAVES = 4
    HEADS_PER_WG = 16  # N of the 16x16x32 MFMA

    # sqrt(a / b) of _balanced_splits(): B1 Hq32 Hkv8 Skv8192 D128 takes 80 us with one workgroup per kv head and
    # 0.7 us more for every further one (their four partials each, and the merge); beyond 64 partials a head the
    # merge kernel no longer holds them in registers
    SPLIT_COEFF = 0.117
    MAX_WGS_PER_KV_HEAD = 16
    # ... and where a workgroup merges its waves' partials first (AE_WG_FIRST of ae_decode.hip: a quarter of the merge
    # traffic), the counts that _workgroups() chooses from: up to 8 any, beyond those that the builds of
    # ae_decode.hip take as constants (5, 6, 7 or 8 eighths of a power of two)
    GROUPED_WGS_PER_KV_HEAD = (1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32, 48, 64)

    def __init__(self, qkv_meta, custom_fwd_inputs, score_mod, mask_mod, online_func, mask_value,
                 target_workgroups=256, tune=False, tune_file="", allow_spills=None):
        self.allow_spills = allow_spills
        self._init_tuning(tune, tune_file)
        q_meta, k_meta, v_meta = qkv_meta
        self.dtype = q_meta.dtype
        self.D, self.DV = int(q_meta.shape[3]), int(v_meta.shape[3])
        if self.D % 32 or self.DV % 16:
            raise NotImplementedError(f"decode head dims (D={self.D}, DV={self.DV}) must be multiples of 32 / 16")
        if mask_mod is not None:
            # the reference's GQA decode cannot take a mask_mod either (its lowering calls
            # create_mask with the wrong arity, lower_decode_gqa.py:394)
            raise NotImplementedError("GQA decode takes mask_mod=None")
        self.functors = L.trace_functors(score_mod, None, online_func, custom_fwd_inputs, self.dtype, mask_value)
        self.names = self.functors.final_rowscale_names
        self.n_rowscales = len(self.names)
        if self.n_rowscales > rt.AE_MAX_ROWSCALES or len(self.functors.customs) > rt.AE_MAX_CUSTOM:
            raise NotImplementedError("too many rowscales / custom inputs")
        self.functor_src = L.render_functors(self.functors) + lower_combine(online_func, self.names)
        self._host = host.new_host(self.D, self.DV, self.dtype, self.functors.customs, self.n_rowscales)
        # the merge may go by workgroup first (AE_WG_FIRST of ae_decode.hip)
        self.grouped_merge = merges_in_any_order(online_func, self.names)
        self.target_workgroups = target_workgroups
        # True: the split-KV partials go to the work buffer built into libae_hip.so (ae_decode_fwd_noalloc)
        # instead of two tensors allocated per call -- for callers under HIP graph capture or in loops that
        # must not allocate; launches whose partials exceed rt.NOALLOC_SCRATCH_BYTES are refused
        self.static_workspace = False
        self.v_pad = (64 - (2 * self.DV) % 256) % 256 or 256
        self._merges = Merges(self.D, self.DV, self.dtype, self.n_rowscales, self.functor_src, self.grouped_merge,
                              64 if self.DV <= 256 else 128, allow_spills)
        self._builds = {}             # what _variant() compiled: counts of splits share a kernel
        self.final_rowscales = {}
        self.block_mask = None
        self._variants = {}
        self._plans = {}              # ((B, Hq, Hkv, Skv), tuned splits, target workgroups) -> plan_splits(...)
        self.meta_shape = tuple(int(x) if not isinstance(x, str) else 0
                                for x in (q_meta.shape[0], q_meta.shape[1], v_meta.shape[1], v_meta.shape[2]))
        self.source = self.functor_src
        B, Hq, Hkv, Skv = self.meta_shape
        if Skv > 0 and B > 0:
            n_split, _ = self.plan_splits(B, Hq, Hkv, Skv)
            _, _, _, cfg_src = self._variant(n_split, Skv % self.TILE == 0, self._merge_mode(n_split))
            self.source = cfg_src + "\n" + self.functor_src

    @property
    def static_workspace(self):
        return self._static_workspace

    @static_workspace.setter
    def static_workspace(self, on):
        self._static_workspace = on
        self._host.clear()

    @staticmethod
    @functools.lru_cache(maxsize=1024)
    def _workgroups(units, tiles, width, cus, most):
        """Workgroups that share the kv axis of one of ``units`` (batch, kv head, head tile) of ``tiles`` kv tiles: the
        least that is within 1 % of the cheapest by what a call takes.  ``width``: bytes of a key and a value row in
        units of 512.

        A trip of a workgroup (one tile a wave) takes 1.4 us where it has a CU to itself (1.7 past the memory-side
        cache; D64 0.8, D256 3.8), 3.0 (3.7) where two share it - a CU has only so many lines on the way -, and never
        less than the chip's memory needs for all that run (8.1 TB/s out of the memory-side cache, 6.2 past it).  So 257 workgroups take
        nearly twice as long as 256 of the same length, and rounds of two a CU follow each other, half as if a round had
        to wait for the one before, half without a gap.  Each further workgroup costs the merge 0.08 us.  Workgroup k of
        an axis runs on XCD k mod 8 where their number is a multiple of 8: if the last of them have no tiles left, whole
        XCDs idle (B19 Hq64 Hkv8 Skv2204: 8 workgroups 40.8 us, 7 30.8).

        Fitted to 1819 timings (216 shapes of fp16 and bf16, batch 1 to 128, 128 to 32768 keys, D128), where the choice is
        0.4 % slower than the best one on average, 7 % at most; at D256 (25 shapes) 0.1 and 2 %.  Head dim 64 has constants
        of its own: three workgroups share a CU, and starting and ending them is what more of them cost (fitted to 114 shapes; on 37 others the
        choice is 1.2 % off the best on average, 11 % at most, and by the constants of D128 B48 Hq16 Hkv2 Skv871 took 10.3 us
        instead of 7.5).  Against the power of two that fills the CUs, which was
        the rule before: B67 Hq32 Hkv4 Skv13634 471 -> 346 us, B71 Skv3876 138 -> 113, B65 Hq16 Hkv2 Skv2082 32.6 -> 25.5,
        B19 Hq64 Hkv8 Skv3372 54 -> 42."""
        kib = 16 * width                                     # of keys and values in a wave's tile
        cached = units * tiles * kib <= 300e3                # (of 256 MB: some of it still hits a little beyond)
        if width <= 0.5:
            per_cu, power, fixed, ends, gap, merge = 3, 1.41, 1.7, 0.98, 0.0, (1.18, 0.068)
            alone, rate, share = 0.68 if cached else 0.65, 12.3 if cached else 7.3, 0.632
        else:
            per_cu, power, fixed, ends, gap, merge = 2, 4, 3.6, 0.0, 0.45, (0.8, 0.08)
            alone, rate = (1.4, 8.1) if cached else (1.7, 6.2)
            alone *= 0.2 + 0.8 * width if width <= 1 else 1 + 1.7 * (width - 1)
            share = alone * (2.15 if width <= 1 else 2.75) / 2       # (wider rows: one workgroup fits a CU)
        best = []
        for x in GQADecodeOp.GROUPED_WGS_PER_KV_HEAD:
            if x > most:
                break
            trips = -(-tiles // (GQADecodeOp.N_WAVES * x))
            live = -(-tiles // (GQADecodeOp.N_WAVES * trips))
            xcds = math.gcd(x, 8)
            rounds, rest = divmod(units * xcds * -(-live // xcds), per_cu * cus)

            def trip(n):
                here = -(-n // cus)
                return (max(alone, share * here if here > 1 else 0.0) ** power + (n * 4096e-6 * kib / rate) ** power) ** (1 / power)
            full, last = trip(per_cu * cus), trip(rest) if rest else 0.0
            us = full if rounds else last
            if rounds + (rest > 0) > 1:
                us = 0.5 * (rounds * full + last + (rounds + rest / (per_cu * cus)) * full + gap)
            best.append((fixed + us * trips + ends * max(1.0, units * x / cus) + (merge[0] + merge[1] * x if x > 1 else 0.0), x))
        least = min(best)[0]
        return next(x for us, x in best if us <= 1.01 * least)

    def plan_splits(self, B, Hq, Hkv, Skv):
        """(number of partials, kv positions per partial).  One partial per wave.  Where a workgroup merges its waves'
        partials first, the workgroups that share a kv axis are chosen by what the call takes (``_workgroups``); a
        combine() that wants all of them gets a power of two of workgroups, only until ``target_workgroups`` exist (one
        per CU of an MI355X) and no more than its merge is worth (``_balanced_splits``)."""
        group = Hq // Hkv
        head_tiles = -(-group // self.HEADS_PER_WG)
        base_wgs = B * Hkv * head_tiles
        tiles_total = -(-Skv // self.TILE)
        max_x = max(1, tiles_total // self.N_WAVES)          # at least one tile per wave
        x = self._tuned.get((B, Hq, Hkv, Skv))
        if x is None and self.grouped_merge:
            # (the entry point with a built-in work buffer runs the same plan: no finer than what fits there)
            fits = rt.NOALLOC_SCRATCH_BYTES // (B * Hq * self.N_WAVES * (self.DV + 1) * 4)
            # (four workgroups a CU already: no split gains)
            most = max(1, min(max_x, fits)) if base_wgs < 4 * self.target_workgroups else 1
            x = self._workgroups(base_wgs, tiles_total, (self.D + self.DV) / 256, self.target_workgroups, most)
        if x is None:
            x = min(-(-self.target_workgroups // base_wgs), self._balanced_splits(self.SPLIT_COEFF, Skv),
                    self.MAX_WGS_PER_KV_HEAD)
        x = max(1, min(max_x, x))
        while x & (x - 1) and not (self.grouped_merge and x in self.GROUPED_WGS_PER_KV_HEAD):
            x -= 1
        n_split = x * self.N_WAVES
        tiles_per_split = -(-tiles_total // n_split)
        return n_split, tiles_per_split * self.TILE

    def _split_count(self, key, x):
        """Workgroups per (batch, kv head, head tile) that plan_splits() makes of a wish of x."""
        old = self._tuned.get(key)
        self._tuned[key] = x
        got = self.plan_splits(*key)[0] // self.N_WAVES
        if old is None:
            del self._tuned[key]
        else:
            self._tuned[key] = old
        return got

    def merges_in_workgroup(self, n_split):
        """One workgroup per (batch, kv head, head tile): its waves hold every partial result, meet in LDS and
        write the merged output themselves (AE_MERGE_IN_WG of ae_decode.hip) - one launch, no work buffers.
        The entry point without allocations keeps the two launches it is declared with."""
        return (n_split == self.N_WAVES and not self.static_workspace
                and os.environ.get("AE_DECODE_MERGE_IN_WG", "1") != "0")      # (0: keep the two launches)

    def merges_in_last_workgroup(self, n_split):
        """Launches that share a kv axis out over several workgroups: the workgroup that finishes last merges
        (AE_MERGE_LAST of ae_decode.hip) instead of a second launch -- at batch 1 a third of the call.  Needs work
        buffers with arrival counters that stay zero between launches, so they are kept (per size and stream, Work of
        csrc/ae_host.cpp) instead of allocated per call: calls on one stream run one after the other and may share
        them.  A graph captured on a stream that has run the call before goes on using that stream's buffers, which
        then stay as long as the operator -- replay it on that stream, or not at the same time as eager calls of this
        operator there (AE_DECODE_MERGE_LAST=0 gives every call buffers of its own again); one captured on a stream
        without them has buffers of its own.  Not for the entry point without allocations, whose buffer is the
        library's."""
        return (n_split > self.N_WAVES and not self.static_workspace
                and os.environ.get("AE_DECODE_MERGE_LAST", "1") != "0")       # (0: keep the two launches)

    def _merge_mode(self, n_split):
        """TileCfg.merge_in_wg of a launch with ``n_split`` partial results a head."""
        return 1 if self.merges_in_workgroup(n_split) else (2 if self.merges_in_last_workgroup(n_split) else 0)

    def _wg_first(self, n_split, merge):
        return self.grouped_merge and merge != 1 and n_split > self.N_WAVES

    def _variant(self, n_split, even_kv, merge):
        """(module, split cfg, combine cfg, config source) of a launch's split kernel.  ``merge`` (0: two
        launches; 1: the split kernel merges its waves' partial results itself, AE_MERGE_IN_WG; 2: its last workgroup
        merges, AE_MERGE_LAST) is part of the key: it depends on ``static_workspace`` and environment variables, which
        may change between calls, and a kernel compiled for one form must never be launched as another (the kernel
        that merges in the workgroup leaves the work buffers unwritten; the others store through them)."""
        merge = int(merge)
        key = (n_split, even_kv, merge)
        v = self._variants.get(key)
        if v is None:
            lds = self.N_WAVES * self.TILE * (2 * self.DV + self.v_pad)
            # Two waves a SIMD (256 registers each) where the kernel fits them; a build that spills at that size
            # (value heads of 256: 85 registers through scratch memory, 1.56 ms where the chip's HBM allows 0.6 for
            # B64 Hq32 Hkv8 Skv8192) is built again for one wave a SIMD and the whole register file: 0.68 ms.
            # several workgroups per kv head: merged by workgroup first, where combine() allows it (AE_WG_FIRST)
            wg_first = self._wg_first(n_split, merge)
            per = self.N_WAVES if wg_first else 1
            # what the build holds the weights of: the partial results that its last workgroup merges, or its waves'
            most = merge_capacity(n_split // per, self.grouped_merge) if merge == 2 else self.N_WAVES
            build = self._builds.get((most, even_kv, merge, wg_first))
            if build is None:
                for waves_per_eu in (2, 1):
                    cfg_src = render_decode_config(self.D, self.DV, self.dtype, self.N_WAVES, waves_per_eu, self.v_pad,
                                                   self.n_rowscales, self.functors.o_scale_one, even_kv, most,
                                                   merge == 1, merge == 2, wg_first)
                    headers = {"ae_config.h": cfg_src, "ae_functors.h": self.functor_src}
                    module = rt.compile_module("ae_decode.hip", headers, allow_spills=True)
                    if not module.kernel_info()["ae_decode_split_kernel"].get(".vgpr_spill_count", 0):
                        break
                rt.check_spills(module, "ae_decode.hip", self.allow_spills)
                build = self._builds[(most, even_kv, merge, wg_first)] = module, cfg_src
            module, cfg_src = build
            if merge == 1 or wg_first:
                lds += self.n_rowscales * self.N_WAVES * 16 * 4       # the waves' row scales, behind the V tiles
            cfg = rt.TileCfg(block_m=self.HEADS_PER_WG, block_n=self.TILE, threads=64 * self.N_WAVES,
                             lds_bytes=lds, head_dim=self.D, head_dim_v=self.DV, elem_bytes=2,
                             n_rowscales=self.n_rowscales, mask_mode=0, merge_in_wg=merge)
            if merge == 0:
                cfg_src += self._merges.config(n_split // per, per)
            v = self._variants[key] = (module, cfg, self._merges.cfg(n_split // per, per), cfg_src)
        return v

    def __call__(self, q, k, v, *extra):
        done = self._host.run(q, k, v, *extra)             # a shape that has run before: csrc/ae_host.cpp
        if done is not None:
            self.final_rowscales = dict(zip(self.names, done[1:]))
            return done[0]
        n_custom = len(self.functors.customs)
        if len(extra) == n_custom + 1:
            extra = extra[:-1]     # the reference appends an all-ones mask here (lower_decode_gqa.py:390-396)
        if len(extra) != n_custom:
            raise TypeError(f"expected {n_custom} custom input tensor(s), got {len(extra)}")
        for name, t in (("q", q), ("k", k), ("v", v)):
            if not (isinstance(t, torch.Tensor) and t.is_cuda):
                raise RuntimeError(f"{name} must be a tensor on the GPU (there is no CPU path)")
            if t.dtype != self.dtype:
                raise TypeError(f"{name} has dtype {t.dtype}, the engine was built for {self.dtype}")
            if t.dim() != 4:
                raise ValueError(f"{name} must be [batch, seq, heads, dim]")
        B, Sq, Hq, D = q.shape
        _, Skv, Hkv, _ = k.shape
        if Sq != 1:
            raise ValueError("decode takes one query token per sequence (q is [B,1,Hq,D])")
        if (D, k.shape[3], v.shape[3]) != (self.D, self.D, self.DV) or Hq % Hkv or v.shape[:3] != k.shape[:3]:
            raise ValueError("inconsistent q/k/v shapes")
        q, k, v = (rt.rows_for_kernels(t) for t in (q, k, v))
        dev = q.device
        key = (B, Hq, Hkv, Skv)
        if self._tune_file and key not in self._tuned:
            x0 = self.plan_splits(*key)[0] // self.N_WAVES       # workgroups per (batch, kv head, head tile)
            self._tuned[key] = x0
            cands = [x for x in (x0, x0 // 2, 2 * x0, 4 * x0) if x >= 1]
            cands = [x for i, x in enumerate(cands) if self._split_count(key, x) == x and x not in cands[:i]]
            self._tune_splits(key, cands, lambda: self.__call__(q, k, v, *extra),
                              lambda x: self._split_count(key, x) == x)
        plan_key = (key, self._tuned.get(key), self.target_workgroups)
        plan = self._plans.get(plan_key)
        if plan is None:
            if len(self._plans) >= 64:
                self._plans.clear()
            plan = self._plans[plan_key] = self.plan_splits(B, Hq, Hkv, Skv)
        n_split, kv_per_split = plan
        stream = rt.current_stream(dev)
        merge = self._merge_mode(n_split)       # once per call: every later decision reads this value
        module, cfg, ccfg, _ = self._variant(n_split, Skv % self.TILE == 0, merge)
        out = torch.empty((B, 1, Hq, self.DV), dtype=self.dtype, device=dev)
        rowscales = [torch.empty((B, Hq, 1), dtype=torch.float32, device=dev) for _ in range(self.n_rowscales)]
        p = rt.AttnParams()
        p.q, p.k, p.v, p.out = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
        keep = []
        # partial results that go to memory: one per wave, or per workgroup where its waves merge theirs first
        o_rows = B * Hq * (n_split // self.N_WAVES if self._wg_first(n_split, merge) else n_split)
        rs_floats = max(1, self.n_rowscales) * B * Hq * n_split
        counters = B * Hkv * -(-(Hq // Hkv) // self.HEADS_PER_WG) if merge == 2 else 0
        if merge == 2:        # kept buffers, whose counters are zero between launches (ae_host.cpp: Work)
            keep = list(self._host.work(o_rows, rs_floats, counters, dev.index, stream))
        elif not self.static_workspace and merge == 0:
            keep = [torch.empty((o_rows, self.DV), dtype=torch.float32, device=dev),
                    torch.empty(rs_floats, dtype=torch.float32, device=dev)]
        if keep:
            p.partial_o, p.partial_rs = keep[0].data_ptr(), keep[1].data_ptr()
        for i, r in enumerate(rowscales):
            p.rowscale_out[i] = r.data_ptr()
        for i, (desc, t) in enumerate(zip(self.functors.customs, extra)):
            t = t.to(device=dev, dtype=desc.torch_dtype).contiguous()
            keep.append(t)
            p.custom[i] = t.data_ptr()
        p.q_stride_b, p.q_stride_s, p.q_stride_h, _ = q.stride()
        p.k_stride_b, p.k_stride_s, p.k_stride_h, _ = k.stride()
        p.v_stride_b, p.v_stride_s, p.v_stride_h, _ = v.stride()
        p.o_stride_b, p.o_stride_s, p.o_stride_h, _ = out.stride()
        p.batch, p.heads_q, p.heads_kv, p.seqlen_q, p.seqlen_kv = B, Hq, Hkv, 1, Skv
        p.num_splits, p.kv_per_split = n_split, kv_per_split
        launch = rt.decode_fwd_noalloc if self.static_workspace else rt.decode_fwd
        split, combine, modules = module.kernel("ae_decode_split_kernel"), None, (module,)
        if not merge:
            per = self.N_WAVES if self._wg_first(n_split, merge) else 1
            modules += (self._merges.module(n_split // per, per),)
            combine = modules[1].kernel("ae_decode_combine_kernel")
        launch(split, combine, p, cfg, ccfg, stream)
        if not self.static_workspace:
            host.add_forward(self._host, host.DECODE, B, 1, Hq, Hkv, Skv, dev, modules, split, cfg, combine=combine, ccfg=ccfg,
                             n_split=n_split, kv_per_split=kv_per_split, o_rows=o_rows, counters=counters,
                             env=("AE_DECODE_MERGE_IN_WG", "AE_DECODE_MERGE_LAST"))
        self.final_rowscales = dict(zip(self.names, rowscales))
        self._keepalive = keep
        return out


def render_mla_config(d1, d2, dv, dtype, block_n, k_pad, n_rowscales, o_scale_one, n_split, softmax=None,
                      paged=False, heads_per_wg=64) -> str:
    extra = [f"#define AE_PAGED {1 if paged else 0}"]
    if heads_per_wg != 64:
        extra.append(f"#define AE_HPW {heads_per_wg}")
    if softmax is not None:
        extra += [f"#define AE_SM_SCALE {L.float_literal(softmax[0])}", f"#define AE_SM_M {softmax[1]}",
                  f"#define AE_SM_R {softmax[2]}"]
    return "\n".join([
        "// generated by core/lower/lower_decode.py -- do not edit",
        f"#define AE_D1 {d1}",
        f"#define AE_D2 {d2}",
        f"#define AE_DV {dv}",
        f"#define AE_DTYPE_BF16 {1 if dtype == torch.bfloat16 else 0}",
        f"#define AE_N_ROWSCALES {n_rowscales}",
        f"#define AE_O_SCALE_ONE {1 if o_scale_one else 0}",
        f"#define AE_K_PAD {k_pad}",
        f"#define AE_NSPLIT {n_split}",
        *extra,
        "",
    ])


class MLADecodeOp(_SplitTuning):
    """Shared-latent-KV decode (``kv_shared=True``).

    TileLang call form (attn_script/mla_decode.py:115-118):
        mod(q [B,1,H,DV], q_pe [B,1,H,D-DV], kv [B,S,G,DV], k_pe [B,S,G,D-DV]) -> o [B,1,H,DV]
    CuTe call form (attn_script/mla_decode_cute.py:300-303; paged cache of 64-token pages with the
    identity block table the reference builds, attn_engine.py:193-206):
        mod(q [B,1,H,D], kv_cache [B*S/64, 64, G, D]) -> (out [B,1,H,DV], lse [B,H,1])
    ... and with the page order and the per-entry lengths the reference's engine binds as keyword
    arguments of ``flash_mla_with_kvcache`` (cute_template_kvshared/flash_mla_interface.py:73-111):
        mod(q [B,1,H,D], kv_cache [pages, page_size, G, D], block_table=int32 [B, max_pages_per_entry],
            cache_seqlens=int32 [B])
    Entry b attends to its first cache_seqlens[b] tokens; token t lives in row t % page_size of page
    block_table[b, t // page_size].  page_size must be a multiple of the 32-token kv tile.  An entry of
    length 0 returns zeros and lse -inf.  In a split launch an entry whose keys all lie in the first split writes its
    result itself; only longer entries go through the partial results and the merge.
    """

    BLOCK_N = 32
    HEADS_PER_WG = 64
    # wave-specialised kernel, per round of workgroups: query heads a workgroup -> (us to start and end, us per tile)
    ROUND_COST = {16: (1.9, 0.585), 32: (3.7, 0.73), 64: (4.9, 0.81)}
    # ... and where the entries of a paged cache are split by their lengths
    LENGTH_COST = {16: (3.03, 0.591), 32: (4.53, 0.784), 64: (6.48, 0.937)}
    K_PAD = 0
    # sqrt(a / b) of _balanced_splits(): B1 H128 Skv4096 takes 112 us unsplit and about 0.3 us more per split
    SPLIT_COEFF = 0.30
    MAX_SPLITS = 64
    N_STAGES = 3      # AE_NSTAGE of csrc/kernels/ae_mla_decode.hip
    WS_STAGES = 4     # AE_NSTAGE of csrc/kernels/ae_mla_decode_ws.hip
    PAGE_TABLE_ENTRIES = 1024    # AE_PTAB of the same: block-table entries of one split kept in LDS

    def __init__(self, qkv_meta, custom_fwd_inputs, score_mod, mask_mod, online_func, mask_value,
                 cute_convention=False, target_workgroups=256, tune=False, tune_file="", allow_spills=None):
        self.allow_spills = allow_spills
        self._init_tuning(tune, tune_file)
        q_meta, k_meta, v_meta = qkv_meta
        self.dtype = q_meta.dtype
        self.D, self.DV = int(q_meta.shape[3]), int(v_meta.shape[3])
        self.D2 = self.D - self.DV
        if self.D2 <= 0 or self.D2 % 16 or self.DV % 64:
            raise NotImplementedError(f"kv_shared needs D > DV with DV % 64 == 0 and (D-DV) % 16 == 0, got D={self.D} DV={self.DV}")
        if mask_mod is not None:
            raise NotImplementedError("MLA decode takes mask_mod=None")
        self.cute = bool(cute_convention)
        self.functors = L.trace_functors(score_mod, None, online_func, custom_fwd_inputs, self.dtype, mask_value)
        self.names = self.functors.final_rowscale_names
        self.n_rowscales = len(self.names)
        if self.functors.customs:
            raise NotImplementedError("custom inputs are not supported by the MLA decode path")
        self.functor_src = L.render_functors(self.functors) + lower_combine(online_func, self.names)
        self._host = host.new_host(self.D, self.DV, self.dtype, self.functors.customs, self.n_rowscales)
        self.target_workgroups = target_workgroups
        self.final_rowscales = {}
        self.block_mask = None
        self._merges = Merges(self.D, self.DV, self.dtype, self.n_rowscales, self.functor_src,
                              merges_in_any_order(online_func, self.names), 128, allow_spills)
        self._variants = {}
        self.source = self.functor_src
        shape = [q_meta.shape[0], q_meta.shape[1], v_meta.shape[1], v_meta.shape[2]]
        if not any(isinstance(x, str) for x in shape):
            B, Hq, Hkv, Skv = (int(x) for x in shape)
            heads, n_split, _ = self.plan(B, Hq, Hkv, Skv)
            self.source = self._variant(n_split, heads=heads)[2] + "\n" + self.functor_src
            if n_split > 1:
                self.source = self._merges.config(n_split) + self.source

    @staticmethod
    @functools.lru_cache(maxsize=1024)
    def _cheapest(units, group, tiles, n_splits, cus, d, dv, paged):
        """(query heads of a workgroup, splits) that a call of the wave-specialised kernel over ``units`` (batch entry, latent
        head) of ``group`` heads and ``tiles`` kv tiles takes least time with; ``n_splits``: the candidates, first and last.

        Its microseconds, up to a constant: one workgroup fits a CU, so it takes as many rounds as there are workgroups per
        CU, each a start and an end (f) and its tiles (c); the cache cannot arrive faster than it is read (5.7 TB/s); partial
        results cost by the byte (written, and read again by the merge), the merge by the split.  Fitted to 1073 timings - 40
        shapes, batch 1 to 128, 16 / 64 / 128 heads, 300 to 8000 keys, bf16, every split count up to 64 -, where the choice by
        it is 0.2 % slower on average than the best one measured, 2.8 % at most.  A paged cache counts half as if every entry
        filled its table, half as if they were spread evenly up to that: ``live``, the share of the splits that hold keys;
        those that do are not spread evenly, so a round is full at 1/1.4 of the CUs (B8 H128, 2048 tokens at most, 16 heads: 5
        splits, 192 live workgroups 19.4 us, 6, 224 22.9).

        Kept by the number of tiles: a latent cache that grows by a token a call asks anew every 32 calls (25 to 35 us, paged 45 to
        65; the 3 x 64 candidates evaluated at every length took 130 to 270, more than the choice gains, and with a function called
        for each candidate it is 60 to 85, 105 to 145)."""
        read = units * tiles * MLADecodeOp.BLOCK_N * 2e-6 * d / 5.7
        partial = 0.31 * units * group * 4e-6 * dv
        splits = sorted({-(-tiles // -(-tiles // n)) for n in range(n_splits[0], n_splits[1] + 1)})      # (none without tiles)
        best = None
        for heads, (f, c) in MLADecodeOp.ROUND_COST.items():
            if heads != 16 and group <= heads // 2:
                continue
            wgs = units * -(-group // heads)
            for n in splits:
                trip = f + c * -(-tiles // n)
                us = ((-(-wgs * n // cus) * trip) ** 4 + read ** 4) ** 0.25
                if n > 1:
                    us += 1.2 + 0.077 * n + partial * n
                if paged:
                    live = (n + 1) / (2 * n)
                    rounds = math.ceil(math.ceil(wgs * n * (live * 1.4 if n > 1 else 1.0) - 1e-6) / cus)
                    us += ((rounds * trip) ** 4 + (read * (0.5 if n > 1 else 1.0)) ** 4) ** 0.25
                    if n > 1:
                        us += 1.2 + 0.077 * n + partial * n * live
                if best is None or (us, -heads, n) < best:
                    best = us, -heads, n
        return -best[1], best[2]

    @staticmethod
    def _call_us(units, group, tiles, heads, n, cus, d, dv, spread):
        """``_cheapest``'s cost of one choice; ``spread``: entries spread evenly up to the table's width."""
        f, c = MLADecodeOp.ROUND_COST[heads]
        read = units * tiles * MLADecodeOp.BLOCK_N * 2e-6 * d / 5.7
        wgs = units * -(-group // heads)
        live = (n + 1) / (2 * n) if spread else 1.0
        rounds = math.ceil(math.ceil(wgs * n * (live * 1.4 if spread and n > 1 else 1.0) - 1e-6) / cus)
        us = ((rounds * (f + c * -(-tiles // n))) ** 4 + (read * (0.5 if spread and n > 1 else 1.0)) ** 4) ** 0.25
        return us + (1.2 + 0.077 * n + 0.31 * units * group * 4e-6 * dv * n * live if n > 1 else 0.0)

    @staticmethod
    def _length_us(batch, group, tiles, heads, most, n_wgs, cus, d, dv, spread):
        """... and of one plan by the entries' lengths: rounds, the read at 4.8 TB/s, 0.32 us a MB of partial results (written, and
        read by the merge), 0.05 a place of an entry in the merge, 0.5 for it.  The kernel's cut in closed form: of full tables every
        entry has as many splits as its share of the workgroups; of lengths that are spread evenly (``total`` tiles) an entry's last
        split is half full on average.  Fitted to 1738 calls of 62 shapes, every form."""
        total = (tiles * (batch + 1) + batch - 1) / 2 if spread else tiles * batch
        if spread:
            per = max(4, math.ceil((total - batch / 2) / (n_wgs - batch / 2)), -(-tiles // most))
            splits = min(n_wgs, math.ceil(total / per + batch / 2 * (1 - 1 / per)))
        else:
            per = max(4, -(-tiles // min(most, n_wgs // batch)))
            splits = batch * -(-tiles // per)
        f, c = MLADecodeOp.LENGTH_COST[heads]
        read = total * MLADecodeOp.BLOCK_N * 2e-6 * d / 4.8
        return (((-(-splits * -(-group // heads) // cus) * (f + c * per)) ** 4 + read ** 4) ** 0.25 + 0.32 * group * 4e-6 * dv * splits
                + 0.05 * most + 0.5)

    @staticmethod
    def _second_round(spans, n, n_ht, cus):
        """Whether equal spans, ``n`` an entry and ``n_ht`` head tiles each, take a second round of the CUs; ``spans``: how many of
        them hold keys, by entry.  More workgroups than CUs do.  Fewer may have to wait: ``ae_mla_decode_fwd`` pads an entry's ids
        to an odd number, an XCD deals its workgroups to its four shader engines in turn, in the order of their ids, and
        where the turn comes to an engine whose CUs are taken - by an empty workgroup too -, all behind it wait until one of those
        has ended.  Right about 563 of 566 full tables and 456 of 457 with lengths of 0.8 to 1 of them (B21 H64 2624 tokens, 32 heads a
        workgroup, 6 splits, 252 workgroups: full tables 40.6 us, entries spread evenly 23.7)."""
        if sum(spans) * n_ht > cus:
            return True
        ids = n | 1 if len(spans) * n * n_ht > 128 else n
        engine = max(1, cus // 32)
        for xcd in range(8):
            taken, waits, turn = [0] * 4, False, 0
            for unit in range(xcd, len(spans) * ids, 8):
                live = unit % ids < spans[unit // ids]
                for _ in range(n_ht):
                    waits = waits or taken[turn & 3] == engine
                    if waits and live:
                        return True
                    taken[turn & 3] += live
                    turn += 1
        return False

    @staticmethod
    @functools.lru_cache(maxsize=1024)
    def _splits_by_length(batch, group, tiles, fixed, cus, d, dv):
        """(query heads of a workgroup, the most splits of an entry, workgroups a head tile) for a paged call whose kernel cuts the
        entries by their lengths (``ae_split_by_length`` of csrc/kernels/ae_device.h), None where ``fixed``, (heads, splits) of
        equal spans of the table, is the better plan.

        Equal spans are planned for tables that may be full, and shorter entries leave workgroups without keys.  Cut by length,
        the workgroups of one round have about as many tiles each, but they wait for the lengths in front of their first request,
        0.2 to 0.8 us.  So tables whose equal spans are one round keep them: full ones would lose what spread entries gain (us,
        spread | full: B8 H128 2048 tokens 18.7 -> 17.4 | 19.9 -> 20.2, B9 H128 1792 20.0 -> 17.2 | 20.2 -> 21.7, B5 H128 4736 23.7 -> 20.7 |
        23.7 -> 24.5, B11 H64 3712 21.3 -> 19.0 | 22.5 -> 24.3).  By length go tables

        - whose equal spans take more than one round when they are full and also with lengths of 0.8 to 1 of the table (``_second_round``):
          of many spans the last ones of such entries are empty, and the others may fit a round (B16 H64, 8 spans: 1.05 of the time);
        - whose head tiles share a round's workgroups evenly (cut in shares of 85 and 42, 96 heads took up to 1.4 of the time),
          with no more than a fifth of them without a split when the entries are full (B46 H96, 0.28 of them: full tables 1.02 of the time);
        - with as many splits for a long entry as twice its share, so that it may be twice the mean, and more than equal spans
          give it (one long entry of 64: 46 us with 4 splits, 40 with 6, equal spans 43);
        - if by the costs spread entries take at most 0.96 of the time, and a spread and 0.7 of a full call no more than with equal
          spans (the costs of spread entries are 6 % off, of full tables 12 %: these decide little, the rounds most).

        905 such shapes (5 to 64 entries, 32 to 128 heads), time over that of equal spans, geometric mean (largest): lengths spread 0.76 (1.00), full
        0.75 (1.00), drawn evenly 0.77 (1.01), 0.8 to 1 of the table 0.79 (0.95), all half of it 0.69 (0.97), a quarter and all of it in
        turn 0.79 (1.02), one long entry among short ones 0.79 (0.98).  us, spread | full: B64 H128 4096 85.7 -> 61.9 | 130.8 -> 93.1, B21 H64 2624
        23.7 -> 20.9 | 40.6 -> 26.8.  Planned in 5 to 60 us, once a table width."""
        heads_fixed, n_fixed = fixed
        if batch < 4 or n_fixed == 1:
            return None
        best = None
        for heads in MLADecodeOp.LENGTH_COST:
            n_ht = -(-group // heads)
            n_wgs = cus // n_ht
            if (heads != 16 and group <= heads // 2) or cus % n_ht or batch > n_wgs or batch * (n_wgs // batch) < 0.8 * n_wgs:
                continue
            least = max(2 * n_wgs / batch, n_fixed + 1 if heads >= heads_fixed else 0)
            most = next((n for n in (2, 3, 4, 6, 8, 12, 16, 24) if n >= least), None)
            if most is None or 2 * most > tiles:
                continue
            full, spread = (MLADecodeOp._length_us(batch, group, tiles, heads, most, n_wgs, cus, d, dv, s) for s in (False, True))
            if best is None or spread + 0.7 * full < best[0]:
                best = spread + 0.7 * full, spread, (heads, most, n_wgs)
        if best is None:
            return None
        full, spread = (MLADecodeOp._call_us(batch, group, tiles, *fixed, cus, d, dv, s) for s in (False, True))
        if best[1] > 0.96 * spread or best[0] > spread + 0.7 * full:
            return None
        n_ht, per = -(-group // heads_fixed), -(-tiles // n_fixed)
        nearly_full = [min(n_fixed, math.ceil(tiles * (0.8 + i * 37 % 64 / 320) / per)) for i in range(batch)]
        if all(MLADecodeOp._second_round(spans, n_fixed, n_ht, cus) for spans in ([n_fixed] * batch, nearly_full)):
            return best[2]
        return None

    def plan(self, B, Hq, Hkv, Skv, page=None):
        """(query heads of a workgroup, number of splits, kv positions per split); with a paged cache a split spans at
        most as many pages as the kernel keeps table entries for, and where the kernel cuts the entries by their lengths
        (``_splits_by_length``) there is a fourth number, the workgroups a head tile that share them, and the second is the most splits of an entry.

        The wave-specialised kernel has forms for 16, 32 and 64 heads a workgroup: the fewer, the shorter a trip over
        one tile (0.59 / 0.73 / 0.81 us, paged 0.53 with 16 heads: the plans by this cost are 0.7 % off the best there)
        and the fewer splits - partial results - fill the chip, but the tiles are fetched by as many more workgroups.  B4 H128 Skv2048: 18.8 us with 64 heads and 16 splits, 13.9 with 16 and 8; B85 H64
        Skv445 39.4 us with 64 and 4 splits (340 workgroups: a second round for 84 of them), 18.4 with 32 and none;
        B128 H128 Skv4096 163.6 us with 64, 225.6 with 32."""
        group = Hq // Hkv
        tiles = -(-Skv // self.BLOCK_N)
        least = 1 if page is None else -(-Skv // ((self.PAGE_TABLE_ENTRIES - 2) * page))
        tuned = self._tuned.get((B, Hq, Hkv, Skv))

        def clamped(n):
            return max(1, min(tiles, max(n, least)))
        if self._wave_specialised():
            span = (clamped(tuned),) * 2 if tuned else (clamped(least), clamped(self.MAX_SPLITS))
            heads, n_split = self._cheapest(B * Hkv, group, tiles, span, self.target_workgroups, self.D, self.DV, page is not None)
            if page is not None and Hkv == 1 and B <= 64 and Skv // page + 2 <= self.PAGE_TABLE_ENTRIES and Skv <= 1 << 24 and not tuned:
                by_length = self._splits_by_length(B, group, tiles, (heads, n_split), self.target_workgroups, self.D, self.DV)
                if by_length is not None:
                    return by_length[0], by_length[1], -(-tiles // by_length[1]) * self.BLOCK_N, by_length[2]
        else:
            # as many splits as fill the chip, but no more than the merge is worth: B1 H128 Skv4096 takes 24 us with
            # 16 splits, 92 us with the 128 that would occupy every CU
            base = B * Hkv * -(-group // self.HEADS_PER_WG)
            want = clamped(tuned or min(-(-self.target_workgroups // base), self._balanced_splits(self.SPLIT_COEFF, Skv),
                                        self.MAX_SPLITS))
            heads, n_split = self.HEADS_PER_WG, -(-tiles // -(-tiles // want))           # no split without tiles
        return heads, n_split, -(-tiles // n_split) * self.BLOCK_N

    def plan_splits(self, B, Hq, Hkv, Skv, page=None):
        """(number of splits, kv positions per split) of ``plan``."""
        return self.plan(B, Hq, Hkv, Skv, page)[1:3]

    def _wave_specialised(self):
        """The wave-specialised kernel (scores computed once, a third of the LDS traffic) runs where the graph is the
        online softmax of scaled scores; the generic kernel runs any functor."""
        return (self.functors.softmax is not None and self.D % 64 == 0 and self.DV % 128 == 0 and self.D2 % 32 == 0
                and self.D // 16 >= 27      # its softmax is spread over 27 of the D/16 k-steps
                and os.environ.get("AE_MLA_KERNEL", "") != "generic")

    def _stamped(self, n_split):
        """AE_CLOCK_STAMPS=1 (a measurement switch, read by ``bench.py --mfma-probe``): single-split launches of the
        wave-specialised kernel report the shader clock their workgroups ran at (``self.clock_stamps``)."""
        return n_split == 1 and os.environ.get("AE_CLOCK_STAMPS", "") == "1" and self._wave_specialised()

    def _variant(self, n_split, paged=False, heads=64, by_length=False):
        """(module, cfg, config source) of the split kernel, one for every count of splits above 1.  ``heads``: query heads of a
        workgroup (AE_HPW of the wave-specialised kernel); ``by_length``: the entries of a paged cache are split by their lengths."""
        key = (n_split > 1, paged, heads, by_length, self._stamped(n_split))
        v = self._variants.get(key)
        if v is None:
            ws = self._wave_specialised()
            self.template = "ae_mla_decode_ws.hip" if ws else "ae_mla_decode.hip"
            cfg_src = render_mla_config(self.DV, self.D2, self.DV, self.dtype, self.BLOCK_N, self.K_PAD,
                                        self.n_rowscales, self.functors.o_scale_one, 2 if n_split > 1 else 1,
                                        self.functors.softmax if ws else None, paged, heads)
            if paged and ws and not by_length:
                cfg_src += "#define AE_BY_LENGTH 0\n"
            if key[-1]:
                cfg_src += "#define AE_CLOCK_STAMPS 1\n"
            module = rt.compile_module(self.template, {"ae_config.h": cfg_src, "ae_functors.h": self.functor_src},
                                       allow_spills=self.allow_spills)
            if ws:
                threads = 512
                lds = (self.WS_STAGES * self.BLOCK_N * 2 * self.D + 2 * heads * 80 + 2 * (heads * 4 + 16)
                       + heads * (8 if heads == 64 else 2 * 8 + 12)
                       + (4 * self.PAGE_TABLE_ENTRIES if paged else 0))
            else:
                threads = 512
                lds = self.N_STAGES * self.BLOCK_N * 2 * self.D
            cfg = rt.TileCfg(block_m=heads, block_n=self.BLOCK_N, threads=threads, lds_bytes=lds,
                             head_dim=self.D, head_dim_v=self.DV, elem_bytes=2,
                             n_rowscales=self.n_rowscales, mask_mode=0, paged=(2 if by_length else 1) if paged else 0)
            v = self._variants[key] = (module, cfg, cfg_src)
        return v

    def _call_paged(self, q, cache, block_table, cache_seqlens):
        """mod(q, kv_cache, block_table=..., cache_seqlens=...): the cache is read through the table."""
        for name, t in (("q", q), ("kv_cache", cache)):
            self._check_tensor(name, t)
        if block_table is None or cache_seqlens is None:
            raise TypeError("a paged call needs both block_table and cache_seqlens")
        for name, t in (("block_table", block_table), ("cache_seqlens", cache_seqlens)):
            if not (isinstance(t, torch.Tensor) and t.is_cuda and t.dtype == torch.int32):
                raise TypeError(f"{name} must be an int32 tensor on the GPU")
        if q.shape[-1] != self.D or cache.shape[-1] != self.D:
            raise ValueError(f"q / kv_cache last dim must be {self.D}")
        B, Sq, Hq, _ = q.shape
        n_pages, page, Hkv, _ = cache.shape
        if Sq != 1:
            raise ValueError("decode takes one query token per sequence")
        if Hq % Hkv:
            raise ValueError("inconsistent MLA shapes")
        if page % self.BLOCK_N:
            raise NotImplementedError(f"pages of {page} tokens: the kv tile of {self.BLOCK_N} tokens must not straddle pages")
        if block_table.dim() != 2 or block_table.shape[0] != B or block_table.stride(1) != 1:
            raise ValueError("block_table must be [batch, max pages per entry] with a contiguous last dimension")
        if cache_seqlens.shape != (B,) or not cache_seqlens.is_contiguous():
            raise ValueError("cache_seqlens must be a contiguous [batch] tensor")
        q = rt.rows_for_kernels(q)
        cache = rt.rows_for_kernels(cache)
        # the launch is planned for the longest entry the table can describe; the kernels stop at each
        # entry's own length (no device-to-host copy of cache_seqlens here)
        Skv = block_table.shape[1] * page
        return self._launch(q[..., :self.DV], q[..., self.DV:], cache[..., :self.DV], cache[..., self.DV:],
                            B, Hq, Hkv, Skv, paged=(block_table, cache_seqlens, page, n_pages))

    def __call__(self, *args, block_table=None, cache_seqlens=None):
        # a shape that has run before: csrc/ae_host.cpp
        done = (self._host.run_mla(*args) if block_table is None and cache_seqlens is None
                else self._host.run_mla(*args, block_table, cache_seqlens))
        if done is not None:
            self.final_rowscales = dict(zip(self.names, done[1:]))
            return done if self.cute else done[0]
        if block_table is not None or cache_seqlens is not None:
            if len(args) != 2:
                raise TypeError("block_table / cache_seqlens go with the call form mod(q, kv_cache)")
            return self._call_paged(args[0], args[1], block_table, cache_seqlens)
        if len(args) == 2:
            q, cache = args
            for name, t in (("q", q), ("kv_cache", cache)):
                self._check_tensor(name, t)
            if q.shape[-1] != self.D or cache.shape[-1] != self.D:
                raise ValueError(f"q / kv_cache last dim must be {self.D}")
            B = q.shape[0]
            Hkv = cache.shape[2]
            cache = cache if cache.is_contiguous() else cache.contiguous()
            kv_all = cache.reshape(B, -1, Hkv, self.D)          # identity block table: pages in order
            q = rt.rows_for_kernels(q)
            q1, q2 = q[..., :self.DV], q[..., self.DV:]
            k1, k2 = kv_all[..., :self.DV], kv_all[..., self.DV:]
        elif len(args) == 4:
            q1, q2, k1, k2 = args
            for name, t in (("q", q1), ("q_pe", q2), ("kv", k1), ("k_pe", k2)):
                self._check_tensor(name, t)
            q1, q2, k1, k2 = (rt.rows_for_kernels(t) for t in (q1, q2, k1, k2))
            if (q1.shape[3], q2.shape[3], k1.shape[3], k2.shape[3]) != (self.DV, self.D2, self.DV, self.D2):
                raise ValueError("q/q_pe/kv/k_pe head dims do not match the engine")
        else:
            raise TypeError("MLA decode is called as mod(q, q_pe, kv, k_pe) or mod(q, kv_cache)")
        B, Sq, Hq, _ = q1.shape
        _, Skv, Hkv, _ = k1.shape
        if Sq != 1:
            raise ValueError("decode takes one query token per sequence")
        if Hq % Hkv or k1.shape[0] != B or k2.shape[:3] != k1.shape[:3] or q2.shape[:3] != q1.shape[:3]:
            raise ValueError("inconsistent MLA shapes")
        return self._launch(q1, q2, k1, k2, B, Hq, Hkv, Skv)

    def _launch(self, q1, q2, k1, k2, B, Hq, Hkv, Skv, paged=None):
        dev = q1.device
        key = (B, Hq, Hkv, Skv)
        if self._tune_file and key not in self._tuned:
            page = paged[2] if paged is not None else None
            n0 = self.plan_splits(*key, page=page)[0]
            cands = [0] if len(self.plan(*key, page=page)) == 4 else []      # (0: the entries split by their lengths)
            self._tuned[key] = n0

            def made_of(n):
                self._tuned[key] = n
                got = self.plan_splits(*key, page=page)[0]
                self._tuned[key] = n0
                return got
            for n in (n0, n0 // 2, 2 * n0, 4 * n0, 8 * n0):
                got = made_of(max(1, n))
                if got not in cands:
                    cands.append(got)
            self._tuned[key] = n0
            self._tune_splits(key, cands, lambda: self._launch(q1, q2, k1, k2, B, Hq, Hkv, Skv, paged),
                              lambda n: n > 0 and made_of(n) == n)
        heads, n_split, kv_per_split, *by_length = self.plan(B, Hq, Hkv, Skv, page=paged[2] if paged is not None else None)
        module, cfg, _ = self._variant(n_split, paged is not None, heads, bool(by_length))
        ccfg = self._merges.cfg(n_split)
        out = torch.empty((B, 1, Hq, self.DV), dtype=self.dtype, device=dev)
        rowscales = [torch.empty((B, Hq, 1), dtype=torch.float32, device=dev) for _ in range(self.n_rowscales)]
        p = rt.AttnParams()
        p.q, p.q2, p.k, p.k2, p.v, p.out = (q1.data_ptr(), q2.data_ptr(), k1.data_ptr(), k2.data_ptr(),
                                            k1.data_ptr(), out.data_ptr())
        partial_o = partial_rs = None
        if n_split > 1:      # a single split writes `out` directly, no work buffers
            partial_o = torch.empty((B, Hq, n_split, self.DV), dtype=torch.float32, device=dev)
            partial_rs = torch.empty(max(1, self.n_rowscales) * B * Hq * n_split + (B if by_length else 0), dtype=torch.float32, device=dev)
            p.partial_o, p.partial_rs = partial_o.data_ptr(), partial_rs.data_ptr()
        if self._stamped(n_split):
            n_ht = -(-(Hq // Hkv) // heads)
            n_wg = -(-(B * Hkv) // 8) * 8 * n_ht
            self._stamp_buffer = torch.zeros(6 * n_wg, dtype=torch.int64, device=dev)
            self.clock_stamps = self._stamp_buffer[:2 * n_wg].view(n_wg, 2)     # (cycles, 100 MHz ticks) per workgroup
            self.phase_ticks = self._stamp_buffer[2 * n_wg:].view(n_wg, 4)      # entry, tile 0 landed, loop done, exit
            p.partial_o = self._stamp_buffer.data_ptr()
        for i, r in enumerate(rowscales):
            p.rowscale_out[i] = r.data_ptr()
        p.q_stride_b, p.q_stride_s, p.q_stride_h = q1.stride(0), q1.stride(1), q1.stride(2)
        p.q2_stride_b, p.q2_stride_s, p.q2_stride_h = q2.stride(0), q2.stride(1), q2.stride(2)
        p.k_stride_b, p.k_stride_s, p.k_stride_h = k1.stride(0), k1.stride(1), k1.stride(2)
        p.k2_stride_b, p.k2_stride_s, p.k2_stride_h = k2.stride(0), k2.stride(1), k2.stride(2)
        p.v_stride_b, p.v_stride_s, p.v_stride_h = k1.stride(0), k1.stride(1), k1.stride(2)
        p.o_stride_b, p.o_stride_s, p.o_stride_h = out.stride(0), out.stride(1), out.stride(2)
        p.batch, p.heads_q, p.heads_kv, p.seqlen_q, p.seqlen_kv = B, Hq, Hkv, 1, Skv
        p.num_splits, p.kv_per_split = n_split, kv_per_split
        if paged is not None:
            block_table, cache_seqlens, page, n_pages = paged
            p.block_table, p.seqlens_k = block_table.data_ptr(), cache_seqlens.data_ptr()
            p.block_table_stride, p.page_block_size, p.num_pages = block_table.stride(0), page, n_pages
            p.tail_slots = by_length[0] if by_length else 0
        split, combine, modules = module.kernel("ae_mla_decode_split_kernel"), None, (module,)
        if n_split > 1:
            modules += (self._merges.module(n_split),)
            combine = modules[1].kernel("ae_decode_combine_kernel")
        rt.mla_decode_fwd(split, combine, p, cfg, ccfg, rt.current_stream(dev))
        if not self._stamped(n_split) and (self.n_rowscales == 1 or not self.cute):
            host.add_forward(self._host, host.MLA if paged is None else host.MLA_PAGED, B, 1, Hq, Hkv, Skv, dev, modules, split,
                             cfg, combine=combine, ccfg=ccfg, n_split=n_split, kv_per_split=kv_per_split,
                             page=paged[2] if paged is not None else 0, tail_slots=by_length[0] if by_length else 0)
        self.final_rowscales = dict(zip(self.names, rowscales))
        self._keepalive = [partial_o, partial_rs, q1, q2, k1, k2, paged]
        if self.cute:
            lse = rowscales[0] if rowscales else None
            return out, lse
        return out

    def _check_tensor(self, name, t):
        if not (isinstance(t, torch.Tensor) and t.is_cuda):
            raise RuntimeError(f"{name} must be a tensor on the GPU (there is no CPU path)")
        if t.dtype != self.dtype:
            raise TypeError(f"{name} has dtype {t.dtype}, the engine was built for {self.dtype}")
        if t.dim() != 4:
            raise ValueError(f"{name} must be 4-dimensional")
