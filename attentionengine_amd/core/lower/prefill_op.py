"""Prefill operator: owns the compiled kernel variants of one AttentionEngine and launches them.

Host-side counterpart of the reference's generated ``_attention.forward`` + ``tl.compile`` result
(attention_engine/core/template/tl_template/attn/attn_tl.py:523-528, 567-580; block-sparse:
blockattn_tl.py:401-447): takes q/k/v ``[B,S,H,D]`` plus the CustomIO tensors (and, when a block
mask is in play, that mask as the LAST positional argument), allocates ``o`` and the final
rowscales, launches on torch's current stream, returns ``o``.
"""
from __future__ import annotations

import functools
import math
import os
from dataclasses import astuple

import torch

from ..runtime import hip_rt as rt
from ..runtime import host
from ..transform.core import _convert_mask_to_block_mask, is_causal_mask
from . import lower as L
from .lower_decode import Merges, lower_combine, merges_in_any_order
from .mask import plan_mask, survey_mask


def _dim(x, default):
    return default if isinstance(x, str) else int(x)


class PrefillOp:
    MASK_ROWS_PER_TILE = 8      # block-mask rows one q tile may span (AE_TT_ROWS of csrc/kernels/ae_tile_table.h)

    def __init__(self, qkv_meta, custom_fwd_inputs, score_mod, mask_mod, online_func, mask_value,
                 infer_mask=True, infer_mask_block_M=128, infer_mask_block_N=128,
                 extern_block_mask=False, split_kv=False, target_workgroups=256,
                 tiles=None, tune=False, tune_file="", tune_bwd=False, tune_file_bwd="",
                 exact_scale=None, defer_norm=None, allow_spills=None):
        self._ctor = ((qkv_meta, custom_fwd_inputs, score_mod, mask_mod, online_func, mask_value),
                      dict(infer_mask=infer_mask, infer_mask_block_M=infer_mask_block_M,
                           infer_mask_block_N=infer_mask_block_N, extern_block_mask=extern_block_mask,
                           split_kv=split_kv, target_workgroups=target_workgroups,
                           exact_scale=exact_scale, defer_norm=defer_norm, allow_spills=allow_spills))
        # numerics switches (see AttentionEngine): None = the default of the kernel / lowering
        self.exact_scale = exact_scale
        # None: a build that moves register tuples through scratch memory is reported, False: it is refused
        # (hip_rt.check_spills); where the pipelined kernel was this operator's own choice it then gives way to the
        # generic one, see _gives_way_to_the_generic_kernel
        self.allow_spills = allow_spills
        self._tiles_given = tiles is not None
        q_meta, k_meta, v_meta = qkv_meta
        self.dtype = q_meta.dtype
        self.D = int(q_meta.shape[3])
        self.DV = int(v_meta.shape[3])
        if int(k_meta.shape[3]) != self.D:
            raise ValueError("q and k head dims differ")
        if self.D % 16 or self.DV % 32:
            raise NotImplementedError(f"head dims (D={self.D}, DV={self.DV}) must be multiples of 16 / 32")
        # Value head dim 512 with head dim 64 / 128 / 256 (attn_script/retention.py: D 256, DV 512) runs in one
        # launch of the direct-to-LDS kernel: 256 accumulator registers per lane, one wave per SIMD, its
        # epilogue working block by block.  Other value head dims above 256 run as several launches over
        # column slices of V and of the output (the scores are recomputed per slice; the row scales of every
        # launch are the same); AE_DV_SLICE=1 forces that form.
        self.DV_launch = self.DV
        single_pass = (self.D in (64, 128, 256) and self.DV == 512 and os.environ.get("AE_DV_SLICE", "") != "1"
                       and not split_kv)
        if self.DV > 256 and not single_pass:
            self.DV_launch = next(c for c in (256, 192, 128, 96, 64, 32) if self.DV % c == 0)
        self.mask_mod, self._probed, self._surveys = mask_mod, None, {}
        self.elementwise_mask = mask_mod is not None and mask_value == "-inf"
        self.mask_value_zero = mask_value == "0"
        self.extern_block_mask = bool(extern_block_mask)
        self.mask_block = (int(infer_mask_block_M), int(infer_mask_block_N))
        self.functors = L.trace_functors(score_mod, mask_mod, online_func, custom_fwd_inputs,
                                         self.dtype, mask_value, defer_norm=defer_norm)
        self._graph = (score_mod, online_func, custom_fwd_inputs)     # the backward traces score_mod again
        self.functor_src = L.render_functors(self.functors)
        # what the software-pipelined kernel can run: the proven online softmax, or an elementwise graph
        # (masked scores are -inf before score_mod there, as in the reference: not with mask_value "0")
        self._pipe_softmax = None if self.mask_value_zero else self.functors.softmax
        self._pipe_elementwise = (self._pipe_softmax is None and self.functors.elementwise
                                  and not self.mask_value_zero)
        self.tiles = L.choose_prefill_tiles(self.D, self.DV_launch, _dim(q_meta.shape[2], 0),
                                            self._pipe_softmax,
                                            _dim(q_meta.shape[0], 1) * _dim(q_meta.shape[1], 1),
                                            elementwise=self._pipe_elementwise,
                                            seqlen_kv=_dim(k_meta.shape[2], 0),
                                            bf16=self.dtype == torch.bfloat16, masked=mask_mod is not None)
        # Masks that reach the kernel as a tile table (anything but none / exactly causal) go to the generic
        # kernel: with its 128-row q tiles fewer tiles are partly visible, and its masked path costs less than
        # the pipelined kernel's (B2 H32 S4096 D128, sliding window of 256: 0.13 against 0.31 ms; a random block
        # mask that keeps 27 %: 0.22 against 0.35 ms).  tune=True still measures both.
        if self.tiles.rows_per_wave == 64 and os.environ.get("AE_PREFILL_KERNEL", "") != "pipelined" and (
                self.extern_block_mask or (mask_mod is not None and self._probe_mask(q_meta, v_meta).mode == 2)):
            self.tiles = L.PrefillTiles()
        self._table_tiles = L.PrefillTiles() if split_kv else self.tiles     # ... of a call that brings a block mask
        # Band masks are read in 32-key tiles (B2 H32 S4096 D128, window of 256: 94.8 -> 88.4 us with them, of 1024 184 -> 180):
        # less of the band's edges is multiplied.  At head dim 64, whose tiles cost more to start than to multiply, only
        # narrow ones (B3 H16 S2719, window 133: 22.0 -> 20.3; B1 H16 S6102 of 655 55.5 against 59.6 with 32 keys, B4 H16
        # S1278 of 856 23.5 against 24.4; 26 windows of 180 to 1000 keys: 3 % on average, 12 at most).
        if self.mask_mod is not None and self.tiles == L.PrefillTiles() and self.D in (64, 128) and self.DV in (64, 128):
            band = self._probe_mask(q_meta, v_meta).band
            if band is not None and band[1] is not None and (max(self.D, self.DV) > 64 or band[1] - band[0] < 180):
                self.tiles = L.PrefillTiles(block_n=32)
        # Launches that leave the chip idle with these tiles: waves that share the kv axis.  That depends on the extents
        # of a call, so an engine declared at such extents decides again for every shape it is called with (tiles_for);
        # self.tiles are the declared shape's, self._base what the other shapes use where the kv axis is not shared.
        self.split_kv = bool(split_kv)
        self._base = L.PrefillTiles() if self.split_kv else self.tiles
        shape = (q_meta.shape[0], q_meta.shape[1], q_meta.shape[2], v_meta.shape[2])
        self._declared = None if any(isinstance(x, str) for x in shape) else tuple(int(x) for x in shape)
        groups = self._groups = self._kv_group_choice(
            *self._declared, lambda found: self._probe_mask(q_meta, v_meta)) if self._declared else None
        if groups is not None:
            self.tiles = groups
        self._call_tiles = {}      # (B, H, Sq, Skv) other than the declared ones -> tiles_for()
        self._causal_generic = {}  # (B, H, Sq, Skv) -> _causal_choice() takes the generic kernel
        # tune=True (attn_tl.py:465-521 of the reference): the tile configuration comes from the record of
        # this problem in tune_file, or is measured at the first call and recorded there.  Launches whose
        # tiles are bound to something else (split-KV, an external block mask) keep the fixed choice.
        self._tune_file, self._tune_pending, self._tune_found, self.tune_times = "", False, False, None
        self._tune_bwd = (bool(tune_bwd), tune_file_bwd)
        if tiles is not None:
            self.tiles = tiles
        elif tune and tune_file and not split_kv and not extern_block_mask:
            from . import tuner
            self._tune_file = tune_file
            self._tune_keys = tuner.problem_keys(q_meta.shape, self.D, self.DV)
            found = tuner.decode_tiles(tuner.lookup(tune_file, self._tune_keys), self._tune_candidates())
            if found is not None:
                self.tiles, self._tune_found = found, True
            else:
                self._tune_pending = True
        # Split-KV ("MHA decode": a few query tokens against a long KV, attn_engine.py:273-290 and
        # core/lower/lower_decode.py:287-313 of the reference): the kv axis is shared out over several
        # workgroups per q tile and the partial results are merged with the user's combine().
        self.target_workgroups = int(target_workgroups)
        # Bytes of work memory that one call may take for launches that share tiles out over several workgroups where the chip
        # would idle (_tail, PrefillBwdOp.dkv_parts), or that keep ds for the dq launch (PrefillBwdOp.keeps_ds): allocated per
        # call, given back with it.  None: 128 MB in the forward, 256 MB and, for ds, 2.5 GB in the backward.  0: no tile is
        # shared out, nothing kept.
        self._work_limit = None
        if self.split_kv:
            if self.tiles.template == "ae_prefill_simple.hip" or max(self.D, self.DV) > 128:
                raise NotImplementedError("split-KV prefill needs head dims 64 or 128")
            if self.DV_launch != self.DV:
                raise NotImplementedError("split-KV prefill with a value head dim above 256")
            if not hasattr(online_func, "combine"):
                raise NotImplementedError("split-KV needs OnlineFunc.combine to merge the partial results")
            if tiles is None and groups is None:
                self.tiles = L.PrefillTiles()      # the generic kernel carries the split-KV mode
            names = self.functors.final_rowscale_names
            self.functor_src += lower_combine(online_func, names)
            self._merges = Merges(self.D, self.DV, self.dtype, len(names), self.functor_src, merges_in_any_order(online_func, names),
                                  self.COMBINE_THREADS, allow_spills)
        if self.extern_block_mask and self.tiles.rows_per_wave != 32 and (
                self.mask_block[1] % self.tiles.block_n or
                (self.tiles.block_m % self.mask_block[0] and self.mask_block[0] % self.tiles.block_m)):
            self.tiles = L.PrefillTiles()     # the pipelined kernel's kv tile is fixed; use the generic one
        if self.extern_block_mask:
            # a q tile covers whole block-mask rows, a kv tile sits inside one block-mask column
            while self.tiles.block_n > self.mask_block[1] and self.tiles.block_n > 32:
                self.tiles.block_n //= 2
            if self.tiles.block_m > self.MASK_ROWS_PER_TILE * self.mask_block[0]:
                self.tiles = L.PrefillTiles(block_n=self.tiles.block_n)   # 128-row q tiles span fewer table rows
            if (self.tiles.block_m % self.mask_block[0] and self.mask_block[0] % self.tiles.block_m) or \
                    self.mask_block[1] % self.tiles.block_n or \
                    self.tiles.block_m > self.MASK_ROWS_PER_TILE * self.mask_block[0]:
                raise NotImplementedError(f"block mask granularity {self.mask_block} does not fit the tiles")
        if self.tiles.kv_groups == 1 and self.tiles is not groups:
            self._base = self.tiles
        if self._tiles_given or self.extern_block_mask or self._tune_found:
            self._table_tiles = self._base
        self.n_rowscales = len(self.functors.final_rowscale_names)
        if self.n_rowscales > rt.AE_MAX_ROWSCALES or len(self.functors.customs) > rt.AE_MAX_CUSTOM:
            raise NotImplementedError("too many rowscales / custom inputs")
        self.final_rowscales = {}
        self.block_mask = None
        # calls of a shape that has run before (csrc/ae_host.cpp)
        self._host = host.new_host(self.D, self.DV, self.dtype, self.functors.customs, self.n_rowscales)
        self._variants = {}   # (mask_mode, even_q, even_kv) -> (module, cfg, config_src)
        self._plans = {}      # (B|1, H|1, Sq, Skv) -> MaskPlan with device table
        self.meta_shape = (_dim(q_meta.shape[0], 1), _dim(q_meta.shape[1], 1), _dim(q_meta.shape[2], 0),
                           _dim(v_meta.shape[2], 0))
        # compile for the declared shape now (hipRTC needs no GPU) so construction reports
        # lowering/compile errors, like the reference's constructor does
        B, H, Sq, Skv = self.meta_shape
        self.source = self.functor_src
        if Sq > 0:
            try:
                self._compile_declared_shape(B, H, Sq, Skv, infer_mask, mask_mod)
            except rt.SpillError:
                if not self._gives_way_to_the_generic_kernel():
                    raise
                self._compile_declared_shape(B, H, Sq, Skv, infer_mask, mask_mod)

    @property
    def work_limit(self):
        return self._work_limit

    @work_limit.setter
    def work_limit(self, n):
        self._work_limit = n
        self._host.clear()         # (plans made under the old one)

    def work_limit_mb(self, default):
        return default if self._work_limit is None else self._work_limit * 1e-6

    def _gives_way_to_the_generic_kernel(self) -> bool:
        """A build of the software-pipelined kernel that spills registers is refused (hip_rt.check_spills).  Where
        that kernel was this operator's own choice -- not the caller's (``tiles=``, the tuner) -- the operator
        switches to the generic kernel, whose two waves per SIMD leave the compiler room, for every later launch:
        True if it did.  (The pipelined kernel holds 64 query rows per wave in one wave per SIMD and fills the
        register file; its fp16 builds fit, some bf16 builds at head dim 128 spill a few values.)"""
        if self._tiles_given or self._base.template != "ae_prefill_pipe.hip":
            return False
        if self.tiles == self._base:
            self.tiles = L.PrefillTiles()
        self._base = self._table_tiles = L.PrefillTiles()
        self._call_tiles.clear()
        self._causal_generic.clear()
        self._variants.clear()
        self._plans.clear()
        self._host.clear()
        self._bwd = None            # (the backward reads this operator's mask plans: built again on demand)
        self.gave_way_to_generic = True
        return True

    def _compile_declared_shape(self, B, H, Sq, Skv, infer_mask, mask_mod):
        tiles = self._launch_tiles(B, H, Sq, Skv, self.tiles_for(B, H, Sq, Skv))
        plan = self._plan(B, H, Sq, Skv, device=None, tiles=tiles)
        mode = 2 if self.extern_block_mask else plan.mode
        n_split, _ = self.plan_splits(B, H, Sq, Skv, tiles)
        _, _, cfg_src = self._variant(tiles, mode, Sq, Skv, n_split,
                                      self._table_rows(self.mask_block[0] if self.extern_block_mask else plan.block_m, tiles),
                                      plan.heavy_last and not self.extern_block_mask,
                                      None if self.extern_block_mask else self._band(plan, tiles))
        self.source = cfg_src + "\n" + self.functor_src
        if n_split > 1:
            self.source = self._merges.config(n_split) + self.source
        if infer_mask and mask_mod is not None and not self.extern_block_mask:
            self.block_mask = self._reference_block_mask(B, H, Sq, Skv)

    def _probe_mask(self, q_meta, v_meta):
        """The mask plan at the declared sequence lengths (4096 where they are dynamic), for batch entry and head 0:
        mode 2 = the mask needs a tile table (or is a band)."""
        if self._probed is None:
            sq, skv = _dim(q_meta.shape[2], 4096), _dim(v_meta.shape[2], 4096)
            self._probed = plan_mask(self.mask_mod, self.functors.mask, 1, 1, sq, skv, 128, 64,
                                     elementwise=self.elementwise_mask, survey=self._mask_survey(1, 1, sq, skv))
        return self._probed

    def _mask_survey(self, B, H, Sq, Skv):
        """The mask evaluated at these extents: once for all tile shapes that are tried there (the last few are kept)."""
        lm = self.functors.mask
        key = (B if lm.uses_b else 1, H if lm.uses_h else 1, Sq, Skv)
        found = self._surveys.get(key)
        if found is None:
            if len(self._surveys) >= 4:
                self._surveys.pop(next(iter(self._surveys)))
            found = self._surveys[key] = survey_mask(self.mask_mod, lm, B, H, Sq, Skv)
        return found

    def _kv_group_choice(self, B, H, Sq, Skv, mask_plan):
        """Tiles whose waves share the kv axis, where this engine's graph, its mask (``mask_plan(tiles)``) and the extents
        allow and want them: a merge the kernel knows (the proven online softmax, or no row state), no mask table, no
        tensor read per score."""
        wide = (self.D, self.DV) == (192, 128)          # (measured for causal softmax only)
        if (not (B and H and Sq and Skv) or not (wide or (self.D in (64, 128) and self.DV in (64, 128)))
                or (wide and (self.mask_mod is None or self._pipe_softmax is None or self.split_kv))
                or not self._groups_can_meet()):
            return None
        if self.split_kv:
            return L.kv_group_tiles_split(Sq, B * H) if self.mask_mod is None else None
        if self.mask_mod is not None and max(self.D, self.DV) == 64:
            # (a window's workgroups do not differ in length as a causal mask's do: four groups a CU are too many where
            # 64-row tiles outnumber the places for them.  B3 H16 S755, window 121: 11.7 -> 8.4 us, B3 H16 S1155 of 862
            # 24.1 -> 19.0, B1 H16 S3095 of 146 11.9 -> 11.1)
            two = L.window_group_tiles(B * H, Sq)
            band = mask_plan(two).band if two is not None else None
            if band is not None and band[1] is not None and not (self.functors.mask.uses_b or self.functors.mask.uses_h):
                return two
        found = L.kv_group_tiles(self.D, self.DV, B * H, Sq, Skv, self.mask_mod is not None)
        if found is not None and self.mask_mod is not None:
            lm = self.functors.mask
            if lm.uses_b or lm.uses_h:
                return None
            plan = mask_plan(found)
            if not (plan.mode == 1 or (plan.band is not None and not wide)):
                return None
        return found

    def _groups_can_meet(self):
        """Whether this engine's graph lets waves share the kv axis, and nothing asks for another kernel."""
        return not (self.extern_block_mask or not (self._pipe_softmax is not None or self._pipe_elementwise)
                    or any(c.per_kv for c in self.functors.customs) or os.environ.get("AE_PREFILL_KERNEL", ""))

    def tiles_for(self, B, H, Sq, Skv):
        """The tile configuration of a call with these extents."""
        key = (B, H, Sq, Skv)
        if key == self._declared or (self.tiles.kv_groups == 1 and self.tiles is not self._groups):
            return self._call_choice(key, self.tiles)
        tiles = self._call_tiles.get(key)
        if tiles is None:
            tiles = self._call_tiles[key] = self._kv_group_choice(
                *key, lambda found: self._plan(*key, device=None, tiles=found)) or self._base
        return self._call_choice(key, tiles)

    def _call_choice(self, key, tiles):
        """``tiles``, or where they are this operator's own choice what is faster for a call with these extents."""
        if self._tiles_given or self._tune_file or self.extern_block_mask or self.split_kv or (self.D, self.DV) != (128, 128):
            return tiles
        if self.mask_mod is not None:
            return self._causal_choice(key, tiles)
        B, H, Sq, Skv = key
        if (tiles == L.PrefillTiles() and (self._pipe_softmax is not None or self._pipe_elementwise) and Sq and Skv
                and not any(c.per_kv for c in self.functors.customs) and not os.environ.get("AE_PREFILL_KERNEL", "")
                and L.short_key_tiles_pay(B * H, Sq, Skv)):
            return L.PrefillTiles(block_n=32)
        return tiles

    def _causal_choice(self, key, tiles):
        """``tiles``, or the generic kernel's where they are the pipelined kernel's by this operator's own choice, would be at
        these extents too, and a causal call is faster in the generic one (lower.pipelined_pays)."""
        B, H, Sq, Skv = key
        if tiles.template != "ae_prefill_pipe.hip" or self._pipe_softmax is None or Sq != Skv or not Sq:
            return tiles
        generic = self._causal_generic.get(key)
        if generic is None:
            bf16 = self.dtype == torch.bfloat16
            generic = self._causal_generic[key] = (
                os.environ.get("AE_PREFILL_KERNEL", "") != "pipelined" and not L.pipelined_pays(bf16, B * H, Sq)
                and L.choose_prefill_tiles(self.D, self.DV, Sq, self._pipe_softmax, B * H, seqlen_kv=Skv, bf16=bf16) == tiles
                and self._plan(*key, device=None, tiles=tiles).mode == 1)
        return L.PrefillTiles() if generic else tiles

    # ---- tuning ------------------------------------------------------------------------
    def _tune_candidates(self):
        from . import tuner
        cands = tuner.prefill_candidates(self.D, self.DV_launch, self._pipe_softmax, self._pipe_elementwise)
        return cands if self._groups is None else cands + [self._groups]

    def _tune(self, q, k, v, *extra):
        """Measures every candidate tile configuration on the caller's tensors, becomes the fastest one and
        records it under this engine's problem keys (AE_TUNE_VERBOSE=1 prints the measurements)."""
        from . import tuner
        self._tune_pending = False
        args, kw = self._ctor
        log = print if os.environ.get("AE_TUNE_VERBOSE", "") == "1" else None
        cands = self._tune_candidates()
        mine = self.block_mask      # the engine appends this very object to every call: see _forward

        def run(o):
            return o._forward(q, k, v, *[o.block_mask if (mine is not None and x is mine) else x for x in extra])
        best, op, times = tuner.pick(
            cands, lambda t: self if t == self.tiles else PrefillOp(*args, **kw, tiles=t), run, log)
        if op is not self:
            keep = (self._ctor, self._tune_file, self._tune_keys, self._tune_bwd, self._work_limit, mine)
            self.__dict__.update(op.__dict__)
            self._ctor, self._tune_file, self._tune_keys, self._tune_bwd, self._work_limit, self.block_mask = keep
            self._bwd = None        # the backward reads this operator's mask plans: built again on demand
        self._tune_pending = False
        self.tune_times = {tuple(tuner.encode_tiles(cands[i])): ms for i, ms in times.items()}
        tuner.store(self._tune_file, self._tune_keys, tuner.encode_tiles(best))

    # ---- mask --------------------------------------------------------------------------
    def _plan(self, B, H, Sq, Skv, device, tiles=None):
        tiles = tiles or self.tiles_for(B, H, Sq, Skv)
        key = (B, H, Sq, Skv, tiles.block_m, tiles.block_n)
        plan = self._plans.get(key)
        if plan is None:
            plan = plan_mask(self.mask_mod, self.functors.mask, B, H, Sq, Skv, tiles.block_m, tiles.block_n,
                             elementwise=self.elementwise_mask,
                             survey=self._mask_survey(B, H, Sq, Skv) if self.mask_mod is not None else None)
            self._plans[key] = plan
        if device is not None and plan.table is not None and plan.table.device != device and self._band(plan, tiles) is None:
            plan.table = plan.table.to(device)
        return plan

    def _reference_block_mask(self, B, H, Sq, Skv):
        """The block mask the reference would keep on ``mod.block_mask`` (lower.py:721-738):
        int8 [B,H,Sq/bm,Skv/bn] "any element visible", or None when it is exactly block-causal
        (dense template)."""
        bm, bn = self.mask_block
        lm = self.functors.mask
        mb, mh = (B if lm.uses_b else 1), (H if lm.uses_h else 1)
        rows = []
        kv = torch.arange(Skv).view(1, 1, 1, Skv)
        for r0 in range(0, Sq, bm * 8):
            r1 = min(Sq, r0 + bm * 8)
            q = torch.arange(r0, r1).view(1, 1, -1, 1)
            m = self.mask_mod(torch.arange(mb).view(mb, 1, 1, 1), torch.arange(mh).view(1, mh, 1, 1), q, kv)
            if not isinstance(m, torch.Tensor):
                m = torch.tensor(bool(m))
            m = m.to(torch.bool).expand(mb, mh, r1 - r0, Skv)
            rows.append(_convert_mask_to_block_mask(m, bm, bn)[0])
        blocks = torch.cat(rows, dim=2).expand(B, H, -1, -1)
        if Sq == Skv and bool(is_causal_mask(blocks, bm, bn)):
            return None
        return blocks.contiguous()

    # ---- kernels -------------------------------------------------------------------------
    COMBINE_THREADS = 128

    # Head dim 128: tiles of a split launch whose workgroups have a CU each.  Three stages keep two tiles on their way while one
    # is multiplied; with two, what is on its way drains at the end of every trip (not where eight waves multiply for 1.4 us:
    # B7 H16 Sq192 Skv12126 199.9 us, 201.1 with three).  name -> (tiles, microseconds of a
    # workgroup's start and end, of a trip over its kv groups' next tiles)
    SPLIT_FORMS = {"32": (dict(n_waves=1, kv_groups=2, block_n=32, kv_stages=3), 3.14, 0.69),
                   "64": (dict(n_waves=2, kv_groups=2, block_n=32, kv_stages=3), 3.2, 0.72),
                   "128": (dict(kv_stages=3), 3.3, 1.0),
                   "256": (dict(n_waves=8), 3.3, 1.43)}

    def _launch_tiles(self, B, H, Sq, Skv, tiles):
        """The tiles of a split launch with these extents: those of ``SPLIT_FORMS`` that cost least instead of ``tiles``
        (``tiles_for``), where the graph allows them.  Not at other head dims, nor where 128- or 256-row tiles fill the chip
        without a split (two workgroups a CU then hide each other's waits: B10 H32 Sq108 Skv2102 79 us, 92 with three stages),
        nor where ``tiles`` are one launch that is as good (``_own_tiles_pay``)."""
        if (not self.split_kv or self.mask_mod is not None or (self.D, self.DV) != (128, 128) or self._tiles_given
                or not (B and H and Sq and Skv) or Sq > 256 or (Sq > 64 and -(-(B * H) // 8) * 8 > self.target_workgroups)
                or not self._groups_can_meet() or self._own_tiles_pay(B, H, Sq, Skv, tiles)):
            return tiles
        names = ("32",) if Sq <= 32 else ("64",) if Sq <= 64 else ("64", "128", "256")
        return L.PrefillTiles(**self.SPLIT_FORMS[self._cheapest_form(names, B * H, Sq, -(-Skv // 32), self.target_workgroups)[0]][0])

    def _own_tiles_pay(self, B, H, Sq, Skv, tiles):
        """Whether up to 64 rows keep ``tiles``: one split of them, with two stages, against the cheapest of ``SPLIT_FORMS``.  Short
        caches, where four kv groups share the trips (32-row tiles) and no partial result is written, up to a number of heads:
        B3 H32 Sq30 Skv704 12.9 -> 11.2 us, B3 H16 Sq19 Skv353 9.6 -> 7.7, B3 H32 Sq37 Skv651 14.2 -> 12.7; 0.956 of the time
        on 101 shapes of at most 32 rows (1.06 at most); but B5 H32 Sq45 Skv500 1.11.  More than 32 rows of more heads than there
        are CUs: two workgroups share a CU, with three stages the last ones wait for a place: B9 H32 Sq61 Skv521 28.7 -> 23.2, B16 H32
        Sq61 Skv521 35.5 -> 31.2, 0.80 of the time up to 800 keys, 0.97 at 3000 to 4000, where the plan starts to split."""
        heads, cus = B * H, self.target_workgroups
        short = Skv <= 768 and heads <= (cus * 5 // 8 if Sq <= 32 else cus // 2)
        return Sq <= 64 and (short or (Sq > 32 and heads > cus)) and self.plan_splits(B, H, Sq, Skv, tiles)[0] == 1

    def _split_form_of(self, tiles):
        """The name in ``SPLIT_FORMS`` of tiles that ``_launch_tiles`` chose, or None."""
        if (self.D, self.DV) != (128, 128):
            return None
        return next((n for n, f in self.SPLIT_FORMS.items() if tiles == L.PrefillTiles(**f[0])), None)

    @classmethod
    @functools.lru_cache(maxsize=1024)
    def _cheapest_form(cls, names, heads, rows, kv_tiles, cus):
        """(tiles, splits) of a split launch at head dim 128 that takes least time, ``kv_tiles`` counted in 32 keys.  Every CU has
        one workgroup at a time, so a launch takes whole rounds of starts and trips; the cache arrives at 6.4 TB/s; partial
        results are written and merged.  Fitted to 1000 timings of 94 shapes (batch 1 to 8, 8 to 32 heads, 1 to 256 rows, 512
        to 16384 keys, bf16), 3.6 % off in the root mean square; the choice is 0.6 % off the best measured on average and
        takes 0.93 of the time of two stages with a split for every CU (1.05 at most).  us: B6 H32 Sq50 Skv2562 60 -> 51,
        B8 H8 Sq115 Skv521 15.9 -> 12.2, B1 H16 Sq4 Skv8393 20.7 -> 19.2, B5 H32 Sq216 Skv3498 112 -> 99, B1 H32 Sq128 Skv8192
        42.2 -> 39.4.  Splits that take a second round where one split would not start and drain twice, 12 % of
        the read by 3600 shapes: B5 H32 Sq61 Skv15254, 232 with two stages, 244 with three splits, 226 with one."""
        read = heads * kv_tiles * 32 * 512e-6 / 6.4
        best = []
        for name in names:
            tiles, start, trip = cls.SPLIT_FORMS[name]
            tiles = L.PrefillTiles(**tiles)
            n = -(-kv_tiles * 32 // tiles.block_n)
            wgs = -(-rows // tiles.block_m) * (-(-heads // 8) * 8)
            for x in range(1, min(64, n) + 1):
                if x > 1 and wgs * x > 4 * cus:
                    break
                per = -(-n // x)
                if -(-n // per) != x:
                    continue
                body = -(-wgs * x // cus) * (start + trip * -(-per // tiles.kv_groups))
                us = (body ** 2.25 + read ** 2.25) ** (1 / 2.25)
                if wgs <= cus < wgs * x:
                    us += 0.12 * read
                if x > 1:
                    us += 1.8 + 0.047 * x + 0.42 * heads * rows * x * 512e-6
                best.append((us, x, name))
        least = min(best)[0]
        _, x, name = min((b for b in best if b[0] <= 1.01 * least), key=lambda b: (b[1], b[0]))
        return name, x

    # microseconds of a workgroup's start and end, and of a trip over its kv groups' next tiles, by the rows of its q tile
    SPLIT_COST = {32: (3.0, 0.92), 64: (1.8, 0.66), 128: (1.3, 0.91), 256: (5.2, 1.39)}
    # head dim 64: (start and end, trip, what a trip takes of each workgroup that shares the CU, workgroups a CU holds)
    SPLIT_COST_64 = {32: (2.04, 0.63, 0.44, 2), 64: (2.25, 0.53, 0.31, 4), 128: (1.66, 0.77, 0.57, 4), 256: (4.7, 1.0, 0.0, 2)}

    @classmethod
    @functools.lru_cache(maxsize=1024)
    def _cheapest_splits(cls, wgs, rows, kv_tiles, block_m, block_n, kv_groups, width, cus, heads):
        """Kv tiles of a split, for launches that one split for every CU would leave with two workgroups on some CUs and
        one on the others: two share a CU's issue slots and its lines on the way, so that the launch takes as long as two
        rounds.  A call takes its rounds of starts and trips (half rounds beyond the second, where workgroups no longer
        end together), at least what memory needs for the cache (8.4 TB/s while the memory-side cache holds it, else 6.2),
        and the partial results: written and merged.  Fitted to 1926 timings (150 shapes, batch 1 to 8, 8 to 32 heads, 1
        to 256 rows, 512 to 16384 keys, D128, two tile stages): 1 % above the best count on average.  Measured, one split for every CU ->
        this: B7 H16 Sq31 Skv522 17.6 -> 9.2 us.  (At head dim 128 only for tiles that ``_launch_tiles`` leaves as they are, as there, and
        at 64 / 128 columns; the others have ``_cheapest_form``.)  ``width``: bytes of a key and a value row in units of 512.

        At head dim 64 two to four workgroups fit a CU, and a launch of two on some CUs is no second round: with the costs of
        D128 17 of 71 choices were slower than one split for every CU (B7 H32 Sq47 Skv5777 70.5 -> 93.9 us).  Its own costs
        are fitted to 130 shapes; where the count is chosen by them, 40 others take 0.89 of the time on average, 1.04 at most
        (that one 63.5 us)."""
        if width <= 0.5:
            return cls._cheapest_splits_64(wgs, rows, kv_tiles, block_m, block_n, kv_groups, cus, heads)
        start, trip = cls.SPLIT_COST[block_m]
        read = heads * kv_tiles * block_n * 512e-6 * width
        read /= 8.4 if read <= 300 else 6.2
        best = []
        for x in range(1, min(64, kv_tiles) + 1):
            per = -(-kv_tiles // x)
            if -(-kv_tiles // per) != x:
                continue
            rounds, r = -(-wgs * x // cus), wgs * x / cus
            if r > 8 and x > 1:
                break
            if r > 2:
                rounds = 0.5 * (rounds + r) + 0.26
            body = rounds * (start + trip * width * -(-per // kv_groups))
            merge = 2.7 + 0.056 * x + 0.285 * rows * x * 512e-6 * width if x > 1 else 0.0
            best.append((2.3 + (body ** 1.85 + read ** 1.85) ** (1 / 1.85) + merge, per))
        least = min(best)[0]
        return next(per for us, per in best if us <= 1.01 * least)

    @classmethod
    def _cheapest_splits_64(cls, wgs, rows, kv_tiles, block_m, block_n, kv_groups, cus, heads):
        start, trip, share, fit = cls.SPLIT_COST_64[block_m]
        read = heads * kv_tiles * block_n * 256e-6
        read /= 7.1 if read <= 300 else 5.3
        best = []
        for x in range(1, min(64, kv_tiles) + 1):
            per = -(-kv_tiles // x)
            if -(-kv_tiles // per) != x:
                continue
            trips, a_cu = -(-per // kv_groups), wgs * x / cus
            if a_cu > 8 and x > 1:
                break
            full = start + max(trip, share * fit) * trips                  # a round of as many workgroups as a CU holds
            rounds, rest = divmod(a_cu, fit)
            body = rounds * full + (start + max(trip, share * math.ceil(rest)) * trips if rest > 0 else 0.0)
            if a_cu > fit:
                body = 0.5 * (body + a_cu / fit * full) + 0.3 * start
            merge = 3.5 + 0.061 * x + 0.315 * rows * x * 256e-6 if x > 1 else 0.0
            best.append((1.2 + (body ** 2.46 + read ** 2.46) ** (1 / 2.46) + merge, per))
        return min(best)[1]

    def plan_splits(self, B, Hq, Sq, Skv, tiles=None):
        """(number of KV splits, kv positions per split): a workgroup for every CU of the chip (more splits cost
        more in partial results and their merge than they gain: B1 H32 Sq128 Skv8192, the shape of
        attn_script/mha_inference.py, two tile stages, 43 us with 8 splits, 44 with 16, 75 with 32), whole kv tiles per split, no
        empty split.  Where that leaves some CUs with two workgroups the cheapest count is taken (``_cheapest_splits``), and
        always for the tiles that are chosen with it (``_launch_tiles``)."""
        if not self.split_kv:
            return 1, Skv
        tiles = tiles or self.tiles_for(B, Hq, Sq, Skv)
        bn = tiles.block_n
        kv_tiles = -(-Skv // bn)
        form = self._split_form_of(tiles)
        if form:
            x = self._cheapest_form((form,), B * Hq, Sq, -(-Skv // 32), self.target_workgroups)[1]
            return x, -(-kv_tiles // x) * bn
        wgs = -(-Sq // tiles.block_m) * (-(-(B * Hq) // 8) * 8)
        want = max(1, min(kv_tiles, -(-self.target_workgroups // wgs)))
        per = -(-kv_tiles // want)
        if wgs * -(-kv_tiles // per) > self.target_workgroups and tiles.block_m in self.SPLIT_COST:
            per = self._cheapest_splits(wgs, B * Hq * Sq, kv_tiles, tiles.block_m, bn, tiles.kv_groups,
                                        (self.D + self.DV) / 256, self.target_workgroups, B * Hq)
        return -(-kv_tiles // per), per * bn

    MAX_TAIL_PARTS = 8        # kMaxParts of ae_prefill_pipe.hip

    @classmethod
    @functools.lru_cache(maxsize=1024)
    def _tail_plan(cls, slots, kv_tiles, cus_per_xcd, width, limit_mb=128):
        """(q tiles of an XCD, workgroups of each, kv tiles of a workgroup) that share their kv axes in an unmasked launch of the
        pipelined kernel with ``slots`` q tiles an XCD (AE_TAIL of ae_prefill_pipe.hip), or None: what is left over when the
        CUs have been filled as often as possible would take a round of its own.  A workgroup takes 7 us to start and end
        and 2.0 us a kv tile (D128); shares are few (the last workgroup reads all of them, about 1.2 us each), and taken
        where the call gains 6 % by this count - what it says is 3 % turned out between -7 and +2.  Measured: softmax B3 H8
        S2944 D128 fp16 162 -> 117 us, bf16 174 -> 120, B1 H32 S2560 sigmoid bf16 155 -> 115 (40 tiles an XCD), B1 H40 S3584
        (70) 301 -> 250, D64 B2 H16 S4200 231 -> 178, sigmoid fp16 B3 H16 S1325 83 -> 68; 56 of 64 tiles: 232 -> 230.  On 49
        shapes beside those the choice is 0.5 % off the best count on average (B2 H8 S2293 bf16, 18 tiles an XCD: 71.7 us, 64.2
        unshared; else 3 % at most), at D64 on 48 shapes 0.4 %, 7 at most."""
        rounds, rest = divmod(slots, cus_per_xcd)
        if not rest:
            return None
        start, trip = 7.0, 2.0 * width
        whole = start + trip * kv_tiles
        best = None
        for n in range(2, cls.MAX_TAIL_PARTS + 1):
            per = -(-kv_tiles // n)
            if -(-kv_tiles // per) != n or 8 * rest * n * 0.136 * width > limit_mb:      # (MB of partial results)
                continue
            us = -(-rest * n // cus_per_xcd) * (start + trip * per) + 3.0 + 1.2 * n * width
            if best is None or us < best[0]:
                best = us, n, per
        if best is None or (rounds * whole + best[0]) > 0.94 * (rounds + 1) * whole:
            return None
        return rest, best[1], best[2]

    def _tail(self, B, H, Sq, Skv, tiles, mode, n_split):
        if (tiles.template != "ae_prefill_pipe.hip" or mode != 0 or n_split > 1 or self.DV_launch != self.DV
                or self._clock_stamps(tiles)):
            return None
        return self._tail_plan(-(-Sq // tiles.block_m) * -(-(B * H) // 8), -(-Skv // tiles.block_n),
                               L._MI355X_CUS // 8, (self.D + self.DV) / 256, self.work_limit_mb(128))

    def _kv_custom_scratch(self, tiles) -> int:
        """LDS a launch needs beyond its K / V stages: the direct-to-LDS kernel redistributes the tiles of custom
        inputs with a kv dimension (fetched in a coalesced layout) through 2560 bytes per wave and 32-row block
        (AE_KV_SCRATCH of ae_prefill.hip; its builds with two waves per SIMD)."""
        if (tiles.template != "ae_prefill.hip" or tiles.waves_per_eu < 2
                or not any(c.per_kv for c in self.functors.customs)):
            return 0
        return tiles.n_waves * (tiles.rows_per_wave // 32) * 2560

    def _clock_stamps(self, tiles):
        """AE_CLOCK_STAMPS=1 (a measurement switch, read by ``bench.py --mfma-probe``): the pipelined kernel is
        built so that every workgroup reports the shader-clock cycles and the 100 MHz ticks it ran for; the
        pairs of the last launch are kept on ``self.clock_stamps`` (int64 [workgroups, 2])."""
        return os.environ.get("AE_CLOCK_STAMPS", "") == "1" and tiles.template == "ae_prefill_pipe.hip"

    def _table_rows(self, mask_block_m, tiles):
        """Block-table rows a q tile spans (1, 2, 4 or 8): the kernels keep that many pairs of 64-bit masks."""
        if not mask_block_m:
            return 1
        rows = max(1, -(-tiles.block_m // int(mask_block_m)))
        return next(r for r in (1, 2, 4, 8) if r >= min(rows, 8))

    def _band(self, plan, tiles):
        """The mask's band (MaskPlan.band) where the kernel takes one instead of the tile table."""
        return plan.band if tiles.template == "ae_prefill.hip" else None

    MERGED_SPLITS, MERGED_VALUES = 8, 8192      # (the first: of ae_merge_last.h)

    def _merges_in_last(self, Hq, Sq, tiles, n_split):
        """Whether the workgroup that finishes last of a q tile merges (AE_MERGE_LAST of ae_prefill.hip) instead of a second
        launch (not in a graph: see ae_host.cpp): few values are read by that one workgroup, few counts are constants of its
        build.  48 shapes (batch 1 to 8, 8 to 32 heads, 1 to 25 rows, 512 to 16384 keys, head dims 64 and 128), time of the call in
        units of that with two launches: 0.94 on average, 0.81 to 1.003 (D64 B3 H8 Sq8 Skv764, 8 splits, 9.9 us -> 8.0; D128
        B4 H32 Sq5 Skv1496, 2 splits, 23.2 -> 21.8; B4 H16 Sq12 Skv14418, 4 splits, 89.4 -> 89.6).  Beyond: 8192 to 16384
        values 0.92 to 1.20, 9 to 12 splits 0.93 to 1.10, 13 to 16 0.95 to 1.18."""
        return (1 < n_split <= self.MERGED_SPLITS and self._can_merge_in_last(tiles)
                and min(Sq, tiles.block_m) * n_split * self.DV <= self.MERGED_VALUES
                and tiles.block_m * Hq * n_split * self.DV < 2**29)

    def _can_merge_in_last(self, tiles):
        """Whether a split launch's build can: the merge's 32 loads a thread in flight take up to 190 registers, which those of 32
        rows have (at most two waves a SIMD)."""
        return (tiles.template == "ae_prefill.hip" and tiles.block_m == 32 and tiles.kv_groups > 1 and tiles.waves_per_eu == 2
                and self._merges.any_order)

    def _variant(self, tiles, mask_mode, Sq, Skv, n_split=1, table_rows=1, heavy_last=False, band=None,
                 tail=False):
        even_q, even_kv = Sq % tiles.block_m == 0, Skv % tiles.block_n == 0
        if mask_mode != 2 or band is not None:
            table_rows = 1
        if mask_mode != 2:
            heavy_last = False
        key = (mask_mode, even_q, even_kv, n_split > 1, table_rows, bool(heavy_last), band, astuple(tiles), tail,
               self._clock_stamps(tiles))
        v = self._variants.get(key)
        if v is None:
            has_mask_mod = self.elementwise_mask and mask_mode != 1
            own_softmax = tiles.template == "ae_prefill.hip" and self._pipe_softmax is not None and tiles.waves_per_eu >= 2
            cfg_src = L.render_config(self.D, self.DV_launch, self.dtype, tiles, mask_mode, has_mask_mod,
                                      self.n_rowscales, self.functors.o_scale_one, even_q, even_kv,
                                      self._pipe_softmax if tiles.rows_per_wave == 64 or tiles.kv_groups > 1 or own_softmax else None,
                                      elementwise=self._pipe_elementwise and tiles.rows_per_wave == 64,
                                      exact_scale=self.exact_scale)
            if self.mask_value_zero:
                cfg_src += "#define AE_MASK_VALUE_ZERO 1\n"
            else:
                if self.functors.softmax is not None:
                    cfg_src += "#define AE_PAD_GIVES_ZERO 1\n"
                if self.functors.elementwise:
                    cfg_src += "#define AE_ELEMENTWISE 1\n"
            if mask_mode == 2:
                cfg_src += f"#define AE_TT_ROWS {table_rows}\n#define AE_HEAVY_LAST {1 if heavy_last else 0}\n"
            if band is not None:
                cfg_src += (f"#define AE_BAND 1\n#define AE_BAND_LO ({band[0]})\n"
                            f"#define AE_BAND_HI {'0x7fffffff' if band[1] is None else f'({band[1]})'}\n")
            if own_softmax:
                cfg_src += "#define AE_OWN_SOFTMAX 1\n"
                if self.split_kv and tiles.kv_groups > 1 and self._split_form_of(tiles):
                    cfg_src += "#define AE_FIRST_REST 1\n"
            if n_split > 1:
                cfg_src += "#define AE_NSPLIT 2\n"       # (a split launch; its count is the launch's)
                if self._can_merge_in_last(tiles):
                    cfg_src += "#define AE_MERGE_LAST 1\n"
            if key[-1]:
                cfg_src += "#define AE_CLOCK_STAMPS 1\n"
            if tail:
                cfg_src += "#define AE_TAIL 1\n"
            module = rt.compile_module(tiles.template, {"ae_config.h": cfg_src,
                                                          "ae_functors.h": self.functor_src},
                                       allow_spills=self.allow_spills,
                                       # the builds in which a spilled tuple came back wrong: 256 accumulator registers
                                       strict_spills=tiles.template == "ae_prefill.hip" and self.DV_launch > 256)
            cfg = rt.TileCfg(block_m=tiles.block_m, block_n=tiles.block_n,
                             threads=tiles.threads,
                             lds_bytes=tiles.lds_bytes(self.D, self.DV_launch) + self._kv_custom_scratch(tiles), head_dim=self.D,
                             head_dim_v=self.DV_launch, elem_bytes=2, n_rowscales=self.n_rowscales,
                             mask_mode=mask_mode if band is None else 1,      # (a band is analytic: no table comes with the call)
                             table_rows=table_rows if mask_mode == 2 and band is None else 0,
                             merge_in_wg=2 if tail else 0)
            v = self._variants[key] = (module, cfg, cfg_src)
        return v

    # ---- launch ----------------------------------------------------------------------------
    def __call__(self, q, k, v, *extra):
        """Forward; records the autograd edge when a gradient of q, k or v is wanted (the reference's
        generated ``_attention`` autograd function, attn_tl.py:530-640).  A call whose shape has run before is
        checked and launched natively (csrc/ae_host.cpp), autograd edge included."""
        if extra and extra[-1] is self.block_mask and self.block_mask is not None and not self.extern_block_mask:
            done = self._host.run(q, k, v, *extra[:-1])        # (the mask inferred from mask_mod itself: see _forward_once)
        else:
            done = self._host.run(q, k, v, *extra)
        if done is not None:
            self.final_rowscales = dict(zip(self.functors.final_rowscale_names, done[1:]))
            return done[0]
        if torch.is_grad_enabled() and any(isinstance(t, torch.Tensor) and t.requires_grad for t in (q, k, v)):
            return _PrefillFunction.apply(self, q, k, v, *extra)
        return self._forward(q, k, v, *extra)

    def backward_op(self):
        if getattr(self, "_bwd", None) is None:
            from .prefill_bwd_op import PrefillBwdOp
            self._bwd = PrefillBwdOp(self, *self._graph, tune=self._tune_bwd[0], tune_file=self._tune_bwd[1],
                                     allow_spills=self.allow_spills)
        return self._bwd

    def _forward(self, q, k, v, *extra):
        try:
            return self._forward_once(q, k, v, *extra)
        except rt.SpillError:
            # (raised by the compilation of a variant, before anything was launched)
            if not self._gives_way_to_the_generic_kernel():
                raise
            return self._forward_once(q, k, v, *extra)

    def _forward_once(self, q, k, v, *extra):
        if self._tune_pending:
            self._tune(q, k, v, *extra)
        n_custom = len(self.functors.customs)
        extern_mask = None
        if len(extra) == n_custom + 1:
            extern_mask = extra[-1]
            extra = extra[:-1]
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
        Bk, Skv, Hkv, Dk = k.shape
        if (D, Dk, v.shape[3]) != (self.D, self.D, self.DV):
            raise ValueError(f"head dims {(D, Dk, v.shape[3])} differ from the compiled {(self.D, self.D, self.DV)}")
        if Bk != B or v.shape[0] != B or v.shape[1] != Skv or v.shape[2] != Hkv or Hq % Hkv:
            raise ValueError("inconsistent q/k/v shapes")
        q, k, v = (rt.rows_for_kernels(t) for t in (q, k, v))
        dev = q.device

        if extern_mask is not None and extern_mask is self.block_mask and not self.extern_block_mask:
            # the block mask this engine inferred from mask_mod itself (AttentionEngine appends it to every
            # call, attn_engine.py:391-392 of the reference): the tile-class table planned from the same
            # mask_mod says the same at the kernel's own tile granularity, whatever infer_mask_block_M/N are
            extern_mask = None
        tiles = self.tiles_for(B, Hq, Sq, Skv)
        if extern_mask is not None:
            tiles = self._table_tiles
            bm, bn = self.mask_block
            if bn % tiles.block_n or (tiles.block_m % bm and bm % tiles.block_m) or \
                    tiles.block_m > self.MASK_ROWS_PER_TILE * bm:
                raise NotImplementedError(
                    f"a block mask of {bm}x{bn} blocks does not fit the kernel's {tiles.block_m}x"
                    f"{tiles.block_n} tiles (construct the engine with extern_block_mask=True)")
            table = extern_mask
            if table.dim() != 4:
                raise ValueError("block_mask must be [B|1, H|1, Sq/bm, Skv/bn]")
            if table.dtype != torch.int8:
                table = table.to(torch.int8)
            table = table.to(dev).contiguous()
            mode, mbm, mbn, band = 2, bm, bn, None
        else:
            tiles = self._launch_tiles(B, Hq, Sq, Skv, tiles)
            plan = self._plan(B, Hq, Sq, Skv, dev, tiles)
            mode, table, mbm, mbn, band = plan.mode, plan.table, plan.block_m, plan.block_n, self._band(plan, tiles)
        n_split, kv_per_split = self.plan_splits(B, Hq, Sq, Skv, tiles)
        tail = self._tail(B, Hq, Sq, Skv, tiles, mode, n_split)
        module, cfg, _ = self._variant(tiles, mode, Sq, Skv, n_split, self._table_rows(mbm, tiles) if mode == 2 else 1,
                                       extern_mask is None and plan.heavy_last, band, tail is not None)
        kern = module.kernel("ae_prefill_kernel")

        out = torch.empty((B, Sq, Hq, self.DV), dtype=self.dtype, device=dev)
        rowscales = [torch.empty((B, Hq, Sq), dtype=torch.float32, device=dev) for _ in range(self.n_rowscales)]
        p = rt.AttnParams()
        p.q, p.k, p.v, p.out = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()
        p.q_stride_b, p.q_stride_s, p.q_stride_h, _ = q.stride()
        p.k_stride_b, p.k_stride_s, p.k_stride_h, _ = k.stride()
        p.v_stride_b, p.v_stride_s, p.v_stride_h, _ = v.stride()
        p.o_stride_b, p.o_stride_s, p.o_stride_h, _ = out.stride()
        p.batch, p.heads_q, p.heads_kv, p.seqlen_q, p.seqlen_kv = B, Hq, Hkv, Sq, Skv
        for i, r in enumerate(rowscales):
            p.rowscale_out[i] = r.data_ptr()
        keep = []
        for i, (desc, t) in enumerate(zip(self.functors.customs, extra)):
            t = t.to(device=dev, dtype=desc.torch_dtype).contiguous()
            keep.append(t)
            p.custom[i] = t.data_ptr()
        if mode == 2 and band is None:
            p.block_mask = table.data_ptr()
            p.mask_b, p.mask_h, p.mask_nq, p.mask_nkv = table.shape
            p.mask_block_m, p.mask_block_n = mbm, mbn
            keep.append(table)
        stream = rt.current_stream(dev)
        if n_split > 1:
            partial_o = torch.empty((B, Sq, Hq, n_split, self.DV), dtype=torch.float32, device=dev)
            partial_rs = torch.empty((max(1, self.n_rowscales), B, Sq, Hq, n_split), dtype=torch.float32, device=dev)
            modules, ccfg = (module, self._merges.module(n_split)), self._merges.cfg(n_split)
            combine = modules[1].kernel("ae_decode_combine_kernel")
            shared = {"n_split": n_split, "kv_per_split": kv_per_split}
            if self._merges_in_last(Hq, Sq, tiles, n_split):       # (from the next call on: the host path keeps the counters)
                shared["counters"] = B * Hq * -(-Sq // tiles.block_m)
            p.partial_o, p.partial_rs = partial_o.data_ptr(), partial_rs.data_ptr()
            p.num_splits, p.kv_per_split = n_split, kv_per_split
            keep += [partial_o, partial_rs]
            rt.prefill_split_fwd(kern, combine, p, cfg, ccfg, stream)
        else:
            modules, combine, ccfg, shared = (module,), None, None, {}
            if tail is not None:
                p.tail_slots, p.num_splits, p.kv_per_split = tail[0], tail[1], tail[2] * tiles.block_n
                shared = {"n_split": tail[1], "kv_per_split": p.kv_per_split, "tail_slots": tail[0], "counters": 8 * tail[0],
                          "o_rows": 8 * tail[0] * tail[1] * (tiles.block_m + 4 * tiles.threads // self.DV)}
                partial_o = torch.empty((shared["o_rows"], self.DV), dtype=torch.float32, device=dev)
                counters = self._host.work(1, 1, shared["counters"], dev.index, stream, True)[1]
                p.partial_o, p.partial_rs = partial_o.data_ptr(), counters.data_ptr() + 4
                keep += [partial_o, counters]
            if self._clock_stamps(tiles):
                n_wg = -(-Sq // tiles.block_m) * (-(-(B * Hq) // 8) * 8)
                self.clock_stamps = torch.zeros((n_wg, 2), dtype=torch.int64, device=dev)
                p.partial_o = self.clock_stamps.data_ptr()
            # one launch per slice of DV_launch value columns (a single one unless DV > 256)
            esz = v.element_size()
            for c0 in range(0, self.DV, self.DV_launch):
                p.v = v.data_ptr() + c0 * esz
                p.out = out.data_ptr() + c0 * esz
                rt.prefill_fwd(kern, p, cfg, stream)
        self.final_rowscales = dict(zip(self.functors.final_rowscale_names, rowscales))
        self._keepalive = keep
        if extern_mask is None and self.DV_launch == self.DV and not self._clock_stamps(tiles):
            host.add_forward(self._host, host.PREFILL_SPLIT if n_split > 1 else host.PREFILL, B, Sq, Hq, Hkv, Skv, dev,
                             modules, kern, cfg, combine=combine, ccfg=ccfg, **shared,
                             table=table if mode == 2 and band is None else None, mask_block=(mbm, mbn), env=("AE_CLOCK_STAMPS",))
        return out


class _PrefillFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, op, q, k, v, *extra):
        # `extra`: the block mask the engine inferred from mask_mod, which it appends to every call (the
        # backward applies mask_mod per element instead); custom inputs and external masks are refused.
        # A graph without a backward still runs forward on tensors that require gradients -- a caller who
        # only wants `out` from leaf tensors gets it -- and says so when .backward() is called, as the
        # reference does (its generated _attention.backward is where a missing rule surfaces,
        # attn_tl.py:582-640).
        try:
            bwd, ctx.no_backward = op.backward_op(), None
        except NotImplementedError as e:
            bwd, ctx.no_backward = None, e
        with torch.no_grad():
            out = op._forward(q.detach(), k.detach(), v.detach(), *extra)
        ctx.op = op
        ctx.n_extra = len(extra)
        if bwd is None:
            return out
        ctx.customs = tuple(extra[:len(op.functors.customs)])       # scalar CustomIO tensors of score_mod
        # the user's block mask of this call (engines built with extern_block_mask=True): last positional
        ctx.block_mask = extra[-1] if (op.extern_block_mask and len(extra) == len(op.functors.customs) + 1) else None
        # the final row scales the backward reads: lse, or every final row scale of an online function whose
        # forward() / backward() are traced
        scales = [op.final_rowscales[n] for n in bwd.rowscale_names] or [q.new_empty(0)]
        ctx.save_for_backward(q, k, v, out, *scales)
        return out

    @staticmethod
    def backward(ctx, dout):
        if ctx.no_backward is not None:
            raise NotImplementedError(str(ctx.no_backward)) from ctx.no_backward
        q, k, v, out, *scales = ctx.saved_tensors
        lse = scales[0] if len(scales) == 1 else scales
        dq, dk, dv = ctx.op.backward_op()(q, k, v, out, lse, dout, ctx.customs, ctx.block_mask)
        return (None, dq, dk, dv) + (None,) * ctx.n_extra
