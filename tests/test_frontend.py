"""CPU tests of the host side: symbolic tracer, mask utilities (product code vs the oracle's brute
force), mask_mod lowering, functor emission + hipRTC compilation (no GPU needed), engine dispatch
and error behaviour."""
import math
import sys

import numpy as np
import pytest
import torch

import attn_cases as C
from attn_engine import AttentionEngine, OnlineFunc
from core import CustomIO, SymbolicArray, SymbolScalar, Var, create_block_mask, create_mask, meta_tensor
from core.lower import lower as L
from core.lower.lower_decode import lower_combine
from core.lower.mask import lower_mask_mod, plan_mask
from core.transform.core import (SymbolicConst, create_block_idx, is_causal_mask, is_less_causal_mask)
from oracle import masks as M


# ---- tracer ---------------------------------------------------------------------------------------
def test_tracer_builds_the_softmax_graph():
    """Node sequence of OnlineSoftmax.online_fwd as traced from attn_script/mha.py:47-63."""
    on = C.OnlineSoftmax()
    scores = SymbolicArray("scores", Var("scores"), shape_idx=["block_M", "block_N"])
    b = h = q = SymbolScalar("b", Var("b"))
    s2, rows, o_scale = on.online_fwd(scores, on.online_rowscales, b, h, q)
    assert s2.code.type == "Exp" and s2.prev[0].code.type == "Sub"
    assert s2.shape_idx == ["block_M", "block_N"]
    m_new = rows["m"]
    assert m_new.code.type == "Max" and m_new.prev[1].code.type == "ReduceMax"
    assert m_new.prev[1].shape_idx == ["block_M"] and m_new.prev[1].varname == "scores_max_0"
    assert rows["r"].code.type == "Add" and rows["r"].prev[1].code.type == "ReduceSum"
    assert o_scale.code.type == "Exp" and o_scale.prev[0].prev[1] is m_new
    # naming rule <varname>[_<suffix>]_<use count>
    assert m_new.varname == "m_0"


def test_python_numbers_become_constants_on_either_side():
    x = SymbolScalar("x", Var("x"))
    y = (x * 2 + 1.5) / 3
    assert y.code.type == "Div" and isinstance(y.prev[1], SymbolicConst) and y.prev[1].code.value == 3
    z = 1 - x
    assert z.code.type == "Sub" and z.prev[0].code.type == "Const" and z.prev[1] is x
    with pytest.raises(TypeError):
        x + "a"


def test_customio_declares_symbolic_tensors():
    io = CustomIO({"softmax_bias": (1,), "slopes": ("heads",)})
    assert io.input_tensors["softmax_bias"].shape_idx == ["1"]
    assert io.input_tensors["slopes"].shape_idx == ["heads"]


# ---- masks (product) vs brute force (oracle) --------------------------------------------------------
@pytest.mark.parametrize("mask_mod", [C.causal_mask, C.causal_plus_one_mask, C.causal_shifted_mask,
                                      C.make_sliding_window_mask(100), C.head_dependent_mask])
def test_create_mask_and_block_mask_match_brute_force(mask_mod):
    B, H, S = 2, 4, 512
    dense = create_mask(mask_mod, B, H, S, S, device="cpu")
    ref = M.dense_mask_grid(mask_mod, B, H, S, S)
    assert dense.dtype == torch.bool and np.array_equal(dense.numpy(), ref)
    blocks = create_block_mask(mask_mod, B, H, S, S, "cpu", 128, 64)
    assert blocks.dtype == torch.int8 and np.array_equal(blocks.numpy(), M.block_any(ref, 128, 64))
    assert bool(is_causal_mask(blocks, 128, 64)) == bool(
        np.array_equal(np.broadcast_to(M.block_causal_pattern(4, 8, 128, 64), blocks.shape), blocks.numpy().astype(bool)))
    assert bool(is_less_causal_mask(blocks, 128, 64)) == M.no_block_above_diagonal(blocks.numpy(), 128, 64)
    idx = create_block_idx(mask_mod, B, H, S, S, "cpu", 128, 64)
    assert idx.shape == (int(blocks.sum()), 4)


def test_block_mask_known_answers_of_the_reference_test_script():
    """attention_engine/tests/test_blockmask.py:3-27 prints these; values hand-derived."""
    for mask_mod, last, causal, less in [(C.causal_mask, [1, 3, 5, 7], True, True),
                                         (C.causal_plus_one_mask, [2, 4, 6, 7], False, False),
                                         (C.causal_shifted_mask, [-1, 1, 3, 5], False, True)]:
        blocks = create_block_mask(mask_mod, 2, 4, 512, 512, "cpu", 128, 64)
        for i, l in enumerate(last):
            assert blocks[0, 0, i].tolist() == [1] * (l + 1) + [0] * (7 - l)
        assert bool(is_causal_mask(blocks, 128, 64)) == causal
        assert bool(is_less_causal_mask(blocks, 128, 64)) == less


def test_ragged_block_mask_pads_with_invisible():
    blocks = create_block_mask(C.causal_mask, 1, 1, 200, 200, "cpu", 128, 64)
    assert blocks.shape == (1, 1, 2, 4)
    assert blocks[0, 0].tolist() == [[1, 1, 0, 0], [1, 1, 1, 1]]


def test_mask_plan_classes_match_oracle():
    for mask_mod in (C.causal_plus_one_mask, C.make_sliding_window_mask(100), C.head_dependent_mask):
        lm = lower_mask_mod(mask_mod)
        plan = plan_mask(mask_mod, lm, 2, 4, 300, 300, 128, 64, chunk_rows=128)
        assert plan.mode == 2
        mb, mh = (2 if lm.uses_b else 1), (4 if lm.uses_h else 1)
        ref = M.block_classes(M.dense_mask_grid(mask_mod, mb, mh, 300, 300), 128, 64)
        assert np.array_equal(plan.table.numpy(), ref)
    lm = lower_mask_mod(C.causal_mask)
    assert plan_mask(C.causal_mask, lm, 2, 4, 300, 300, 128, 64).mode == 1
    assert not lm.uses_b and not lm.uses_h
    assert lower_mask_mod(C.head_dependent_mask).uses_h


def test_mask_mod_lowering_text_and_unsupported_ops():
    lm = lower_mask_mod(C.make_sliding_window_mask(256))
    assert "n_ge" in lm.body and "(bool)(n_ge) & (bool)(n_lt)" in lm.body and "return (bool)" in lm.body

    def bad(b, h, q_idx, kv_idx):
        return torch.sin(q_idx) > kv_idx
    with pytest.raises(NotImplementedError):
        lower_mask_mod(bad)


# ---- functor emission -----------------------------------------------------------------------------
def test_emitted_softmax_functors():
    lf = L.trace_functors(C.make_scale_score_mod(0.125), C.causal_mask, C.OnlineSoftmax(), CustomIO({}),
                          torch.float16)
    assert lf.rowstate_fields == ["m", "r"] and lf.rowstate_init == ["-1e38f", "0.0f"]
    assert lf.final_rowscale_names == ["lse"] and not lf.o_scale_one
    body = lf.online_fwd_body
    assert "ae_row_sum<N>" in body
    # affine folding: the score scale is applied to the row maximum (one multiply per row) and
    # folded with log2(e) into the exponent, one fma + exp2 per element, no separate scaling pass
    assert "ae_row_max<N>(s) * 0.125f" in body
    assert f"ae_exp2(__builtin_fmaf(s[e], {0.125 * 1.4426950408889634!r}f" in body
    assert "s[e] * 0.125f" not in body
    # the graph is recognised as the online softmax: thresholded (lazy) running maximum
    assert "> 5.545177444479562f) ?" in body and "ae_max(st.m" not in body
    assert "frs[0]" in lf.epilogue_body and "ae_log(st.r)" in lf.epilogue_body
    src = L.render_functors(lf)
    for name in ("ae_score_mod", "ae_online_fwd", "ae_epilogue", "ae_mask_mod", "ae_rowstate_init"):
        assert name in src


def test_emitted_identity_and_custom_scalar():
    lf = L.trace_functors(C.make_sigmoid_score_mod(0.1), None, C.OnlineIdentity(),
                          CustomIO({"softmax_bias": (1,)}), torch.float16)
    assert lf.o_scale_one and lf.rowstate_fields == [] and lf.final_rowscale_names == []
    assert lf.customs[0].name == "softmax_bias" and lf.customs[0].torch_dtype == torch.float32
    # ((x*0.5).tanh() + 1) * 0.5 is the logistic function: one exp2 and one reciprocal per score
    assert "ae_rcp(1.0f + ae_exp2(__builtin_fmaf(s[e], -0.14426950" in lf.online_fwd_body
    assert "ae_tanh" not in lf.online_fwd_body and "cust.softmax_bias" in lf.online_fwd_body


def test_affine_of_tanh_forms():
    """a*tanh(x)+b with literal constants: the logistic special case, the general case, and a bare
    tanh (sigmoid script form attn_script/sigmoidattn.py:14-18; tanh semantics tl_gen.py:113-117)."""
    def lower(f):
        return L.trace_functors(f, None, C.OnlineIdentity(), CustomIO({}), torch.float16).online_fwd_body
    gen = lower(lambda s, c, b, h, q, kv: 3.0 - (s * 0.25).tanh() * 2.0)           # a = -2, b = 3
    assert "__builtin_fmaf(ae_rcp(ae_exp2(s[e] * 0.72134752" in gen and ", 4.0f, 1.0f)" in gen
    bare = lower(lambda s, c, b, h, q, kv: (s * 0.25).tanh())
    assert "ae_tanh" in bare
    # the rewritten forms agree with the definition
    import math
    for x in (-30.0, -2.0, -0.1, 0.0, 0.3, 5.0, 40.0):
        e = 2.0 ** (2 * 0.25 * x * 1.4426950408889634)
        assert abs((1.0 / (e + 1.0)) * 4.0 + 1.0 - (3.0 - 2.0 * math.tanh(0.25 * x))) < 1e-12
        assert abs(1.0 / (1.0 + 2.0 ** (-x * 1.4426950408889634)) - 0.5 * (math.tanh(0.5 * x) + 1)) < 1e-12


def test_unsupported_graphs_raise():
    class Bad(OnlineFunc):
        def __init__(self):
            super().__init__({"m": SymbolScalar("m", Var("banana"))}, {}, CustomIO())
    with pytest.raises(NotImplementedError):
        L.trace_functors(None, None, Bad(), CustomIO({}), torch.float16)
    with pytest.raises(NotImplementedError):   # an unknown dimension name in a custom input's shape
        L.trace_functors(lambda s, c, b, h, q, kv: s * c.input_tensors["x"], None, C.OnlineIdentity(),
                         CustomIO({"x": (1, "channels")}), torch.float16)


def test_custom_input_with_a_kv_dimension_is_read_per_score():
    """The retention decay mask (attn_script/retention.py:14-16, lower.py:590-597 of the reference):
    a [1,H,S,S] input is indexed by the lane's row once and by kv position inside the tile loop."""
    lf = L.trace_functors(C.retention_score_mod, C.causal_mask, C.OnlineAbsNorm(), C.retention_custom_inputs(),
                          torch.float16, mask_value="0")
    text = L.render_functors(lf)
    assert lf.customs[0].per_kv and lf.customs[0].torch_dtype == torch.float16
    assert "const ae_elem* mask_row;" in text and "p.custom[0]" in text
    assert "(int64_t)(ctx.h) * (1 * (int64_t)p.seqlen_kv * (int64_t)p.seqlen_q)" in text   # [1, heads, seq_len, seq_len_kv]
    assert "*(const ae_elem4*)src" in text and "ctx.kv_base + ae_kv_off(4 * g)" in text
    assert "(s[e] * cm_mask[e])" in text and "ae_row_abssum<N>" in text
    with pytest.raises(NotImplementedError):   # ... but not in the epilogue, which has no kv position
        class Epi(C.OnlineIdentity):
            @staticmethod
            def online_fwd_epilogue(o, rs, b, h, q_idx):
                return o, {}
        bad = Epi()
        cio = C.retention_custom_inputs()
        bad.online_fwd_epilogue = staticmethod(lambda o, rs, b, h, q_idx: (o * cio.input_tensors["mask"], {}))
        L.trace_functors(None, None, bad, cio, torch.float16)


def test_combine_lowering_finds_the_merged_lse():
    text = lower_combine(C.OnlineSoftmax(), ["lse"])
    assert "ae_arr_max<AE_NSPLIT>(rs[0])" in text and "ae_arr_sum<AE_NSPLIT>" in text
    assert "merged[0] = cb" in text and "nanf" not in text
    text = lower_combine(C.OnlineIdentity(), [])
    assert "w[e] = 1.0f" in text


# ---- engine construction compiles through hipRTC without a GPU ---------------------------------------
def _meta(B, Hq, Hkv, Sq, Skv, D, DV, dt):
    return (meta_tensor(B, Hq, Sq, D, dtype=dt), meta_tensor(B, Hkv, Skv, D, dtype=dt),
            meta_tensor(B, Hkv, Skv, DV, dtype=dt))


def test_engine_dispatch_and_compile_on_cpu():
    from core.lower.lower_decode import GQADecodeOp, MLADecodeOp
    from core.lower.prefill_op import PrefillOp
    sm = C.make_scale_score_mod(0.1)
    pre = AttentionEngine(_meta(1, 2, 2, 256, 256, 64, 64, torch.float16), CustomIO({}), sm, C.causal_mask,
                          C.OnlineSoftmax())
    assert isinstance(pre._op, PrefillOp) and "#define AE_MASK_MODE 1" in pre.tl_code
    assert pre.block_mask is None     # exactly block-causal -> dense template in the reference
    win = AttentionEngine(_meta(1, 2, 2, 512, 512, 64, 64, torch.bfloat16), CustomIO({}), sm,
                          C.make_sliding_window_mask(128), C.OnlineSoftmax())
    assert "#define AE_MASK_MODE 2" in win.tl_code and "#define AE_DTYPE_BF16 1" in win.tl_code
    assert win.block_mask.shape == (1, 2, 4, 4) and win.block_mask.dtype == torch.int8
    dec = AttentionEngine(_meta(2, 32, 8, 1, 1024, 128, 128, torch.float16), CustomIO({}), sm, None,
                          C.OnlineSoftmax())
    assert isinstance(dec._op, GQADecodeOp) and "ae_combine" in dec.tl_code
    mla = AttentionEngine(_meta(2, 128, 1, 1, 512, 576, 512, torch.bfloat16), CustomIO({}), sm, None,
                          C.OnlineSoftmax(), kv_shared=True)
    assert isinstance(mla._op, MLADecodeOp)
    gqa = AttentionEngine(_meta(1, 8, 2, 256, 256, 64, 64, torch.float16), CustomIO({}), sm, C.causal_mask,
                          C.OnlineSoftmax())
    assert isinstance(gqa._op, PrefillOp)
    # MHA decode (attn_script/mha_inference.py): a few query tokens against a long KV -> split-KV prefill
    mhad = AttentionEngine(_meta(1, 32, 32, 128, 8192, 128, 128, torch.float16), CustomIO({}), sm, None,
                           C.OnlineSoftmax())
    assert isinstance(mhad._op, PrefillOp) and mhad._op.split_kv
    assert mhad._op.plan_splits(1, 32, 128, 8192) == (8, 1024)
    assert mhad._op.plan_splits(2, 4, 5, 1000) == (16, 64)       # never an empty split, whole tiles
    assert "#define AE_NSPLIT 8" in mhad.tl_code and "ae_combine" in mhad.tl_code
    # tuner / backend arguments of the reference scripts are accepted
    AttentionEngine(_meta(1, 2, 2, 128, 128, 64, 64, torch.float16), CustomIO({}), sm, C.causal_mask,
                    C.OnlineSoftmax(), tune=True, tune_file="x.json", tune_bwd=True, backend="cute")
    # identity online function may be None (reference CuTe scripts)
    AttentionEngine(_meta(1, 2, 2, 128, 128, 64, 64, torch.float16), CustomIO({}), C.make_relu_score_mod(0.1),
                    None, None)


def test_engine_error_behaviour():
    sm = C.make_scale_score_mod(0.1)
    with pytest.raises(KeyError):       # unsupported dtype, as attn_engine.py:225-228 / 304
        AttentionEngine(_meta(1, 2, 2, 128, 128, 64, 64, torch.float32), CustomIO({}), sm, None, C.OnlineSoftmax())
    with pytest.raises(AssertionError):  # decode asserts q_len == 1 (attn_engine.py:255)
        AttentionEngine(_meta(1, 8, 2, 4, 1024, 64, 64, torch.float16), CustomIO({}), sm, None, C.OnlineSoftmax())
    # an online function without combine() cannot merge KV splits: the same shape runs unsplit
    unsplit = AttentionEngine(_meta(1, 2, 2, 128, 1024, 64, 64, torch.float16), CustomIO({}), sm, None,
                              C.OnlineIdentity())
    assert not unsplit._op.split_kv and unsplit._op.plan_splits(1, 2, 128, 1024) == (1, 1024)
    with pytest.raises(ValueError):
        AttentionEngine(_meta(1, 2, 2, 128, 128, 64, 64, torch.float16), CustomIO({}), sm, None,
                        C.OnlineSoftmax(), backend="triton")
    mod = AttentionEngine(_meta(1, 2, 2, 128, 128, 64, 64, torch.float16), CustomIO({}), sm, None, C.OnlineSoftmax())
    q = torch.zeros(1, 128, 2, 64, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="no CPU path"):   # the product never falls back to the CPU
        mod(q, q, q)


def test_lazy_maximum_only_for_the_online_softmax():
    """The thresholded running maximum is applied only when the traced graph is provably the online
    softmax; a function that exports m itself keeps the exact update."""
    from attn_engine import OnlineFunc

    class SoftmaxExportingMax(C.OnlineSoftmax):
        @staticmethod
        def online_fwd_epilogue(o, online_rowscales, b, h, q_idx):
            o_new = o / online_rowscales["r"]
            return o_new, {"m": online_rowscales["m"] + 0.0}
    lf = L.trace_functors(C.make_scale_score_mod(0.125), None, SoftmaxExportingMax(), CustomIO({}), torch.float16)
    assert "ae_max(st.m" in lf.online_fwd_body and "5.545" not in lf.online_fwd_body
    lf = L.trace_functors(C.make_scale_score_mod(0.125), None, C.OnlineAbsNorm(), CustomIO({}), torch.float16)
    assert "5.545" not in lf.online_fwd_body


def test_softmax_specialisation_needs_the_exact_graph():
    """Kernels that hard-code exp(c*S - m) (pipelined prefill, wave-specialised MLA decode, the softmax
    backward) may only be chosen for the online softmax OF the modified scores.  Near misses -- another
    function of the scores inside exp, another quantity inside the running maximum, other initial
    values -- stay reference-point invariant (lazy maximum allowed) but must run the generated functor."""
    from attn_engine import OnlineFunc
    sm = C.make_scale_score_mod(0.125)
    assert L.trace_functors(sm, None, C.OnlineSoftmax(), CustomIO({}), torch.float16).softmax == (0.125, "m", "r")

    class TwiceInsideExp(C.OnlineSoftmax):
        @staticmethod
        def online_fwd(scores, online_rowscales, b, h, q_idx):
            m, r = online_rowscales["m"], online_rowscales["r"]
            m_new = m.max(scores.get_reduce("max"))
            scale_tmp = (m - m_new).exp()
            p = (scores * 2.0 - m_new).exp()
            return p, {"m": m_new, "r": r * scale_tmp + p.get_reduce("sum")}, scale_tmp

    class AbsInsideMax(C.OnlineSoftmax):
        @staticmethod
        def online_fwd(scores, online_rowscales, b, h, q_idx):
            m, r = online_rowscales["m"], online_rowscales["r"]
            m_new = m.max(scores.abs().get_reduce("max"))
            scale_tmp = (m - m_new).exp()
            p = (scores - m_new).exp()
            return p, {"m": m_new, "r": r * scale_tmp + p.get_reduce("sum")}, scale_tmp

    class StartsAtZero(C.OnlineSoftmax):
        def __init__(self):
            OnlineFunc.__init__(self, {"m": SymbolScalar("m", Var("0.0")), "r": SymbolScalar("r", Var("0.0"))},
                                {"lse": SymbolScalar("lse", Var("0.0"))}, CustomIO())

    for near_miss in (TwiceInsideExp(), AbsInsideMax(), StartsAtZero()):
        lf = L.trace_functors(sm, None, near_miss, CustomIO({}), torch.float16)
        assert lf.softmax is None, type(near_miss).__name__
        # ... and the generic kernel is what the engine then compiles, even on chip-filling shapes
        tiles = L.choose_prefill_tiles(128, 128, seqlen_q=4096, softmax=lf.softmax, batch_heads=64)
        assert tiles.template == "ae_prefill.hip"
    src = L.render_functors(L.trace_functors(sm, None, TwiceInsideExp(), CustomIO({}), torch.float16))
    assert "0.3606737" in src                    # the functor carries the user's factor: 0.125 * 2 * log2(e)
    # no backward is derived for them either: the softmax gradient is only valid for the exact graph
    from core.lower.prefill_bwd_op import PrefillBwdOp
    from core.lower.prefill_op import PrefillOp
    for near_miss in (TwiceInsideExp(), AbsInsideMax()):
        op = PrefillOp(_meta(1, 2, 2, 256, 256, 64, 64, torch.float16), CustomIO({}), sm, None, near_miss, "-inf")
        with pytest.raises(NotImplementedError):
            PrefillBwdOp(op, sm, near_miss, CustomIO({}))


def test_softmax_proof_takes_the_guarded_division_of_the_sparse_attention_script():
    """attn_script/sparseattn.py:66-72 divides by r + 1e-30.  A row with a visible key has r >= 1 whatever the lagging
    reference, so a constant of at most 1e-20 leaves r unchanged in fp32 and the graph is still the online softmax;
    a constant that can change r (or anything else in the denominator) is not."""
    sm = C.make_scale_score_mod(0.125)

    def guarded(c, wrong_side=False):
        class Guarded(C.OnlineSoftmax):
            @staticmethod
            def online_fwd_epilogue(o, online_rowscales, b, h, q_idx):
                r = online_rowscales["r"]
                den = (c + r) if wrong_side else (r + c)
                return o / den, {"lse": r.log() + online_rowscales["m"]}
        return Guarded()
    for c in (1e-30, 1e-20, 0.0):
        assert L.trace_functors(sm, None, guarded(c), CustomIO({}), torch.float16).softmax == (0.125, "m", "r"), c
    assert L.trace_functors(sm, None, guarded(1e-30, wrong_side=True), CustomIO({}), torch.float16).softmax is not None
    for c in (1e-6, 1.0, -1e-30):
        lf = L.trace_functors(sm, None, guarded(c), CustomIO({}), torch.float16)
        assert lf.softmax is None and "5.545" not in lf.online_fwd_body, c      # neither specialised nor lazy
    src = L.render_functors(L.trace_functors(sm, None, guarded(1e-30), CustomIO({}), torch.float16))
    assert "1e-30" in src or "1.0e-30" in src or "9.99999" in src        # the user's epilogue runs as written


def test_shapes_broadcast_by_name():
    q = SymbolScalar("q_idx", Var("q_idx"), shape_idx=["block_M"])
    kv = SymbolScalar("kv_idx", Var("kv_idx"), shape_idx=["block_N"])
    assert (q - kv).shape_idx == ["block_M", "block_N"]
    assert (kv - q).shape_idx == ["block_M", "block_N"]
    s = SymbolicArray("s", Var("s"), shape_idx=["block_M", "block_N"])
    assert (s - q).shape_idx == ["block_M", "block_N"] and (q * 2).shape_idx == ["block_M"]
    assert s.get_reduce("max").shape_idx == ["block_M"]


def test_symbolic_derivative_matches_autograd():
    """core.transform.autodiff.derivative on traced elementwise graphs (every node type the tracer has),
    evaluated by the oracle's graph interpreter, against torch.autograd of the same function."""
    from core.transform.autodiff import derivative
    from oracle.online_interp import evaluate
    x = torch.linspace(-2.3, 2.7, 41, dtype=torch.float64)
    cases = [
        (lambda s: ((s * 0.125 + 0.3) * 0.5).tanh() * 0.5 + 0.5, lambda t: torch.sigmoid(t * 0.125 + 0.3)),
        (lambda s: (s * 0.7).max(0), lambda t: torch.relu(t * 0.7)),
        (lambda s: (s * s + 1.5).log() / (s.exp() + 2.0), lambda t: torch.log(t * t + 1.5) / (torch.exp(t) + 2.0)),
        (lambda s: (s * 0.4).exp2() - (s * s + 1.0).log2() - s.abs() * 0.25 + (-s) * 0.1,
         lambda t: torch.exp2(t * 0.4) - torch.log2(t * t + 1.0) - t.abs() * 0.25 - t * 0.1),
        (lambda s: 3.0 / (s * s + 1.0) + (2.0 - s) * s, lambda t: 3.0 / (t * t + 1.0) + (2.0 - t) * t),
    ]
    for traced_fn, torch_fn in cases:
        s = SymbolScalar("scores", Var("scores"), shape_idx=[])
        y = traced_fn(s)
        dy = derivative(y, s)
        got = evaluate(dy, {id(s): x})
        t = x.clone().requires_grad_(True)
        (want,) = torch.autograd.grad(torch_fn(t).sum(), t)
        got = got if isinstance(got, torch.Tensor) else torch.full_like(x, float(got))
        assert torch.allclose(got.expand_as(want), want, atol=1e-12, rtol=1e-10)
    # no dependence -> zero
    s, c = SymbolScalar("scores", Var("scores"), shape_idx=[]), SymbolScalar("c", Var("c"), shape_idx=[])
    assert float(evaluate(derivative(c * 2.0, s), {id(c): 1.0})) == 0.0


def test_elementwise_backward_lowering():
    """The backward functors of sigmoid / relu attention are emitted; online functions that keep row
    scales, non-scalar custom inputs and non-identity forward/backward rules are refused."""
    from core.lower.prefill_bwd_op import lower_elementwise_backward
    src = lower_elementwise_backward(C.make_sigmoid_score_mod(0.125), C.OnlineIdentity(),
                                     CustomIO({"softmax_bias": (1,)}), torch.float16)
    assert "ae_bwd_pd" in src and "cust.softmax_bias" in src and "p.custom[0]" in src
    src = lower_elementwise_backward(C.make_relu_score_mod(0.125), C.OnlineIdentity(), CustomIO({}), torch.float16)
    assert "> 0.0f ?" in src
    with pytest.raises(NotImplementedError):
        lower_elementwise_backward(C.make_scale_score_mod(0.125), C.OnlineAbsNorm(), CustomIO({}), torch.float16)
    with pytest.raises(NotImplementedError):
        lower_elementwise_backward(C.retention_score_mod, C.OnlineIdentity(), C.retention_custom_inputs(),
                                   torch.float16)


def test_inferred_block_mask_granularity_does_not_reach_the_kernel():
    """infer_mask_block_M/N only shape the block mask kept on mod.block_mask (lower.py:721-738 of the
    reference); the kernel classifies its own tiles from mask_mod, so a granularity that no kv tile fits
    (96 keys against 64-key tiles) is harmless, and handing the engine such a mask from outside is refused
    instead of skipping visible keys."""
    from core.lower.prefill_op import PrefillOp
    op = PrefillOp(_meta(1, 2, 2, 384, 384, 64, 64, torch.float16), CustomIO({}), C.make_scale_score_mod(0.125),
                   C.make_sliding_window_mask(100), C.OnlineSoftmax(), "-inf", infer_mask=True,
                   infer_mask_block_M=128, infer_mask_block_N=96)
    assert op.block_mask is not None and op.block_mask.shape == (1, 2, 3, 4)
    plan = op._plan(1, 2, 384, 384, device=None)
    assert (plan.block_m, plan.block_n) == (op.tiles.block_m, op.tiles.block_n)


def test_traced_backward_of_an_online_function_with_its_own_row_scale():
    """attn_script/retention.py: OnlineFunc.forward / backward are traced into ae_bwd_pd2 together with the
    derivative of score_mod (the decay mask, read per score); an online function that keeps row scales
    without defining them gets no backward."""
    from core.lower.prefill_bwd_op import lower_traced_backward
    src, names = lower_traced_backward(C.retention_score_mod, C.OnlineRetention(), C.retention_custom_inputs(),
                                       torch.float16)
    assert names == ["r"] and "ae_bwd_pd2" in src
    assert "p.custom[0]" in src and "p.seqlen_kv" in src          # the mask element of (head, q, kv)
    body = src.split("ae_bwd_pd2", 2)[-1]
    assert "const float (&rs)[1]" in body and "rs[0]" in body and "cv_mask" in body and "dp" in body
    with pytest.raises(NotImplementedError, match="forward"):
        lower_traced_backward(C.retention_score_mod, C.OnlineAbsNorm(), C.retention_custom_inputs(), torch.float16)


def test_traced_backward_reads_every_final_row_scale():
    """An online function with two final row scales whose forward() / backward() read both (the reference hands
    every final row scale to them, core/lower/lower.py:413-453): both arrive in the functor, in declaration order."""
    from core.lower.prefill_bwd_op import lower_traced_backward

    class TwoScales(C.OnlineSoftmax):
        def __init__(self):
            super().__init__()
            self.final_rowscales = {"m": SymbolScalar("m", Var("0.0")), "r": SymbolScalar("r", Var("0.0"))}

        @staticmethod
        def online_fwd_epilogue(o, online_rowscales, b, h, q_idx):
            return o / online_rowscales["r"], {"m": online_rowscales["m"], "r": online_rowscales["r"]}

        @staticmethod
        def forward(scores, final_rowscales, b, h, q_idx, kv_idx):
            return (scores - final_rowscales["m"]).exp() / final_rowscales["r"]

        @staticmethod
        def backward(dp, scores, final_rowscales, doosum_rowscales, b, h, q_idx, kv_idx):
            return scores * (dp - doosum_rowscales)
    src, names = lower_traced_backward(C.make_scale_score_mod(0.125), TwoScales(), CustomIO({}), torch.float16)
    assert names == ["m", "r"]
    body = src.split("ae_bwd_pd2", 2)[-1]
    assert "const float (&rs)[2]" in body and "rs[0]" in body and "rs[1]" in body and "doosum" in body
    lf = L.trace_functors(C.make_scale_score_mod(0.125), None, TwoScales(), CustomIO({}), torch.float16)
    assert lf.softmax is None and lf.final_rowscale_names == ["m", "r"]     # not the graph with the fixed backward


def test_symbol_backward_leaves_gradient_expressions_on_the_leaves():
    """SymbolScalar.backward (core/transform/core.py:119-199 of the reference): after
    ``f(x, y).backward(g)`` the leaves carry g * df/dx and g * df/dy as traced expressions; evaluated by the
    oracle's graph interpreter against torch.autograd."""
    from oracle.online_interp import evaluate
    x = SymbolScalar("x", Var("x"), shape_idx=[])
    y = SymbolScalar("y", Var("y"), shape_idx=[])
    g = SymbolScalar("g", Var("g"), shape_idx=[])
    f = (x * y + x.exp()) / (y * y + 2.0) - (x * 0.5).tanh()
    f.backward(g)
    assert x.grad is not None and y.grad is not None
    xv = torch.linspace(-1.5, 1.2, 17, dtype=torch.float64).requires_grad_(True)
    yv = torch.linspace(0.3, 2.1, 17, dtype=torch.float64).requires_grad_(True)
    gv = torch.linspace(-0.7, 0.9, 17, dtype=torch.float64)
    ref = (xv * yv + xv.exp()) / (yv * yv + 2.0) - (xv * 0.5).tanh()
    gx, gy = torch.autograd.grad(ref, (xv, yv), gv)
    env = {id(x): xv.detach(), id(y): yv.detach(), id(g): gv}
    assert torch.allclose(evaluate(x.grad, env), gx, atol=1e-12)
    assert torch.allclose(evaluate(y.grad, env), gy, atol=1e-12)


def test_elementwise_graphs_are_recognised():
    """out = sum_kv f(s) v (no row state, no reduction over the tile, no kv index): the functor may be applied
    to any subset of a tile, which is what lets the software-pipelined kernel call it pairwise."""
    import attn_script as C
    from core.lower import lower as L
    f16 = torch.float16
    sig = L.trace_functors(C.make_sigmoid_score_mod(0.125), None, C.OnlineIdentity(),
                           CustomIO({"softmax_bias": (1,)}), f16)
    relu = L.trace_functors(C.make_relu_score_mod(0.125), C.causal_mask, C.OnlineIdentity(), CustomIO({}), f16)
    soft = L.trace_functors(C.make_scale_score_mod(0.125), None, C.OnlineSoftmax(), CustomIO({}), f16)
    assert sig.elementwise and relu.elementwise and not soft.elementwise
    assert sig.softmax is None and soft.softmax is not None

    def uses_kv(score, custom_fwd_inputs, b, h, q_idx, kv_idx):
        return score * 0.125 + kv_idx
    assert not L.trace_functors(uses_kv, None, C.OnlineIdentity(), CustomIO({}), f16).elementwise

    class TileNormalised(C.OnlineIdentity):      # no row state, but a reduction over the tile
        @staticmethod
        def online_fwd(scores, online_rowscales, b, h, q_idx):
            return scores / scores.get_reduce("abssum"), online_rowscales, C.OnlineIdentity.online_fwd(
                scores, online_rowscales, b, h, q_idx)[2]
    try:
        lf = L.trace_functors(C.make_scale_score_mod(0.125), None, TileNormalised(), CustomIO({}), f16)
    except Exception:
        lf = None
    assert lf is None or not lf.elementwise
    # tile choice: a chip-filling elementwise problem takes the pipelined kernel, a small one the generic one
    big = L.choose_prefill_tiles(128, 128, seqlen_q=4096, softmax=None, batch_heads=64, elementwise=True)
    small = L.choose_prefill_tiles(128, 128, seqlen_q=512, softmax=None, batch_heads=4, elementwise=True)
    assert big.template == "ae_prefill_pipe.hip" and small.template == "ae_prefill.hip"
    cfg = L.render_config(128, 128, f16, big, 0, False, 0, True, True, True, None, elementwise=True)
    assert "#define AE_PIPE_KIND 1" in cfg


def test_per_tile_renormalisation_is_deferred_to_the_epilogue(monkeypatch):
    """scores / r_new with o_scale = r_old / r_new (retention's running sum of |s|): the factors telescope, so
    the lowering accumulates unscaled and divides once by the final row scale - no rescale of the accumulator
    per tile.  The row state and the final row scale are untouched; graphs of another form are left alone."""
    import attn_script as C
    from core.lower import lower as L
    f16 = torch.float16
    lf = L.trace_functors(C.retention_score_mod, C.causal_mask, C.OnlineRetention(), C.retention_custom_inputs(),
                          f16, "0")
    assert lf.deferred_norm == "r" and lf.o_scale_one
    src = L.render_functors(lf)
    fwd = src[src.index("AE_DEV float ae_online_fwd"):src.index("AE_DEV void ae_epilogue")]
    assert " / " not in fwd.split("#endif")[-1] and "const float ae_o_scale = 1.0f;" in fwd
    epi = src[src.index("AE_DEV void ae_epilogue"):]
    assert "1.0f / st.r" in epi and "frs[0] = st.r;" in epi
    assert L.trace_functors(C.make_scale_score_mod(0.125), None, C.OnlineSoftmax(), CustomIO({}), f16).deferred_norm is None
    assert L.trace_functors(C.make_relu_score_mod(0.125), None, C.OnlineIdentity(), CustomIO({}), f16).deferred_norm is None

    class ScaledDifferently(C.OnlineAbsNorm):        # o_scale does not match the normalisation of the scores
        @staticmethod
        def online_fwd(scores, online_rowscales, b, h, q_idx):
            s, rs, o_scale = C.OnlineAbsNorm.online_fwd(scores, online_rowscales, b, h, q_idx)
            return s, rs, o_scale * 0.5
    assert L.trace_functors(C.make_scale_score_mod(0.125), None, ScaledDifferently(), CustomIO({}), f16).deferred_norm is None
    monkeypatch.setenv("AE_DEFER_NORM", "0")
    lf0 = L.trace_functors(C.retention_score_mod, C.causal_mask, C.OnlineRetention(), C.retention_custom_inputs(),
                           f16, "0")
    assert lf0.deferred_norm is None and not lf0.o_scale_one


def test_tuner_cache_records(tmp_path):
    """tune=True / tune_file: the json records of the reference's tuner (attn_tl.py:465-500: a list of the five
    problem keys plus ``tuned_config``), looked up at construction; nothing is measured or written without a GPU
    call."""
    import json
    from core.lower import tuner
    f = str(tmp_path / "tuned.json")
    pk = tuner.problem_keys((2, "heads", 1024, 128), 128, 128)
    assert pk == {"batch": 2, "heads": 32, "seq_len": 1024, "dim": 128, "dimv": 128}   # dynamic dims: attn_tl.py:465-472
    assert tuner.lookup(f, pk) is None
    cands = tuner.prefill_candidates(128, 128, softmax=(0.1, "m", "r"), elementwise=False)
    assert len(cands) == 4 and cands[0].template == "ae_prefill_pipe.hip"
    assert len(tuner.prefill_candidates(128, 128, None, False)) == 3
    assert [c.block_n for c in tuner.prefill_candidates(256, 512, None, False)] == [32]
    assert [(c.waves_per_eu, c.block_n) for c in tuner.prefill_candidates(192, 128, None, False)] == \
        [(2, 64), (2, 32), (1, 64), (1, 32)]
    assert [(c.template, c.block_n) for c in tuner.prefill_candidates(192, 192, None, False)] == \
        [("ae_prefill_simple.hip", 32), ("ae_prefill_simple.hip", 64)]
    tuner.store(f, pk, tuner.encode_tiles(cands[2]))
    tuner.store(f, {**pk, "batch": 4}, [128, 128, 2, 256, False])     # a record as the reference writes it
    recs = json.load(open(f))
    assert [sorted(r) for r in recs] == [sorted(list(pk) + ["tuned_config"])] * 2
    assert recs[0]["tuned_config"] == [128, 32, 2, 256, 2, "ae_prefill.hip"]
    assert tuner.decode_tiles(tuner.lookup(f, pk), cands) == cands[2]
    assert tuner.decode_tiles(tuner.lookup(f, {**pk, "batch": 4}), cands) is None   # not one of this build's tiles

    sm = C.make_scale_score_mod(0.1)
    hit = AttentionEngine(_meta(2, 32, 32, 1024, 1024, 128, 128, torch.float16), CustomIO({}), sm, C.causal_mask,
                          C.OnlineSoftmax(), tune=True, tune_file=f)
    assert hit._op.tiles == cands[2] and not hit._op._tune_pending
    assert "#define AE_BN 32" in hit.tl_code
    miss = AttentionEngine(_meta(4, 32, 32, 1024, 1024, 128, 128, torch.float16), CustomIO({}), sm, C.causal_mask,
                           C.OnlineSoftmax(), tune=True, tune_file=f)
    assert miss._op._tune_pending and miss._op.tiles == cands[0]      # measured at the first call on a GPU
    plain = AttentionEngine(_meta(2, 32, 32, 1024, 1024, 128, 128, torch.float16), CustomIO({}), sm, C.causal_mask,
                            C.OnlineSoftmax(), tune_file=f)
    assert plain._op.tiles == cands[0] and not plain._op._tune_pending
    tuner.store(f, pk, tuner.encode_tiles(cands[1]))                  # replaces the record of that problem
    assert len(json.load(open(f))) == 2 and tuner.decode_tiles(tuner.lookup(f, pk), cands) == cands[1]
    assert json.load(open(f)) == recs[1:] + [{**pk, "tuned_config": tuner.encode_tiles(cands[1])}]


def test_tuner_store_survives_a_damaged_file(tmp_path):
    """A tune_file that was cut short in the middle of a write (or written by two processes at once) still gives
    up its complete records, and the next store keeps them; the store itself replaces the file in one step and
    leaves no temporary file behind."""
    import json
    import os
    from core.lower import tuner
    f = str(tmp_path / "tuned.json")
    pk = {"batch": 2, "heads": 32, "seq_len": 1024, "dim": 128, "dimv": 128}
    for b in (1, 2, 3):
        tuner.store(f, {**pk, "batch": b}, [128, 64, 2, 256, 2, "ae_prefill.hip"])
    text = open(f).read()
    third = text.rindex("{")
    open(f, "w").write(text[:third + 40])             # the third record is torn, the closing bracket is gone
    with pytest.raises(ValueError):
        json.load(open(f))
    assert tuner.lookup(f, {**pk, "batch": 1}) == [128, 64, 2, 256, 2, "ae_prefill.hip"]
    assert tuner.lookup(f, {**pk, "batch": 3}) is None
    tuner.store(f, {**pk, "batch": 4}, [256, 64, 2, 256, 1, "ae_prefill_pipe.hip"])
    recs = json.load(open(f))                          # whole again
    assert [r["batch"] for r in recs] == [1, 2, 4]
    assert os.listdir(tmp_path) == ["tuned.json"]
    open(f, "w").write("not json at all")
    assert tuner.lookup(f, pk) is None
    tuner.store(f, pk, [1])
    assert json.load(open(f)) == [{**pk, "tuned_config": [1]}]


def test_decode_kernel_cache_is_keyed_by_the_merge_form(monkeypatch):
    """GQADecodeOp keeps one compiled kernel pair per (splits, even kv, merge form).  Whether the split kernel
    merges its waves' partial results itself (AE_MERGE_IN_WG) depends on ``static_workspace`` and on an
    environment variable, both of which may change between two calls of one engine; a kernel compiled for one
    form must never be handed to the launch of the other (the merging kernel leaves the work buffers unwritten,
    the other one stores through them).  hipRTC runs on the CPU, so the variants are really compiled here."""
    from core.lower.lower_decode import GQADecodeOp
    dt = torch.float16
    B, Hq, Hkv, Skv, D = 128, 32, 8, 777, 128          # plans 4 splits: the waves of one workgroup
    meta = (meta_tensor(B, Hq, 1, D, dtype=dt), meta_tensor(B, Hkv, Skv, D, dtype=dt), meta_tensor(B, Hkv, Skv, D, dtype=dt))
    op = GQADecodeOp(meta, CustomIO({}), C.make_scale_score_mod(D ** -0.5), None, C.OnlineSoftmax(), "-inf")
    n_split, _ = op.plan_splits(B, Hq, Hkv, Skv)
    assert n_split == op.N_WAVES
    monkeypatch.delenv("AE_DECODE_MERGE_IN_WG", raising=False)
    # the constructor compiled the merging form
    assert set(op._variants) == {(4, False, 1)}
    merged = op._variant(n_split, False, op._merge_mode(n_split))
    assert "#define AE_MERGE_IN_WG 1" in merged[3] and merged[1].merge_in_wg == 1
    # the documented toggle: the launch without allocations keeps the merge kernel
    op.static_workspace = True
    assert not op.merges_in_workgroup(n_split)
    plain = op._variant(n_split, False, op._merge_mode(n_split))
    assert plain is not merged and plain[0] is not merged[0]
    assert "#define AE_MERGE_IN_WG 0" in plain[3] and plain[1].merge_in_wg == 0
    op.static_workspace = False
    assert op._variant(n_split, False, op._merge_mode(n_split)) is merged
    # ... and the environment variable that keeps the two launches
    monkeypatch.setenv("AE_DECODE_MERGE_IN_WG", "0")
    assert op._variant(n_split, False, op._merge_mode(n_split)) is plain
    assert set(op._variants) == {(4, False, 1), (4, False, 0)}


def test_decode_splits_over_several_workgroups_merge_in_the_last_one(monkeypatch):
    """A small batch spreads one kv axis over several workgroups; the one that finishes last merges
    (AE_MERGE_LAST, merge_in_wg = 2) unless the launch must not keep buffers of its own (``static_workspace``)
    or the environment asks for the two launches.  Compiled here by hipRTC, without register spills."""
    from core.lower.lower_decode import GQADecodeOp
    dt = torch.float16
    B, Hq, Hkv, Skv, D = 1, 32, 8, 8192, 128
    meta = (meta_tensor(B, Hq, 1, D, dtype=dt), meta_tensor(B, Hkv, Skv, D, dtype=dt), meta_tensor(B, Hkv, Skv, D, dtype=dt))
    monkeypatch.delenv("AE_DECODE_MERGE_LAST", raising=False)
    op = GQADecodeOp(meta, CustomIO({}), C.make_scale_score_mod(D ** -0.5), None, C.OnlineSoftmax(), "-inf")
    n_split, _ = op.plan_splits(B, Hq, Hkv, Skv)
    assert n_split > op.N_WAVES and op._merge_mode(n_split) == 2
    assert set(op._variants) == {(n_split, True, 2)}
    last = op._variant(n_split, True, 2)
    assert "#define AE_MERGE_LAST 1" in last[3] and "#define AE_MERGE_IN_WG 0" in last[3] and last[1].merge_in_wg == 2
    op.static_workspace = True
    assert op._merge_mode(n_split) == 0
    op.static_workspace = False
    monkeypatch.setenv("AE_DECODE_MERGE_LAST", "0")
    assert op._merge_mode(n_split) == 0
    plain = op._variant(n_split, True, 0)
    assert "#define AE_MERGE_LAST 0" in plain[3] and plain[0] is not last[0]


def test_decode_build_that_spills_is_built_again_for_one_wave_a_simd():
    """Value heads of 256 do not fit the 256 registers of two waves a SIMD (85 spilled registers, 2.3x the time on
    the chip); the operator then builds the kernel for one wave a SIMD, which does not spill.  Head dims of 128
    keep two waves."""
    import warnings
    from core.lower.lower_decode import GQADecodeOp
    dt = torch.float16
    for D, want in ((256, 1), (128, 2)):
        B, Hq, Hkv, Skv = 64, 32, 8, 8192
        meta = (meta_tensor(B, Hq, 1, D, dtype=dt), meta_tensor(B, Hkv, Skv, D, dtype=dt), meta_tensor(B, Hkv, Skv, D, dtype=dt))
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            op = GQADecodeOp(meta, CustomIO({}), C.make_scale_score_mod(D ** -0.5), None, C.OnlineSoftmax(), "-inf")
        (module, _, _, src), = op._variants.values()
        assert f"#define AE_WAVES_PER_EU {want}" in src
        assert module.kernel_info()["ae_decode_split_kernel"].get(".vgpr_spill_count", 0) == 0


def test_numerics_keywords_of_the_constructor(monkeypatch):
    """``exact_scale`` / ``defer_norm`` reach the generated configuration; left at None they follow the defaults
    (and the environment switches the tests use)."""
    monkeypatch.delenv("AE_PREFILL_PRESCALE", raising=False)
    monkeypatch.delenv("AE_DEFER_NORM", raising=False)
    monkeypatch.setenv("AE_PREFILL_KERNEL", "pipelined")
    f16 = torch.float16
    sm = C.make_scale_score_mod(0.1)
    meta = _meta(2, 32, 32, 1024, 1024, 128, 128, f16)
    default = AttentionEngine(meta, CustomIO({}), sm, C.causal_mask, C.OnlineSoftmax())
    exact = AttentionEngine(meta, CustomIO({}), sm, C.causal_mask, C.OnlineSoftmax(), exact_scale=True)
    folded = AttentionEngine(meta, CustomIO({}), sm, C.causal_mask, C.OnlineSoftmax(), exact_scale=False)
    assert default._op.tiles.template == "ae_prefill_pipe.hip"
    assert "AE_PRESCALE" not in default.tl_code
    assert "#define AE_PRESCALE 0" in exact.tl_code and "#define AE_PRESCALE 1" in folded.tl_code
    monkeypatch.setenv("AE_PREFILL_PRESCALE", "0")          # the keyword wins over the environment
    assert "#define AE_PRESCALE 1" in AttentionEngine(meta, CustomIO({}), sm, None, C.OnlineSoftmax(),
                                                      exact_scale=False).tl_code
    monkeypatch.delenv("AE_PREFILL_KERNEL")
    rmeta = _meta(1, 2, 2, 256, 256, 64, 64, f16)
    args = (rmeta, C.retention_custom_inputs(), C.retention_score_mod, C.causal_mask, C.OnlineRetention())
    assert AttentionEngine(*args, mask_value="0").attention.functors.deferred_norm == "r"
    assert AttentionEngine(*args, mask_value="0", defer_norm=False).attention.functors.deferred_norm is None
    monkeypatch.setenv("AE_DEFER_NORM", "0")
    assert AttentionEngine(*args, mask_value="0").attention.functors.deferred_norm is None
    assert AttentionEngine(*args, mask_value="0", defer_norm=True).attention.functors.deferred_norm == "r"


def test_tile_classes_of_a_user_block_mask():
    """PrefillBwdOp.block_mask_tile_classes (the tables the backward launches read when the forward ran on a block
    mask the user supplied) against brute force over the expanded mask, for block sizes below, equal to and above
    the tile sizes and sequence lengths that are not multiples of either."""
    from core.lower.prefill_bwd_op import PrefillBwdOp
    g = torch.Generator().manual_seed(2)
    for bm, bn, Sq, Skv in ((128, 128, 1024, 1024), (32, 64, 640, 576), (64, 128, 448, 450), (256, 32, 700, 333),
                            (48, 96, 500, 400)):
        nq, nk = -(-Sq // bm), -(-Skv // bn)
        blocks = (torch.rand(2, 3, nq, nk, generator=g) < 0.5).to(torch.int8)
        dense = blocks.bool().repeat_interleave(bm, 2).repeat_interleave(bn, 3)[:, :, :Sq, :Skv]
        for tm, tn in ((128, 64), (256, 64), (64, 128)):
            got = PrefillBwdOp.block_mask_tile_classes(blocks, bm, bn, Sq, Skv, tm, tn)
            assert got.shape == (2, 3, -(-Sq // tm), -(-Skv // tn)) and got.dtype == torch.int8
            for i in range(got.shape[2]):
                for j in range(got.shape[3]):
                    t = dense[:, :, i * tm:(i + 1) * tm, j * tn:(j + 1) * tn]
                    some, every = t.any(-1).any(-1), t.all(-1).all(-1)
                    want = some.to(torch.int8) + (some & every).to(torch.int8)
                    assert torch.equal(got[:, :, i, j], want), (bm, bn, Sq, Skv, tm, tn, i, j)


def test_options_of_one_template_stay_with_it(monkeypatch):
    """Compiler options that a single template adds (hip_rt.TEMPLATE_OPTS) do not change what is compiled after it in the
    same process, and are part of the key of its code objects."""
    import ctypes
    from core.runtime import hip_rt as rt
    headers = {}
    compiled = rt._compile_module
    monkeypatch.setattr(rt, "_compile_module", lambda t, h, *a: headers.setdefault(t, h) and compiled(t, h, *a))
    for kernel in ("generic", "pipelined"):
        monkeypatch.setenv("AE_PREFILL_KERNEL", kernel)
        AttentionEngine((meta_tensor(1, 2, 256, 128, dtype=torch.float16),) * 3, CustomIO({}),
                        C.make_scale_score_mod(0.1), C.causal_mask, C.OnlineSoftmax())

    def code(template):
        monkeypatch.setattr(rt, "_modules", {})
        m = compiled(template, headers[template], None, False)
        data, n = ctypes.c_void_p(), ctypes.c_size_t()
        assert rt.lib().ae_module_code(m.handle, ctypes.byref(data), ctypes.byref(n)) == 0
        return m.key, ctypes.string_at(data, n.value)
    assert set(headers) == {"ae_prefill.hip", "ae_prefill_pipe.hip"} and "ae_prefill_pipe.hip" in rt.TEMPLATE_OPTS
    first = code("ae_prefill.hip")
    with_opts = code("ae_prefill_pipe.hip")
    assert code("ae_prefill.hip") == first
    monkeypatch.setattr(rt, "TEMPLATE_OPTS", {})
    assert code("ae_prefill_pipe.hip")[0] != with_opts[0] and code("ae_prefill.hip") == first


@pytest.mark.parametrize("kind", ["gqa", "mla"])
def test_every_split_count_that_is_tuned_is_launched(monkeypatch, tmp_path, kind):
    """tune=True measures through the operator's own calls, which the native host path serves from the plan that the last
    Python call of the shape left: no candidate may be served by another one's plan."""
    from core.lower import tuner
    if kind == "gqa":
        meta, more, key = (meta_tensor(1, 8, 1, 128, dtype=torch.float16),) + (meta_tensor(1, 2, 2048, 128, dtype=torch.float16),) * 2, {}, (1, 8, 2, 2048)
    else:
        meta = (meta_tensor(1, 16, 1, 576, dtype=torch.float16), meta_tensor(1, 1, 2048, 576, dtype=torch.float16),
                meta_tensor(1, 1, 2048, 512, dtype=torch.float16))
        more, key = {"kv_shared": True}, (1, 16, 1, 2048)
    op = AttentionEngine(meta, CustomIO({}), C.make_scale_score_mod(0.1), None, C.OnlineSoftmax(), tune=True,
                         tune_file=str(tmp_path / "tuned.json"), **more).attention

    class Host:
        plan = None

        def clear(self):
            self.plan = None
    op._host = Host()
    launched = []

    def run():
        if op._host.plan is None:                    # the Python path: plans, launches and leaves its plan behind
            op._host.plan = op.plan_splits(*key)[0]
        launched.append(op._host.plan)
    ms = iter((3.0, 1.0, 2.0))
    monkeypatch.setattr(tuner, "time_call", lambda f: (f(), next(ms))[1])
    op._tune_splits(key, [2, 4, 8], run)
    assert len(set(launched)) == 3 and op._tuned[key] == 4
    run()
    assert launched[-1] == launched[1]               # ... and the calls that follow run the one that was fastest


def test_mla_plan():
    """Splits cover the cache with none empty, whatever the shape; small batches take few heads a workgroup, the full one
    64; a paged split holds no more pages than the kernel keeps table entries for; target_workgroups = 1 means no splits."""
    from core.lower.lower_decode import MLADecodeOp
    dt = torch.bfloat16
    meta = (meta_tensor(1, 16, 1, 576, dtype=dt), meta_tensor(1, 1, 64, 576, dtype=dt), meta_tensor(1, 1, 64, 512, dtype=dt))
    op = MLADecodeOp(meta, CustomIO({}), C.make_scale_score_mod(192 ** -0.5), None, C.OnlineSoftmax(), "-inf")
    for B in (1, 3, 17, 128):
        for Hq, Hkv in ((1, 1), (16, 1), (40, 2), (128, 1)):
            for Skv in (1, 31, 33, 1000, 8192):
                heads, n_split, per = op.plan(B, Hq, Hkv, Skv)
                assert heads in (16, 32, 64) and per % op.BLOCK_N == 0
                assert n_split * per >= Skv > (n_split - 1) * per and 1 <= n_split <= op.MAX_SPLITS
                assert heads == 16 or Hq // Hkv > heads // 2
    assert op.plan(128, 128, 1, 4096) == (64, 1, 4096)
    assert op.plan(4, 128, 1, 2048)[0] == 16 and op.plan(4, 128, 1, 2048)[1] > 1
    _, n_split, per = op.plan(1, 16, 1, 300000, 64)
    assert per // 64 + 2 <= op.PAGE_TABLE_ENTRIES and n_split * per >= 300000
    op.target_workgroups = 1
    assert op.plan(2, 128, 1, 1000) == (64, 1, 1024)


def test_gqa_plan():
    """Any number of workgroups of a kv axis is one that a kernel is built for, with a tile for every wave, and fits the
    built-in work buffer; keys are covered; a combine() that wants every partial result keeps a power of two."""
    from core.lower.lower_decode import GQADecodeOp
    from core.runtime import hip_rt as rt
    dt = torch.float16
    meta = (meta_tensor(1, 8, 1, 128, dtype=dt), meta_tensor(1, 2, 64, 128, dtype=dt), meta_tensor(1, 2, 64, 128, dtype=dt))
    op = GQADecodeOp(meta, CustomIO({}), C.make_scale_score_mod(0.1), None, C.OnlineSoftmax(), "-inf")
    assert op.grouped_merge
    for B in (1, 3, 17, 128):
        for Hq, Hkv in ((8, 2), (32, 4), (40, 2), (64, 8)):
            for Skv in (1, 33, 300, 2204, 13634, 32768):
                n_split, per = op.plan_splits(B, Hq, Hkv, Skv)
                x = n_split // op.N_WAVES
                assert x in op.GROUPED_WGS_PER_KV_HEAD and n_split % op.N_WAVES == 0 and per % op.TILE == 0
                assert n_split * per >= Skv and x <= max(1, -(-Skv // op.TILE) // op.N_WAVES)
                assert x == 1 or B * Hq * n_split * (op.DV + 1) * 4 <= rt.NOALLOC_SCRATCH_BYTES
    assert op.plan_splits(67, 32, 4, 13634)[0] // op.N_WAVES == 3      # 804 workgroups of a third, not 268 of all keys
    assert op.plan_splits(64, 32, 8, 8001)[0] == op.N_WAVES            # 512 workgroups: two a CU
    op._tuned[(1, 8, 2, 8192)] = 16
    assert op.plan_splits(1, 8, 2, 8192)[0] == 16 * op.N_WAVES
    op.grouped_merge = False
    for B in (1, 5, 33):
        x = op.plan_splits(B, 32, 4, 9000)[0] // op.N_WAVES
        assert x & (x - 1) == 0
    op.grouped_merge, op.target_workgroups = True, 1
    assert op.plan_splits(2, 8, 2, 4096)[0] == op.N_WAVES


def test_split_prefill_plan():
    """Splits cover the cache with none empty and whole tiles, also where the count is chosen by cost; a count that gives
    no CU two workgroups stays."""
    op = AttentionEngine(_meta(1, 16, 16, 4, 512, 128, 128, torch.float16), CustomIO({}), C.make_scale_score_mod(0.1), None,
                         C.OnlineSoftmax())._op
    assert op.split_kv
    for B, H in ((1, 8), (3, 16), (7, 16), (6, 32), (40, 32)):
        for Sq in (1, 31, 64, 90, 230):
            tiles = op.tiles_for(B, H, Sq, 4000)
            for Skv in (1, 300, 522, 9161):
                n_split, per = op.plan_splits(B, H, Sq, Skv, tiles)
                assert per % tiles.block_n == 0 and n_split * per >= Skv > (n_split - 1) * per and n_split >= 1
    tiles = op.tiles_for(7, 16, 31, 522)
    assert op.plan_splits(7, 16, 31, 522, tiles)[0] == 1             # 112 workgroups, not 336 on 256 CUs
    assert op.plan_splits(4, 8, 15, 9539, op.tiles_for(4, 8, 15, 9539))[0] == 8      # 256 workgroups


def test_tail_plan():
    """Shares of what is left over after whole rounds: only where they save time, at least two and at most eight, none empty."""
    from core.lower.prefill_op import PrefillOp
    for slots in range(1, 200):
        for tiles in (16, 46, 110):
            plan = PrefillOp._tail_plan(slots, tiles, 32, 1.0)
            if plan is not None:
                rest, n, per = plan
                assert rest == slots % 32 and 2 <= n <= PrefillOp.MAX_TAIL_PARTS and (n - 1) * per < tiles <= n * per
    assert PrefillOp._tail_plan(64, 46, 32, 1.0) is None and PrefillOp._tail_plan(56, 56, 32, 1.0) is None
    assert PrefillOp._tail_plan(36, 46, 32, 1.0)[0] == 4


def test_causal_prefill_takes_the_faster_kernel(monkeypatch):
    """Causal softmax at head dim 128: the pipelined kernel where its 256-row tiles balance, the generic one elsewhere;
    the caller's tiles, other masks and the environment's choice stay; short calls of a large engine keep its kernel."""
    from core.lower import lower as L
    from core.lower.prefill_op import PrefillOp
    monkeypatch.delenv("AE_PREFILL_KERNEL", raising=False)
    sm, f16 = C.make_scale_score_mod(0.1), torch.float16

    def template(S, mask=C.causal_mask, H=32, B=1, **kw):
        op = PrefillOp(_meta(B, H, H, S, S, 128, 128, f16), CustomIO({}), sm, mask, C.OnlineSoftmax(), "-inf", **kw)
        return op, op.tiles_for(B, H, S, S).template
    op, chosen = template(2009)
    assert chosen == "ae_prefill.hip" and op.tiles.template == "ae_prefill_pipe.hip"
    assert op.tiles_for(2, 32, 4096, 4096).template == "ae_prefill_pipe.hip"
    assert op.tiles_for(1, 32, 100, 100) == op.tiles and op.tiles_for(1, 32, 2009, 4096) == op.tiles
    assert template(4096, B=2)[1] == "ae_prefill_pipe.hip"
    assert template(2009, mask=None)[1] == "ae_prefill_pipe.hip"
    assert template(2009, tiles=L.pipelined_tiles(128, 128))[1] == "ae_prefill_pipe.hip"
    assert not L.pipelined_pays(True, 64, 2867) and L.pipelined_pays(True, 16, 8192) and L.pipelined_pays(False, 16, 9131)
    monkeypatch.setenv("AE_PREFILL_KERNEL", "pipelined")
    assert template(2009)[1] == "ae_prefill_pipe.hip"


def test_a_growing_cache_meets_few_kernels(monkeypatch):
    """Every count of splits that a cache asks for while it grows a token a call runs in a few compiled kernels: the split
    kernels take the count from the launch, merges are built for powers of two.  A combine() that is not the log-sum-exp merge
    has one for its exact count."""
    from core.lower.lower_decode import merge_capacity
    from core.runtime import hip_rt as rt
    built = set()

    class Module:
        def kernel_info(self):
            return {"ae_decode_split_kernel": {}}

    def compiled(template, headers, *a, **kw):
        built.add((template, headers["ae_config.h"]))
        return Module()
    monkeypatch.setattr(rt, "compile_module", compiled)
    monkeypatch.setattr(rt, "check_spills", lambda *a, **kw: None)
    sm, f16 = C.make_scale_score_mod(0.1), torch.float16
    for B, Hq, Hkv in ((1, 32, 8), (4, 32, 8), (19, 64, 8)):
        op = AttentionEngine(_meta(B, Hq, Hkv, 1, 128, 128, 128, f16), CustomIO({}), sm, None, C.OnlineSoftmax()).attention
        built.clear()
        counts = {op.plan_splits(B, Hq, Hkv, S)[0] for S in range(128, 32769, 32)}
        for n in counts:
            _, cfg, ccfg, _ = op._variant(n, True, op._merge_mode(n))
            assert n <= ccfg.block_n < 2 * n and (n == ccfg.block_n or ccfg.merge_in_wg == 1)
        assert len(built) <= 6
    for B, H in ((1, 128), (1, 16), (16, 64)):
        op = AttentionEngine(_meta(B, H, 1, 1, 256, 576, 512, f16), CustomIO({}), sm, None, C.OnlineSoftmax(),
                             kv_shared=True).attention
        built.clear()
        for S in range(256, 8193, 32):
            heads, n, _ = op.plan(B, H, 1, S)
            op._variant(n, False, heads)
            if n > 1:
                op._merges.module(n)
        assert len([1 for t, _ in built if t == "ae_combine.hip"]) <= 6 and len(built) <= 6 + 6
    op = AttentionEngine(_meta(5, 16, 16, 3, 512, 128, 128, f16), CustomIO({}), sm, None, C.OnlineSoftmax()).attention
    built.clear()
    for S in range(512, 16385, 32):
        tiles = op.tiles_for(5, 16, 3, S)
        n, _ = op.plan_splits(5, 16, 3, S, tiles)
        op._variant(tiles, 0, 3, S, n)
        if n > 1:
            op._merges.module(n)
    assert len(built) <= 2 * 2 + 6
    assert [merge_capacity(n, True) for n in (2, 3, 4, 5, 8, 9, 64)] == [2, 4, 4, 8, 8, 16, 64] and merge_capacity(5, False) == 5


def test_a_latent_cache_that_grows_is_planned_once_a_tile():
    """A dense latent cache asks for a plan at every length: the splits are worked out once for all lengths of as many
    tiles, and lengths that were asked for before stay known."""
    from core.lower.lower_decode import MLADecodeOp
    op = AttentionEngine(_meta(3, 128, 1, 1, 256, 576, 512, torch.bfloat16), CustomIO({}), C.make_scale_score_mod(0.1), None,
                         C.OnlineSoftmax(), kv_shared=True).attention
    MLADecodeOp._cheapest.cache_clear()
    plans = [op.plan(3, 128, 1, S) for S in range(4001, 4641)]
    assert MLADecodeOp._cheapest.cache_info().misses == 20 and len(set(plans)) > 1
    assert [op.plan(3, 128, 1, S) for S in range(4001, 4641)] == plans
    assert MLADecodeOp._cheapest.cache_info().misses == 20
    assert all(n * per >= S > (n - 1) * per for S, (_, n, per) in zip(range(4001, 4641), plans))
    assert op.plan(3, 128, 1, 4000, 64)[1] * op.plan(3, 128, 1, 4000, 64)[2] >= 4000         # (a paged call has its own)


def test_the_caller_limits_the_work_memory_of_shared_tiles():
    """``work_limit`` bounds what a call allocates for tiles that several workgroups share, in the forward and in the
    backward: fewer shares, or none; plans made under another limit are dropped."""
    from core.lower.lower import pipelined_tiles
    meta = _meta(2, 32, 8, 2048, 2048, 128, 128, torch.float16)
    op = AttentionEngine(meta, CustomIO({}), C.make_scale_score_mod(0.1), C.causal_mask, C.OnlineSoftmax())._op
    bwd, B, S = op.backward_op(), 2, 1000

    def mb(parts):
        return -(-S // 128) * B * 8 * parts * 128 * 256 * 4e-6 if parts > 1 else 0.0
    free = bwd.dkv_parts(B, 32, 8, S, S, True)
    assert free > 2 and op.work_limit is None
    limits = [int(mb(2) * 1e6) + 1, 0]
    for limit in limits:
        op.work_limit = limit
        got = bwd.dkv_parts(B, 32, 8, S, S, True)
        assert got == (2 if limit else 1) and mb(got) * 1e6 <= limit
    full = AttentionEngine(_meta(3, 8, 8, 2944, 2944, 128, 128, torch.float16), CustomIO({}), C.make_scale_score_mod(0.1), None,
                           C.OnlineSoftmax())._op
    tiles = pipelined_tiles(128, 128)
    rest, n, _ = full._tail(3, 8, 2944, 2944, tiles, 0, 1)
    cleared = []

    class Host:
        def clear(self):
            cleared.append(1)
    full._host = Host()
    full.work_limit = int(8 * rest * (n - 1) * 0.14e6)
    fewer = full._tail(3, 8, 2944, 2944, tiles, 0, 1)
    assert fewer is None or fewer[1] < n
    full.work_limit = 0
    assert full._tail(3, 8, 2944, 2944, tiles, 0, 1) is None and len(cleared) == 2


def test_plans_at_head_dim_64_have_costs_of_their_own():
    """Narrow rows: several workgroups fit a CU, so one split more than a CU each is no second round (split prefill), and a
    short cache is not cut into a workgroup a tile (GQA decode); splits cover the cache with none empty."""
    f16, sm = torch.float16, C.make_scale_score_mod(0.1)
    op = AttentionEngine(_meta(7, 32, 32, 47, 5777, 64, 64, f16), CustomIO({}), sm, None, C.OnlineSoftmax())._op
    assert op.split_kv and op.plan_splits(7, 32, 47, 5777)[0] > 1
    for B, H, Sq in ((1, 8, 1), (5, 16, 40), (7, 32, 130), (3, 16, 250)):
        tiles = op.tiles_for(B, H, Sq, 5000)
        for Skv in (1, 100, 522, 16001):
            n, per = op.plan_splits(B, H, Sq, Skv, tiles)
            assert per % tiles.block_n == 0 and n * per >= Skv > (n - 1) * per
    gqa = AttentionEngine(_meta(48, 16, 2, 1, 871, 64, 64, f16), CustomIO({}), sm, None, C.OnlineSoftmax()).attention
    assert gqa.plan_splits(48, 16, 2, 871)[0] <= 2 * gqa.N_WAVES
    for B, Skv in ((1, 128), (3, 5000), (128, 16000)):
        n, per = gqa.plan_splits(B, 16, 2, Skv)
        assert n // gqa.N_WAVES in gqa.GROUPED_WGS_PER_KV_HEAD and n * per >= Skv


def test_a_build_with_clock_stamps_is_launched_as_one_only(monkeypatch):
    """Kernels built under AE_CLOCK_STAMPS=1 write their stamps through the partial-result pointer, which only a call under
    the same switch sets: builds with and without stamps are kept apart, whatever was compiled in between."""
    sm, f16 = C.make_scale_score_mod(0.1), torch.float16
    mla = AttentionEngine(_meta(128, 128, 1, 1, 256, 576, 512, f16), CustomIO({}), sm, None, C.OnlineSoftmax(),
                          kv_shared=True).attention
    pre = AttentionEngine(_meta(2, 32, 32, 4096, 4096, 128, 128, f16), CustomIO({}), sm, None, C.OnlineSoftmax()).attention
    assert pre.tiles.template == "ae_prefill_pipe.hip"

    def builds():
        got = mla._variant(1), pre._variant(pre.tiles, 0, 4096, 4096)
        assert mla._stamped(1) == ("AE_CLOCK_STAMPS" in got[0][2]) and not mla._stamped(2)
        assert pre._clock_stamps(pre.tiles) == ("#define AE_CLOCK_STAMPS" in got[1][2])
        return got
    plain = builds()
    monkeypatch.setenv("AE_CLOCK_STAMPS", "1")
    stamped = builds()
    mla._variant(4)
    assert builds()[0] is stamped[0] and stamped[0][0] is not plain[0][0] and stamped[1][0] is not plain[1][0]
    monkeypatch.delenv("AE_CLOCK_STAMPS")
    assert builds()[0] is plain[0] and builds()[1] is plain[1]


def test_which_paged_tables_are_cut_by_their_entries_lengths():
    """MLADecodeOp._splits_by_length: no plan below its batch and table limits, none where the equal spans of full tables are
    one round - cut by length those would take longer -, and every plan has a workgroup an entry at least, no more splits
    than tiles, and more splits for a long entry than equal spans give it."""
    from core.lower.lower_decode import MLADecodeOp as Op

    def plan(batch, group, tiles):
        fixed = Op._cheapest(batch, group, tiles, (1, min(Op.MAX_SPLITS, tiles)), 256, 576, 512, True)
        return fixed, Op._splits_by_length(batch, group, tiles, fixed, 256, 576, 512)
    assert plan(3, 128, 64)[1] is None and plan(8, 128, 7)[1] is None
    assert all(plan(*c)[1] is None for c in ((14, 128, 24), (26, 64, 24), (24, 128, 32), (8, 128, 64), (9, 128, 56), (5, 128, 148), (16, 64, 130)))
    by_length = {c: plan(*c) for c in ((64, 128, 128), (5, 128, 80), (21, 64, 82), (32, 64, 80), (31, 64, 66))}
    assert all(p is not None for _, p in by_length.values())
    for batch in range(4, 65):
        for group in (16, 40, 64, 128):
            for tiles in (8, 32, 33, 64, 150):
                c = batch, group, tiles
                fixed, p = plan(*c)
                if p is not None:
                    by_length[c] = fixed, p
    assert len(by_length) >= 15
    for (batch, group, tiles), ((heads0, n0), (heads, most, n_wgs)) in by_length.items():
        assert heads in (16, 32, 64) and 2 <= 2 * most <= tiles and n_wgs >= batch
        assert n_wgs * -(-group // heads) == 256 and most >= 2 * n_wgs / batch
        assert most > n0 or heads < heads0


@pytest.mark.parametrize("spans,n,n_ht,second", [
    ([4] * 8, 4, 8, False),       # 256 workgroups whose padding fits between them
    ([6] * 5, 6, 8, True),        # 240, but an XCD has five units of eight
    ([8] * 16, 8, 1, False),      # 128: not padded
    ([8] * 16, 8, 2, True), ([8] * 16, 8, 3, True),
    ([7] * 16, 8, 2, False),      # the last span of every entry is empty
    ([4] * 3, 4, 8, False), ([1] * 8, 1, 32, False), ([1] * 4, 1, 64, True),
])
def test_when_equal_spans_take_a_second_round(spans, n, n_ht, second):
    """MLADecodeOp._second_round over 256 CUs in 8 XCDs of 4 shader engines, against the same dispatch one workgroup at a time."""
    from core.lower.lower_decode import MLADecodeOp as Op
    assert Op._second_round(spans, n, n_ht, 256) is second
    ids = n | 1 if len(spans) * n * n_ht > 128 else n
    waits = sum(spans) * n_ht > 256
    for xcd in range(8):
        free, stuck = [8] * 4, False
        queue = [unit % ids < spans[unit // ids] for unit in range(len(spans) * ids) if unit % 8 == xcd for _ in range(n_ht)]
        for turn, live in enumerate(queue):
            stuck = stuck or not free[turn % 4]
            waits = waits or (stuck and live)
            free[turn % 4] -= live and not stuck
    assert bool(waits) is second


def test_which_paged_calls_ask_for_splits_by_length():
    """MLADecodeOp.plan: a fourth number where the kernel cuts the entries; equal spans for two latent heads, more entries than
    a wave has lanes, tables of more pages than a workgroup keeps, a dense cache, and a split count that was tuned."""
    from core.lower.lower_decode import MLADecodeOp as Op
    op = AttentionEngine(_meta(64, 128, 1, 1, 256, 576, 512, torch.bfloat16), CustomIO({}), C.make_scale_score_mod(0.1), None,
                         C.OnlineSoftmax(), kv_shared=True).attention
    assert op.plan(64, 128, 1, 4096, 64) == (64, 6, -(-128 // 6) * 32, 128) and op.plan_splits(64, 128, 1, 4096, 64) == (6, 704)
    assert len(op.plan(64, 128, 1, 32 * 1022, 32)) == 4
    for args in ((65, 128, 1, 4096, 64), (64, 128, 1, 4096), (32, 256, 2, 4096, 64), (64, 128, 1, 32 * 1023, 32), (8, 128, 1, 2048, 64)):
        assert len(op.plan(*args)) == 3, args
    op._tuned[64, 128, 1, 4096] = 4
    assert op.plan(64, 128, 1, 4096, 64) == (64, 4, 1024)
    op._tuned[64, 128, 1, 4096] = 0
    assert len(op.plan(64, 128, 1, 4096, 64)) == 4


def _work_of(f, *args):
    """Interpreter steps of one call: what planning costs, without a clock."""
    steps = 0

    def trace(frame, event, _):
        nonlocal steps
        frame.f_trace_opcodes, frame.f_trace_lines = True, False
        steps += event == "opcode"
        return trace
    before = sys.gettrace()
    sys.settrace(trace)
    try:
        f(*args)
    finally:
        sys.settrace(before)
    return steps


def test_the_choice_among_equal_spans_is_cheap():
    """MLADecodeOp._cheapest is asked anew whenever the cache grows by a tile: some 80 interpreter steps a
    candidate and kind of batch (160 with a function called for each)."""
    from core.lower.lower_decode import MLADecodeOp as Op
    for batch, group, tiles in ((1, 128, 64), (8, 128, 64), (33, 128, 128), (64, 64, 128), (21, 64, 66)):
        splits = {-(-tiles // -(-tiles // n)) for n in range(1, min(Op.MAX_SPLITS, tiles) + 1)}
        forms = sum(h == 16 or group > h // 2 for h in Op.ROUND_COST)
        for paged in (False, True):
            work = _work_of(Op._cheapest.__wrapped__, batch, group, tiles, (1, min(Op.MAX_SPLITS, tiles)), 256, 576, 512, paged)
            assert work <= 110 * len(splits) * forms * (1 + paged), (batch, tiles, paged, work)


def test_the_choice_of_splits_by_length_is_cheap():
    """MLADecodeOp._splits_by_length is asked for every new batch and table width: no walk over the entries for each
    candidate (190000 interpreter steps at 64 entries), and the dispatch is followed for the plans that are left."""
    from core.lower.lower_decode import MLADecodeOp as Op
    for batch in (4, 5, 8, 16, 17, 33, 64):
        for group in (16, 64, 128):
            for tiles in (8, 33, 64, 128, 250):
                fixed = Op._cheapest(batch, group, tiles, (1, min(Op.MAX_SPLITS, tiles)), 256, 576, 512, True)
                work = _work_of(Op._splits_by_length.__wrapped__, batch, group, tiles, fixed, 256, 576, 512)
                assert work <= 20000, (batch, group, tiles, work)


def test_a_paged_build_takes_a_number_of_stages():
    """AE_NSTAGE of the wave-specialised latent decode (4: its waits count the requests in flight) may come with the configuration,
    for a paged cache too."""
    from core.lower.lower_decode import render_mla_config
    from core.runtime import hip_rt as rt
    f = L.trace_functors(C.make_scale_score_mod(0.1), None, C.OnlineSoftmax(), CustomIO({}), torch.bfloat16)
    cfg = render_mla_config(512, 64, 512, torch.bfloat16, 32, 0, 1, False, 2, f.softmax, True, 16) + "#define AE_NSTAGE 4\n"
    names = f.final_rowscale_names
    rt.compile_module("ae_mla_decode_ws.hip", {"ae_config.h": cfg, "ae_functors.h": L.render_functors(f) + lower_combine(C.OnlineSoftmax(), names)})
