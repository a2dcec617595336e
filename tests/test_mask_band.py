"""Masks that are a band of q - kv (core/lower/mask.py) and merges that may be grouped (core/lower/lower_decode.py): what
the planners recognise, and the banded kernel against the oracle."""
import math

import pytest
import torch

import attn_cases as C
from attn_engine import AttentionEngine
from core import CustomIO, meta_tensor
from core.lower.lower_decode import merges_in_any_order
from core.lower.mask import lower_mask_mod, plan_mask, survey_mask
from oracle import attention_ref as R
from oracle import masks as OM


def _band(mask_mod, Sq, Skv, H=1, **kw):
    return plan_mask(mask_mod, lower_mask_mod(mask_mod), 1, H, Sq, Skv, 128, 64, **kw).band


def test_bands_are_recognised():
    assert _band(C.make_sliding_window_mask(70), 300, 300) == (0, 69)
    assert _band(C.make_sliding_window_mask(70), 300, 300, chunk_rows=128) == (0, 69)
    assert _band(C.make_sliding_window_mask(500), 300, 300) is None           # plain causal at this size: mode 1
    assert _band(C.causal_mask, 130, 300) == (0, None)
    assert _band(C.causal_plus_one_mask, 300, 300) == (-1, None)
    assert _band(C.causal_shifted_mask, 300, 300) == (128, None)
    assert _band(lambda b, h, q, kv: (q >= kv) & (kv != 5), 300, 300) is None  # a hole
    assert _band(lambda b, h, q, kv: (q // 64) >= (kv // 64), 300, 300) is None
    assert _band(C.head_dependent_mask, 300, 300, H=4) is None
    assert _band(lambda b, h, q, kv: q - 1000 >= kv, 300, 300) is None         # nothing visible
    assert _band(C.make_sliding_window_mask(70), 300, 300, elementwise=False) is None


def test_merges_that_may_be_grouped():
    class Mean(C.OnlineSoftmax):
        @staticmethod
        def combine(final_rowscales):
            lse = final_rowscales["lse"]
            return (lse - lse.get_reduce("max")).exp()
    assert merges_in_any_order(C.OnlineSoftmax(), ["lse"])
    assert not merges_in_any_order(Mean(), ["lse"])
    assert not merges_in_any_order(C.OnlineIdentity(), [])


@pytest.mark.gpu
@pytest.mark.parametrize("name,Sq,Skv", [("window", 1100, 1100), ("window", 300, 500), ("causal", 200, 500), ("causal", 500, 200),
                                         ("plus_one", 513, 513), ("shifted", 700, 700)])
@pytest.mark.parametrize("D", [64, 128])
def test_banded_masks_against_the_oracle(cuda_device, name, Sq, Skv, D):
    """16 heads x 6 batch entries: more q tiles than kv-group tiles are chosen for."""
    mask = {"window": C.make_sliding_window_mask(100), "causal": C.causal_mask, "plus_one": C.causal_plus_one_mask,
            "shifted": C.causal_shifted_mask}[name]
    B, H, dtype = 6, 16, torch.float16
    q, k, v = C.make_inputs(B, Sq, Skv, H, H, D, D, dtype, seed=Sq)

    class NoCombine(C.OnlineSoftmax):                                         # (unequal lengths stay unsplit)
        combine = C.OnlineIdentity.combine

    meta = (meta_tensor(B, H, Sq, D, dtype=dtype), meta_tensor(B, H, Skv, D, dtype=dtype), meta_tensor(B, H, Skv, D, dtype=dtype))
    mod = AttentionEngine(meta, CustomIO({}), C.make_scale_score_mod(1 / math.sqrt(D)), mask,
                          C.OnlineSoftmax() if Sq == Skv else NoCombine())
    assert "#define AE_BAND 1" in mod.tl_code
    out = mod(q.cuda(), k.cuda(), v.cuda()).float().cpu()
    lse = mod.final_rowscales["lse"].cpu()
    b = slice(B - 1, B)
    ref, rlse = R.softmax_attention(q[b], k[b], v[b], causal=False, mask=torch.from_numpy(OM.dense_mask_grid(mask, 1, H, Sq, Skv)))
    seen = torch.isfinite(rlse)
    assert (out[b] - ref.nan_to_num(0.0)).abs().max().item() <= 2e-2
    assert torch.equal(torch.isfinite(lse[b]), seen) and (lse[b][seen] - rlse[seen]).abs().max().item() <= 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("lo,hi", [(0, 0), (0, 31), (0, 96), (0, 97), (0, 128), (0, 500), (-70, 30), (65, 200), (-40, 0)])
@pytest.mark.parametrize("D", [64, 128])
def test_bands_with_two_ends_start_inside_their_range(cuda_device, lo, hi, D):
    """Every kv tile of a q tile's range is multiplied once, wherever the walk starts (AE_ROTATE)."""
    B, H, S, dtype = (9 if D == 64 else 3), 32, 555, torch.float16          # (no groups of waves along the kv axis)
    mask = lambda b, h, q, kv: (q - lo >= kv) & (q - hi <= kv)  # noqa: E731
    q, k, v = C.make_inputs(B, S, S, H, H, D, D, dtype, seed=7)
    meta = tuple(meta_tensor(B, H, S, D, dtype=dtype) for _ in range(3))
    mod = AttentionEngine(meta, CustomIO({}), C.make_scale_score_mod(1 / math.sqrt(D)), mask, C.OnlineSoftmax())
    assert "#define AE_BAND 1" in mod.tl_code
    out = mod(q.cuda(), k.cuda(), v.cuda()).float().cpu()
    lse = mod.final_rowscales["lse"].cpu()
    b = slice(B - 1, B)
    ref, rlse = R.softmax_attention(q[b], k[b], v[b], causal=False, mask=torch.from_numpy(OM.dense_mask_grid(mask, 1, H, S, S)))
    seen = torch.isfinite(rlse)
    assert torch.equal(torch.isfinite(lse[b]), seen) and (lse[b][seen] - rlse[seen]).abs().max().item() <= 1e-3
    # sum of |P rounding| <= 2^-11 (the weights sum to 1), times the largest |v|, and the result's own rounding
    bound = 2.0 ** -10 * v.float().abs().max().item() + 2.0 ** -11 * ref.nan_to_num(0.0).abs().max().item()
    assert (out[b] - ref.nan_to_num(0.0)).abs().max().item() <= bound


@pytest.mark.parametrize("Sq,Skv", [(1, 1), (31, 33), (300, 300), (130, 517), (517, 130), (256, 64)])
@pytest.mark.parametrize("name", ["causal", "plus_one", "window", "head", "holes", "all", "none"])
def test_tables_put_together_from_one_survey(name, Sq, Skv):
    """One evaluation of a mask serves every tile shape: the tables are the oracle's, and band and mode do not depend on
    how it was cut into rows and blocks."""
    mod = {"causal": C.causal_mask, "plus_one": C.causal_plus_one_mask, "window": C.make_sliding_window_mask(70),
           "head": C.head_dependent_mask, "holes": lambda b, h, q, kv: (q >= kv) & (kv % 40 != 5),
           "all": lambda b, h, q, kv: q + kv >= 0, "none": lambda b, h, q, kv: q + kv < 0}[name]
    lm = lower_mask_mod(mod)
    survey = survey_mask(mod, lm, 2, 3, Sq, Skv, chunk_rows=64)
    dense = OM.dense_mask_grid(mod, 2 if lm.uses_b else 1, 3 if lm.uses_h else 1, Sq, Skv)
    for tm, tn in ((32, 32), (64, 32), (128, 32), (128, 64), (256, 64), (64, 128)):
        plan = plan_mask(mod, lm, 2, 3, Sq, Skv, tm, tn, survey=survey)
        alone = plan_mask(mod, lm, 2, 3, Sq, Skv, tm, tn)
        assert (plan.mode, plan.band) == (alone.mode, alone.band)
        assert (plan.mode == 1) == (Sq == Skv and bool((torch.from_numpy(dense)[0, 0] == torch.ones(Sq, Skv).tril().bool()).all()))
        if plan.mode == 2:
            assert torch.equal(plan.table, alone.table)
            assert torch.equal(plan.table, torch.from_numpy(OM.block_classes(dense, tm, tn)).to(torch.int8))
        if plan.band is not None:
            lo, hi = plan.band
            d = torch.arange(Sq).view(-1, 1) - torch.arange(Skv).view(1, -1)
            assert torch.equal((d >= lo) & (d <= (Sq if hi is None else hi)), torch.from_numpy(dense)[0, 0])


def test_construction_evaluates_a_mask_once(monkeypatch):
    """... whatever tiles are tried on the way (bands, waves that share the kv axis)."""
    from core.lower import mask
    seen = []
    real = mask.survey_mask
    monkeypatch.setattr("core.lower.prefill_op.survey_mask", lambda *a, **k: seen.append(a[4:6]) or real(*a, **k))
    monkeypatch.setattr(mask, "survey_mask", lambda *a, **k: seen.append(a[4:6]) or real(*a, **k))
    for mod, S in ((C.causal_mask, 333), (C.causal_mask, 4096), (C.make_sliding_window_mask(256), 4096)):
        seen.clear()
        AttentionEngine((meta_tensor(1, 32, S, 128, dtype=torch.float16),) * 3, CustomIO({}), C.make_scale_score_mod(0.1), mod,
                        C.OnlineSoftmax())
        assert seen == [(S, S)]
