"""Masks that are a band of q - kv (core/lower/mask.py) and merges that may be grouped (core/lower/lower_decode.py): what
the planners recognise, and the banded kernel against the oracle."""
import math

import pytest
import torch

import attn_cases as C
from attn_engine import AttentionEngine
from core import CustomIO, meta_tensor
from core.lower.lower_decode import merges_in_any_order
from core.lower.mask import lower_mask_mod, plan_mask
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
