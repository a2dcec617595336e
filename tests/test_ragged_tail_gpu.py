"""Keys past the end of a sequence whose length is not a multiple of the kv tile: they take no part in the result, whatever
the strides of K and V and whatever a score of them would be."""
import math

import pytest
import torch

import attn_cases as C
from attn_engine import AttentionEngine
from core import CustomIO, meta_tensor
from oracle import attention_ref as R

pytestmark = pytest.mark.gpu

# (environment of the constructor, heads): waves that share the kv axis (the small default), the generic and the
# software-pipelined kernel
KERNELS = {"groups": "", "generic": "generic", "pipelined": "pipelined"}


def _engine(monkeypatch, kernel, score_mod, H, S, D, dtype, mask=None, custom=("softmax_bias",)):
    monkeypatch.setenv("AE_PREFILL_KERNEL", KERNELS[kernel])
    meta = (meta_tensor(1, H, S, D, dtype=dtype),) * 3
    mod = AttentionEngine(meta, CustomIO({n: (1,) for n in custom}), score_mod, mask, C.OnlineIdentity())
    assert mod._op.functors.elementwise and "#define AE_EVEN_KV 0" in mod._op.source
    assert (mod._op.tiles.kv_groups > 1) == (kernel == "groups")
    assert (mod._op.tiles.rows_per_wave == 64) == (kernel == "pipelined")
    return mod


def _sigmoid(q, k, v, bias, causal):
    s = torch.einsum("bqhd,bkhd->bhqk", q.double(), k.double()) / math.sqrt(q.shape[-1]) + bias
    if causal:
        s = s.masked_fill(~torch.ones(s.shape[-2:], dtype=torch.bool).tril(), -math.inf)
    return torch.einsum("bhqk,bkhd->bqhd", torch.sigmoid(s), v.double())


def _layout(t, how):
    """A [1, S, H, D] tensor with rows that overlap: expanded along the sequence (stride 0), or 8 elements apart."""
    if how == "own":
        return t
    if how == "expanded":
        return t[:, :1].expand(-1, t.shape[1], -1, -1)
    _, S, H, D = t.shape
    flat = t.permute(2, 0, 1, 3).reshape(H, -1)[:, :8 * (S - 1) + D].contiguous()
    return flat.as_strided((1, S, H, D), (flat.numel(), 8, flat.shape[1], 1)) if flat.shape[1] % 8 == 0 else None


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kl,vl", [("own", "expanded"), ("expanded", "expanded"), ("own", "near"), ("near", "own")])
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
def test_rows_of_k_and_v_may_overlap(cuda_device, monkeypatch, kernel, causal, kl, vl, D, dtype):
    H, S = 2, 130
    print(f"case overlap {kernel} causal={causal} {kl} {vl} D{D}", flush=True)
    mod = _engine(monkeypatch, kernel, C.make_sigmoid_score_mod(1 / math.sqrt(D)), H, S, D, dtype,
                  C.causal_mask if causal else None)
    q, k, v = (t.cuda() for t in C.make_inputs(1, S, S, H, H, D, D, dtype, seed=5))
    k, v = _layout(k, kl), _layout(v, vl)
    ref = _sigmoid(q.cpu(), k.cpu(), v.cpu(), -1.0, causal)
    for _ in range(2):                       # (the second call of a shape is launched natively)
        out = mod(q, k, v, torch.tensor([-1.0], device="cuda")).double().cpu()
        # weights and results are rounded to the input type: S weights of at most 1 and as many terms of V
        eps = 2.0 ** (-11 if dtype == torch.float16 else -8)
        bound = eps * (ref.abs() + (v.double().abs().cpu()).sum(dim=1, keepdim=True)) + 1e-6
        assert ((out - ref).abs() <= bound).all()


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_an_infinite_query_spoils_nothing_where_the_weight_saturates(cuda_device, monkeypatch, kernel, dtype):
    H, S, D = 2, 130, 64
    mod = _engine(monkeypatch, kernel, C.make_sigmoid_score_mod(1 / math.sqrt(D)), H, S, D, dtype)
    q, k, v = C.make_inputs(1, S, S, H, H, D, D, dtype, seed=6)
    q[0, 7, :, 3], q[0, 129, :, 0] = math.inf, -math.inf
    k[k.abs() < 2 ** -6] = 2 ** -6           # (no inf * 0 among the keys that exist)
    out = mod(q.cuda(), k.cuda(), v.cuda(), torch.tensor([-1.0], device="cuda")).double().cpu()
    ref = _sigmoid(q, k, v, -1.0, False)
    assert torch.isfinite(ref).all() and torch.isfinite(out).all()
    eps = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert ((out - ref).abs() <= eps * (ref.abs() + v.double().abs().sum(dim=1, keepdim=True)) + 1e-6).all()


@pytest.mark.parametrize("kernel", KERNELS)
def test_the_weight_of_a_zero_score_may_overflow_the_input_type(cuda_device, monkeypatch, kernel):
    """Scores of about -65536 under a bias of 70000: every weight fits fp16, the one of a score of 0 does not."""
    H, S, D = 2, 130, 64

    def score_mod(score, custom_fwd_inputs, b, h, q_idx, kv_idx):
        return (score + custom_fwd_inputs.input_tensors["softmax_bias"]).max(0)
    mod = _engine(monkeypatch, kernel, score_mod, H, S, D, torch.float16)
    q = torch.full((1, S, H, D), 32.0, dtype=torch.float16)
    k = torch.full((1, S, H, D), -32.0, dtype=torch.float16)
    v = (C.make_inputs(1, S, S, H, H, D, D, torch.float16, seed=8)[2].float() / 1024).half()
    out = mod(q.cuda(), k.cuda(), v.cuda(), torch.tensor([70000.0], device="cuda")).double().cpu()
    ref = 4464.0 * v.double().sum(dim=1, keepdim=True).expand_as(out)      # (4464 is a value of fp16: the weights are exact)
    assert ((out - ref).abs() <= 2.0 ** -10 * ref.abs() + 1e-3).all()


def _softmax_engine(monkeypatch, kernel, S, D, dtype, mask=None):
    monkeypatch.setenv("AE_PREFILL_KERNEL", KERNELS[kernel])
    meta = (meta_tensor(1, 2, S, D, dtype=dtype),) * 3
    mod = AttentionEngine(meta, CustomIO({}), C.make_scale_score_mod(1 / math.sqrt(D)), mask, C.OnlineSoftmax())
    assert (mod._op.tiles.kv_groups > 1) == (kernel == "groups")
    assert (mod._op.tiles.rows_per_wave == 64) == (kernel == "pipelined")
    return mod


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kl,vl", [("own", "expanded"), ("expanded", "own"), ("near", "near")])
def test_rows_may_overlap_under_the_softmax(cuda_device, monkeypatch, kernel, causal, kl, vl):
    S, D, dtype = 130, 128, torch.float16
    mod = _softmax_engine(monkeypatch, kernel, S, D, dtype, C.causal_mask if causal else None)
    q, k, v = (t.cuda() for t in C.make_inputs(1, S, S, 2, 2, D, D, dtype, seed=15))
    k, v = _layout(k, kl), _layout(v, vl)
    ref, rlse = R.softmax_attention(q.cpu(), k.cpu(), v.cpu(), causal=causal)
    for _ in range(2):
        out = mod(q, k, v).float().cpu()
        assert (out - ref).abs().max().item() <= 2e-2
        assert (mod.final_rowscales["lse"].cpu() - rlse).abs().max().item() <= 1e-3


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("where", [3, 70, 129])
@pytest.mark.parametrize("value", [math.nan, math.inf])
@pytest.mark.parametrize("causal", [False, True])
def test_a_key_that_is_not_finite_spoils_the_rows_that_see_it(cuda_device, monkeypatch, kernel, where, value, causal):
    S, D, dtype = 130, 64, torch.bfloat16
    mod = _softmax_engine(monkeypatch, kernel, S, D, dtype, C.causal_mask if causal else None)
    q, k, v = C.make_inputs(1, S, S, 2, 2, D, D, dtype, seed=16)
    q = q.abs() + 2 ** -6                        # (an infinite key scores +inf with every row, and inf - inf is NaN)
    ref, _ = R.softmax_attention(q, k, v, causal=causal)
    k[:, where], k[:, where, :, 1] = 0.0, value
    out = mod(q.cuda(), k.cuda(), v.cuda()).float().cpu()
    sees = torch.arange(S) >= where if causal else torch.ones(S, dtype=torch.bool)
    assert torch.isnan(out[:, sees]).all()
    assert not causal or (out[:, ~sees] - ref[:, ~sees]).abs().max().item() <= 2e-2
