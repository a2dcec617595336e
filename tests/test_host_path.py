"""The native host path of repeated calls (csrc/ae_host.cpp): a second call of a shape runs there, gives what the first
one gave, and calls that its plans do not cover go back to the operators' Python code."""
import math

import pytest
import torch

import attn_cases as C
from attn_engine import AttentionEngine
from core import CustomIO, meta_tensor


def _engine(B, Hq, Hkv, Sq, Skv, D, dtype=torch.float16, mask=None, sigmoid=False):
    meta = (meta_tensor(B, Hq, Sq, D, dtype=dtype), meta_tensor(B, Hkv, Skv, D, dtype=dtype),
            meta_tensor(B, Hkv, Skv, D, dtype=dtype))
    if sigmoid:
        return AttentionEngine(meta, CustomIO({"softmax_bias": (1,)}), C.make_sigmoid_score_mod(1 / math.sqrt(D)), mask,
                               C.OnlineIdentity())
    return AttentionEngine(meta, CustomIO({}), C.make_scale_score_mod(1 / math.sqrt(D)), mask, C.OnlineSoftmax())


def test_without_a_plan_or_a_gpu_tensor_nothing_runs():
    mod = _engine(1, 2, 2, 64, 64, 64, mask=C.causal_mask)
    q = torch.zeros(1, 64, 2, 64, dtype=torch.float16)
    host = mod._op._host
    assert len(host) == 0 and host.run(q, q, q) is None and host.run(q, q) is None
    with pytest.raises(RuntimeError, match="on the GPU"):
        mod(q, q, q)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["causal", "window", "sigmoid", "gqa_decode", "gqa_decode_split", "mha_split"])
def test_repeated_calls_run_natively_and_agree(cuda_device, monkeypatch, case):
    B, Hq, Hkv, Sq, Skv, D, mask = {
        "causal": (2, 4, 2, 333, 333, 64, C.causal_mask), "window": (1, 4, 4, 300, 300, 64, C.make_sliding_window_mask(70)),
        "sigmoid": (1, 2, 2, 130, 130, 64, None), "gqa_decode": (64, 8, 2, 1, 300, 128, None),
        "gqa_decode_split": (1, 8, 2, 1, 3001, 128, None), "mha_split": (1, 2, 2, 33, 1000, 64, None)}[case]
    mod = _engine(B, Hq, Hkv, Sq, Skv, D, mask=mask, sigmoid=case == "sigmoid")
    extra = (torch.tensor([-3.0], device=cuda_device),) if case == "sigmoid" else ()
    host, hits = mod._op._host, []

    class Counted:
        def __getattr__(self, name):
            f = getattr(host, name)
            return f if name != "run" else (lambda *a: hits.append(f(*a)) or hits[-1])
    mod._op._host = Counted()
    q, k, v = (t.to(cuda_device) for t in C.make_inputs(B, Sq, Skv, Hq, Hkv, D, D, torch.float16))
    first = mod(q, k, v, *extra).clone()
    scales = {n: t.clone() for n, t in mod.final_rowscales.items()}
    assert hits[-1] is None and len(host) == 1
    for _ in range(3):
        out = mod(q, k, v, *extra)
        assert hits[-1] is not None and torch.equal(out, first)
        assert set(mod.final_rowscales) == set(scales)
        assert all(torch.equal(mod.final_rowscales[n], scales[n]) for n in scales)
    # strides the kernels cannot read, another dtype of a custom input, another shape: not this path
    odd = torch.empty(B, Skv, Hkv, D + 4, dtype=torch.float16, device=cuda_device)[..., 4:].copy_(k)
    assert torch.equal(mod(q, odd, v, *extra), first) and hits[-1] is None
    if extra:
        assert torch.equal(mod(q, k, v, extra[0].double()), first) and hits[-1] is None
    with pytest.raises(ValueError):
        mod(q, k[:, :-1], v, *extra)
    # a switch that is read at every call: its plan does not serve the other setting
    if case == "gqa_decode":
        monkeypatch.setenv("AE_DECODE_MERGE_IN_WG", "0")
        assert torch.equal(mod(q, k, v), first) and hits[-1] is None
    if case.startswith("gqa"):
        mod._op.static_workspace = True
        mod(q, k, v)
        assert hits[-1] is None and len(host) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["softmax", "window", "sigmoid"])
def test_repeated_training_steps_run_natively_and_agree(cuda_device, kind):
    B, H, S, D = 2, 4, 200, 64
    mask = {"softmax": C.causal_mask, "window": C.make_sliding_window_mask(70), "sigmoid": None}[kind]
    mod = _engine(B, H, H, S, S, D, mask=mask, sigmoid=kind == "sigmoid")
    extra = (torch.tensor([-3.0], device=cuda_device),) if kind == "sigmoid" else ()
    q, k, v = (t.to(cuda_device).requires_grad_(True) for t in C.make_inputs(B, S, S, H, H, D, D, torch.float16))
    do = torch.randn(B, S, H, D, device=cuda_device).half()
    steps = []
    for i in range(3):
        out = mod(q, k, v, *extra)
        assert ("AttentionEngineBackward" in out.grad_fn.name()) == (i > 0)
        grads = torch.autograd.grad(out, (q, k, v), do if i < 2 else do.transpose(0, 1).contiguous().transpose(0, 1))
        steps.append([out.detach(), *grads])
    for other in steps[1:]:
        assert all(torch.equal(a, b) for a, b in zip(steps[0], other))
    with torch.no_grad():
        assert mod(q, k, v, *extra).grad_fn is None
    out = mod(q, k, v, *extra)
    out.backward(do)
    with pytest.raises(RuntimeError, match="second time"):
        out.backward(do)
