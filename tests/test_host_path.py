"""The native host path of repeated calls (csrc/ae_host.cpp): a second call of a shape runs there, gives what the first
one gave, and calls that its plans do not cover go back to the operators' Python code."""
import math
import sys
import threading
import time

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


def _split_decode(cuda_device, Skv=3001, B=1, Hq=8, Hkv=2, D=128):
    mod = _engine(B, Hq, Hkv, 1, Skv, D)
    q, k, v = (t.to(cuda_device) for t in C.make_inputs(B, 1, Skv, Hq, Hkv, D, D, torch.float16))
    op = mod._op
    n_split, _ = op.plan_splits(B, Hq, Hkv, Skv)
    assert op.merges_in_last_workgroup(n_split) and op.grouped_merge

    def work(stream):      # the buffers of this call on a stream
        return op._host.work(B * Hq * n_split // op.N_WAVES, B * Hq * n_split, B * Hkv, cuda_device.index or 0, stream.cuda_stream)
    return mod, q, k, v, work


@pytest.mark.gpu
def test_kept_work_buffers_outlive_the_plans(cuda_device):
    """A graph captured on a warmed-up stream replays on the buffers that were kept for it, whatever shapes, strides and
    settings the operator has been called with since."""
    mod, q, k, v, work = _split_decode(cuda_device)
    want, s = mod(q, k, v).clone(), torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(2):
            assert torch.equal(mod(q, k, v), want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out = mod(q, k, v)
    kept = [t.data_ptr() for t in work(s)]
    assert work(s)[0].shape[0] == mod._op.plan_splits(1, 8, 2, 3001)[0] * 8 // mod._op.N_WAVES
    odd = torch.empty(*k.shape[:3], k.shape[3] + 4, dtype=k.dtype, device=k.device)[..., 4:].copy_(k)
    for r in range(3):
        with torch.cuda.stream(s):
            for n in range(100, 3001, 41):               # more shapes than plans are kept
                mod(q, k[:, :n], v[:, :n])
            assert torch.equal(mod(q, odd, v), want)     # the Python path: its plan replaces the shape's
            mod._op.target_workgroups = 256              # drops every plan
            assert torch.equal(mod(q, k, v), want)
            out.zero_()
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), r
    assert [t.data_ptr() for t in work(s)] == kept


@pytest.mark.gpu
def test_a_capture_on_a_new_stream_has_its_own_work_buffers(cuda_device):
    """Counters that a capture clears are zero only once that graph has been replayed."""
    mod, q, k, v, work = _split_decode(cuda_device)
    want, s = mod(q, k, v).clone(), torch.cuda.Stream()
    torch.cuda.synchronize()
    graphs, outs = [torch.cuda.CUDAGraph() for _ in range(2)], []
    for g in graphs:
        with torch.cuda.graph(g, stream=s):
            outs.append(mod(q, k, v))
    for i in (1, 1, 0, 1, 0):
        with torch.cuda.stream(s):
            outs[i].zero_()
            graphs[i].replay()
            assert torch.equal(outs[i], want), i
            assert torch.equal(mod(q, k, v), want)       # an eager call on the stream the graphs were captured on
        torch.cuda.synchronize()


class _Labelled(torch.Tensor):
    """A subclass that only overrides what happens to its calls (no dispatch key of its own)."""
    calls = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.calls.append(getattr(func, "__name__", str(func)))
        return super().__torch_function__(func, types, args, kwargs or {})


@pytest.mark.gpu
def test_tensor_subclasses_go_to_python(cuda_device):
    mod = _engine(1, 2, 2, 70, 70, 64, mask=C.causal_mask)
    q, k, v = (t.to(cuda_device) for t in C.make_inputs(1, 70, 70, 2, 2, 64, 64, torch.float16))
    want = mod(q, k, v)
    host = mod._op._host
    assert len(host) == 1 and host.run(q, k, v) is not None and host.run(torch.nn.Parameter(q, False), k, v) is not None
    assert host.run(q.as_subclass(_Labelled), k, v) is None and host.run(q, k, v.as_subclass(_Labelled)) is None
    _Labelled.calls.clear()
    assert torch.equal(mod(q.as_subclass(_Labelled), k, v).as_subclass(torch.Tensor), want) and _Labelled.calls


@pytest.mark.gpu
def test_forward_mode_is_refused_on_every_call(cuda_device):
    import torch.autograd.forward_ad as fw
    mod = _engine(1, 2, 2, 70, 70, 64, mask=C.causal_mask)
    q, k, v = (t.to(cuda_device).requires_grad_(True) for t in C.make_inputs(1, 70, 70, 2, 2, 64, 64, torch.float16))
    for i in range(3):
        out = mod(q, k, v)
        assert ("AttentionEngineBackward" in out.grad_fn.name()) == (i > 0)
        torch.autograd.grad(out, (q, k, v), torch.ones_like(out))
        with fw.dual_level(), pytest.raises(NotImplementedError, match="jvp"):
            mod(fw.make_dual(q, torch.ones_like(q)), k, v)


@pytest.mark.gpu
def test_other_threads_run_while_a_call_launches(cuda_device):
    mod = _engine(1, 2, 2, 70, 70, 64, mask=C.causal_mask)
    q, k, v = (t.to(cuda_device) for t in C.make_inputs(1, 70, 70, 2, 2, 64, 64, torch.float16))
    mod(q, k, v)
    run, turns, stop, old = mod._op._host.run, [0], [], sys.getswitchinterval()

    def other():
        while not stop:
            turns[0] += 1
            time.sleep(0)                   # gives the interpreter lock back
    t = threading.Thread(target=other)
    t.start()
    try:
        sys.setswitchinterval(60.0)         # this thread gives it up of its own accord only
        time.sleep(0.1)                     # (the other one no longer waits by the old interval)
        before = turns[0]
        for i in range(5000):
            run(q, k, v)
        # (50,000 and more where the launches give the lock back; 4 to 400 where they kept it: other parts of a call,
        # the freeing of its results for one, give it back now and then)
        assert turns[0] - before > 2500
    finally:
        sys.setswitchinterval(old)
        stop.append(True)
        t.join()
