"""GPU parity of the backward of softmax attention: dq, dk, dv from libae_hip.so (through
AttentionEngine and torch.autograd) against the CPU oracle's closed-form gradients on the same seeded
inputs.  The oracle consumes the fp16/bf16-rounded inputs and computes in fp32; a gradient element may
differ by 2e-2 + 1% of the largest magnitude of that gradient (the kernels round p and ds to the input
type before the second products and the results to the input type)."""
import math

import pytest
import torch

import attn_cases as C
from attn_engine import AttentionEngine
from core import CustomIO, meta_tensor
from oracle import attention_ref as R
from oracle import masks as M

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _nothing_cached():
    """Tests that limit the allocator's memory count on no room inside what earlier tests' tensors left to it."""
    if torch.cuda.is_available():
        torch.cuda.empty_cache()


class OnlineSoftmaxTwoScales(C.OnlineSoftmax):
    """The online softmax of attn_script/mha.py with its reference point and its row sum exported as TWO final row
    scales (instead of their combination lse), and the recompute / backward rules written against both, in the
    protocol of the reference (attn_engine/attn_engine.py:75-93; every final row scale is handed to forward() and
    backward(), core/lower/lower.py:413-453).  The lowering cannot take it for the softmax it has a fixed backward
    for, so both rules are traced; the function it computes is still softmax attention."""

    def __init__(self):
        super().__init__()
        from core import SymbolScalar, Var
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


def _engine(B, H, Hkv, S, D, DV, dtype, mask_mod, scale):
    meta = (meta_tensor(B, H, S, D, dtype=dtype), meta_tensor(B, Hkv, S, D, dtype=dtype),
            meta_tensor(B, Hkv, S, DV, dtype=dtype))
    return AttentionEngine(meta, CustomIO({}), score_mod=C.make_scale_score_mod(scale), mask_mod=mask_mod,
                           online_func=C.OnlineSoftmax())


def _check(got, ref, what, case):
    tol = 2e-2 + 1e-2 * ref.abs().max().item()
    err = (got.float().cpu() - ref).abs().max().item()
    assert math.isfinite(err) and err <= tol, (what, case, err, tol)


def _run(B, H, Hkv, Sq, Skv, D, DV, dtype, mask_mod, causal, seed=3):
    scale = 1 / math.sqrt(D)
    q, k, v = C.make_inputs(B, Sq, Skv, H, Hkv, D, DV, dtype, seed=seed)
    g = torch.Generator().manual_seed(seed + 100)
    do = torch.randn(B, Sq, H, DV, generator=g).to(dtype)
    mod = _engine(B, H, Hkv, Sq, D, DV, dtype, mask_mod, scale)
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    out = mod(qd, kd, vd)
    out.backward(do.cuda())
    dense = None
    if mask_mod is not None and not causal:
        dense = torch.from_numpy(M.dense_mask_grid(mask_mod, B, H, Sq, Skv))
    ref_out, _ = R.softmax_attention(q, k, v, scale=scale, causal=causal, mask=dense)
    assert (out.detach().float().cpu() - ref_out).abs().max().item() <= 2e-2
    dq, dk, dv = R.softmax_attention_grads(q, k, v, do, scale=scale, causal=causal, mask=dense)
    case = (B, H, Hkv, Sq, Skv, D, DV, dtype, causal)
    _check(qd.grad, dq, "dq", case)
    _check(kd.grad, dk, "dk", case)
    _check(vd.grad, dv, "dv", case)
    assert qd.grad.dtype == dtype and kd.grad.shape == k.shape and vd.grad.shape == v.shape


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,H,Hkv,S,D,dtype", [
    (1, 2, 2, 256, 128, torch.float16),
    (2, 4, 4, 512, 64, torch.float16),
    (1, 2, 2, 384, 128, torch.bfloat16),
    (1, 4, 2, 320, 128, torch.float16),      # grouped heads: dk, dv sum over the group
    (1, 2, 1, 200, 64, torch.bfloat16),      # ragged: S not a multiple of any tile
    (1, 1, 1, 77, 128, torch.float16),
])
def test_softmax_backward(cuda_device, B, H, Hkv, S, D, dtype, causal):
    print(f"case bwd B{B} H{H} Hkv{Hkv} S{S} D{D} {dtype} causal={causal}", flush=True)
    _run(B, H, Hkv, S, S, D, D, dtype, C.causal_mask if causal else None, causal)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Hkv,Sq,Skv", [
    (1, 1, 1, 1, 1),           # one item, one row
    (1, 2, 1, 64, 64),         # one tile per head of the group: every step is on to the next head
    (1, 6, 2, 65, 65),         # ... a last tile of one row
    (2, 3, 3, 129, 129),       # three items: as many as stages; a second kv tile of one row
    (1, 4, 1, 193, 300),       # kv rows past the last query
    (1, 9, 9, 257, 100),       # more heads than XCDs, queries past the last key
])
def test_softmax_backward_item_walk(cuda_device, B, H, Hkv, Sq, Skv, D, causal):
    """Ends of the walk over a kv tile's streamed items (few items, one tile a head, a ragged last tile, rows without a
    partner), which the dk/dv launch's two halves of a wave pair go through one tile apart.  _check's tolerance: p, ds
    and the results are rounded to the input type as at every other shape."""
    print(f"case bwd walk B{B} H{H} Hkv{Hkv} Sq{Sq} Skv{Skv} D{D} causal={causal}", flush=True)
    # (the oracle's own causal mask is square: over unequal lengths it is given the mask's grid)
    _run(B, H, Hkv, Sq, Skv, D, D, torch.float16, C.causal_mask if causal else None, causal and Sq == Skv)


@pytest.mark.parametrize("Sq,Skv,causal", [(1, 1, True), (33, 33, True), (64, 64, True), (65, 65, True), (95, 95, True), (129, 129, True),
                                           (1, 129, False), (31, 65, False), (32, 64, False), (33, 97, False), (63, 31, False), (96, 128, False)])
@pytest.mark.parametrize("Hkv,dtype", [(3, torch.bfloat16), (1, torch.float16)])
def test_dk_dv_at_the_edges_of_their_waves(cuda_device, Sq, Skv, causal, Hkv, dtype):
    """Head dim 128, softmax (AE_BWD_PAIRS): a wave holds 64 kv rows and takes 32 q rows, another 64 rows of dk or of dv: lengths
    around those, so that whole waves have no rows, or no q rows."""
    print(f"case dk dv edges Sq{Sq} Skv{Skv} causal={causal} Hkv{Hkv} {dtype}", flush=True)
    _run(2, 3, Hkv, Sq, Skv, 128, 128, dtype, C.causal_mask if causal else None, causal, seed=Sq)


def test_softmax_backward_headline_shape(cuda_device):
    """The shape bench.py times the backward on (B2 H32 S4096 D128 fp16, causal): every gradient finite,
    and dq, dk, dv of two (batch, head) slices -- which depend on that slice's tensors only -- against the
    oracle's closed-form gradients."""
    B, H, S, D = 2, 32, 4096, 128
    dtype = torch.float16
    scale = 1 / math.sqrt(D)
    q, k, v = C.make_inputs(B, S, S, H, H, D, D, dtype, seed=9)
    do = torch.randn(B, S, H, D, generator=torch.Generator().manual_seed(109)).to(dtype)
    mod = _engine(B, H, H, S, D, D, dtype, C.causal_mask, scale)
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    mod(qd, kd, vd).backward(do.cuda())
    for g in (qd.grad, kd.grad, vd.grad):
        assert torch.isfinite(g).all()
    for b, h in ((0, 0), (1, 31)):
        print(f"case backward at the headline shape: oracle on slice b{b} h{h}", flush=True)
        sl = (slice(b, b + 1), slice(None), slice(h, h + 1))
        dq, dk, dv = R.softmax_attention_grads(q[sl], k[sl], v[sl], do[sl], scale=scale, causal=True)
        _check(qd.grad[sl], dq, "dq", (b, h))
        _check(kd.grad[sl], dk, "dk", (b, h))
        _check(vd.grad[sl], dv, "dv", (b, h))


def test_softmax_backward_elementwise_mask_and_dv(cuda_device):
    """A mask that is not causal is applied per element (sliding window: rows see 37 keys), and the
    value head dim may differ from the key head dim."""
    print("case bwd sliding window", flush=True)
    _run(1, 2, 2, 300, 300, 128, 128, torch.float16, C.make_sliding_window_mask(37), False)
    print("case bwd D128 DV64", flush=True)
    _run(1, 2, 1, 256, 256, 128, 64, torch.float16, C.causal_mask, True)
    print("case bwd D64 DV128", flush=True)
    _run(2, 2, 2, 130, 130, 64, 128, torch.bfloat16, None, False)


def test_softmax_backward_skips_masked_tiles(cuda_device):
    """Masks that are not causal come with two tile-class tables (one per launch): tiles without a
    visible element are skipped, partly visible ones test mask_mod per element.  A narrow sliding window
    over a long sequence (most tiles skipped), a mask that depends on the head (one table per head), a
    shifted causal mask with grouped heads."""
    for name, mask_mod, H, Hkv, S in (("window", C.make_sliding_window_mask(100), 2, 2, 700),
                                      ("head", C.head_dependent_mask, 4, 4, 520),
                                      ("shifted", C.causal_shifted_mask, 4, 2, 333)):
        print(f"case bwd tile classes {name}", flush=True)
        _run(1, H, Hkv, S, S, 128, 128, torch.float16, mask_mod, False, seed=11)
        eng = _engine(1, H, Hkv, S, 128, 128, torch.float16, mask_mod, 1 / math.sqrt(128))
        assert eng._op._plan(1, H, S, S, None).mode == 2


def test_backward_tile_classes_of_a_long_sequence(cuda_device):
    """More than 64 streamed items per workgroup (68 q tiles of 64 rows for each of the two q heads of a kv
    head): the kernels read the tile classes 64 items at a time, so this crosses from one set to the next."""
    print("case bwd tile classes, 136 items per kv tile", flush=True)
    _run(1, 2, 1, 4352, 4352, 64, 64, torch.bfloat16, C.make_sliding_window_mask(300), False, seed=13)


def test_backward_odd_shapes_against_oracle(cuda_device):
    """Seeded sweep: ragged sequence lengths (also Sq != Skv without a mask), grouped heads, both head
    dims for keys and values, both dtypes, no mask / causal / sliding window / head-dependent masks."""
    import random
    rng = random.Random(2024)
    masks = [(None, False), (C.causal_mask, True), (C.make_sliding_window_mask(53), False),
             (C.head_dependent_mask, False)]
    for n in range(14):
        hkv = rng.choice([1, 2, 3])
        B, H = rng.choice([1, 2]), hkv * rng.choice([1, 2, 4])
        D, DV = rng.choice([64, 128]), rng.choice([64, 128])
        dtype = torch.float16 if n % 2 == 0 else torch.bfloat16
        mask_mod, causal = masks[n % len(masks)]
        Sq = rng.randint(1, 450)
        Skv = Sq if mask_mod is not None else rng.randint(1, 450)
        print(f"case bwd odd B{B} H{H} Hkv{hkv} Sq{Sq} Skv{Skv} D{D} DV{DV} {dtype} mask {n % len(masks)}", flush=True)
        _run(B, H, hkv, Sq, Skv, D, DV, dtype, mask_mod, causal, seed=300 + n)


def test_sigmoid_and_relu_backward(cuda_device):
    """Graphs whose online function does nothing (attn_script/sigmoidattn.py, reluattn.py): p = f(s),
    ds = dp f'(s) with f' from the symbolic derivative of the traced score_mod; the sigmoid's bias is a
    scalar CustomIO tensor.  Against the oracle's closed-form gradients."""
    g = torch.Generator().manual_seed(9)
    for kind, causal, B, H, Hkv, S, D, dtype in (("sigmoid", True, 1, 2, 2, 300, 128, torch.float16),
                                                 ("sigmoid", False, 2, 4, 2, 256, 64, torch.bfloat16),
                                                 ("relu", False, 1, 3, 3, 200, 64, torch.float16)):
        print(f"case bwd {kind} causal={causal} B{B} H{H} Hkv{Hkv} S{S} D{D} {dtype}", flush=True)
        scale = 1 / math.sqrt(D)
        q, k, v = C.make_inputs(B, S, S, H, Hkv, D, D, dtype, seed=21)
        do = torch.randn(B, S, H, D, generator=g).to(dtype)
        meta = (meta_tensor(B, H, S, D, dtype=dtype), meta_tensor(B, Hkv, S, D, dtype=dtype),
                meta_tensor(B, Hkv, S, D, dtype=dtype))
        if kind == "sigmoid":
            bias = torch.tensor([-math.log(S)], dtype=torch.float32)
            mod = AttentionEngine(meta, CustomIO({"softmax_bias": (1,)}), score_mod=C.make_sigmoid_score_mod(scale),
                                  mask_mod=C.causal_mask if causal else None, online_func=C.OnlineIdentity())
            extra, kw = (bias.cuda(),), dict(bias=bias.item(), causal=causal)
        else:
            mod = AttentionEngine(meta, CustomIO({}), score_mod=C.make_relu_score_mod(scale), mask_mod=None,
                                  online_func=C.OnlineIdentity())
            extra, kw = (), dict()
        qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
        out = mod(qd, kd, vd, *extra)
        out.backward(do.cuda())
        dq, dk, dv = R.elementwise_attention_grads(q, k, v, do, kind, scale=scale, **kw)
        case = (kind, causal, B, H, Hkv, S, D, dtype)
        _check(qd.grad, dq, "dq", case)
        _check(kd.grad, dk, "dk", case)
        _check(vd.grad, dv, "dv", case)


@pytest.mark.parametrize("B,H,Hkv,S,D,DV,dtype", [
    (1, 2, 2, 256, 64, 128, torch.float16),       # value head dim twice the key head dim, as in the script
    (2, 4, 2, 200, 128, 128, torch.bfloat16),     # ragged tiles, grouped heads, batch > 1 against a [1,H,S,S] mask
    (1, 3, 3, 448, 128, 64, torch.float16),
])
def test_retention_backward(cuda_device, B, H, Hkv, S, D, DV, dtype):
    """attn_script/retention.py with its forward() / backward() rules: the traced backward (the saved row
    scale r as a constant, the decay mask read per score and as the derivative of score_mod) against the
    oracle's closed form."""
    print(f"case retention backward B{B} H{H} Hkv{Hkv} S{S} D{D} DV{DV} {dtype}", flush=True)
    q, k, v = C.make_inputs(B, S, S, H, Hkv, D, DV, dtype, seed=21)
    q = (q.float() * (1 / D) ** 0.5).to(dtype)                       # bench_utils.py:1034-1036 of the reference
    g = torch.Generator().manual_seed(22)
    mask = (torch.rand(1, H, S, S, generator=g) * 1.5).tril().to(dtype).contiguous()
    do = torch.randn(B, S, H, DV, generator=g).to(dtype)
    meta = (meta_tensor(B, H, S, D, dtype=dtype), meta_tensor(B, Hkv, S, D, dtype=dtype),
            meta_tensor(B, Hkv, S, DV, dtype=dtype))
    mod = AttentionEngine(meta, C.retention_custom_inputs(), score_mod=C.retention_score_mod,
                          mask_mod=C.causal_mask, online_func=C.OnlineRetention(), mask_value="0")
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    out = mod(qd, kd, vd, mask.cuda())
    ref, r = R.retention_attention(q, k, v, mask)
    assert (r > 1.0).any() and (r == 1.0).any()
    assert (out.detach().float().cpu() - ref).abs().max().item() <= 2e-2
    out.backward(do.cuda())
    dq, dk, dv = R.retention_attention_grads(q, k, v, mask, do)
    case = (B, H, Hkv, S, D, DV, dtype)
    _check(qd.grad, dq, "dq", case)
    _check(kd.grad, dk, "dk", case)
    _check(vd.grad, dv, "dv", case)


@pytest.mark.parametrize("bm,bn,S,Hkv,dtype", [
    (128, 128, 1024, 3, torch.float16),    # attn_script/blocksparseattn.py's granularity: every backward tile lies in ONE block
    (128, 64, 512, 3, torch.float16),      # the geometry of the reference's tests/test_blockmask.py
    (32, 64, 640, 1, torch.bfloat16),      # finer than the backward's 64- and 128-row tiles: tiles straddle blocks of both
                                           # kinds and test every element against the mask; grouped heads
    (64, 128, 448, 3, torch.float16),      # ragged last tiles of both launches (448 = 3.5 x 128)
])
def test_backward_with_an_external_block_mask(cuda_device, bm, bn, S, Hkv, dtype):
    """attn_script/blocksparseattn.py with gradients (the reference's block-sparse backward,
    blockattn_tl.py:195-470): the user's int8 block mask [B,H,S/bm,S/bn] reaches the two backward launches as
    tile-class tables made from it on the GPU, and tiles that straddle visible and invisible blocks look every
    element up in the mask itself.  Against the oracle's gradients under the expanded dense mask; one q block
    row sees nothing at all (out 0, gradients 0)."""
    print(f"case bwd extern block mask {bm}x{bn} S{S} Hkv{Hkv} {dtype}", flush=True)
    B, H, D = 2, 3, 64
    scale = 1 / math.sqrt(D)
    g = torch.Generator().manual_seed(11)
    nq, nk = -(-S // bm), -(-S // bn)
    blocks = torch.rand(B, H, nq, nk, generator=g) < 0.45
    blocks[..., 0] = True                         # every row sees something ...
    blocks[0, 1, nq - 1] = False                  # ... except one block row of one head
    q, k, v = C.make_inputs(B, S, S, H, Hkv, D, D, dtype, seed=5)
    do = torch.randn(B, S, H, D, generator=g).to(dtype)
    meta = (meta_tensor(B, H, S, D, dtype=dtype), meta_tensor(B, Hkv, S, D, dtype=dtype),
            meta_tensor(B, Hkv, S, D, dtype=dtype))
    mod = AttentionEngine(meta, CustomIO({}), score_mod=C.make_scale_score_mod(scale), mask_mod=None,
                          online_func=C.OnlineSoftmax(), infer_mask=True, extern_block_mask=True,
                          infer_mask_block_M=bm, infer_mask_block_N=bn)
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    out = mod(qd, kd, vd, block_mask=blocks.to(torch.int8).cuda())
    out.backward(do.cuda())
    dense = blocks.repeat_interleave(bm, 2).repeat_interleave(bn, 3)[:, :, :S, :S]
    ref_out, _ = R.softmax_attention(q, k, v, scale=scale, mask=dense)
    assert (out.detach().float().cpu() - ref_out).abs().max().item() <= 2e-2
    dq, dk, dv = R.softmax_attention_grads(q, k, v, do, scale=scale, mask=dense)
    case = (bm, bn, S, Hkv, dtype)
    _check(qd.grad, dq, "dq", case)
    _check(kd.grad, dk, "dk", case)
    _check(vd.grad, dv, "dv", case)
    r0 = (nq - 1) * bm
    assert qd.grad[0, r0:, 1].abs().max().item() == 0.0          # the rows that see nothing
    # a second call with another mask: the tables follow the mask of the call
    blocks2 = torch.ones_like(blocks)
    qd.grad = kd.grad = vd.grad = None
    mod(qd, kd, vd, block_mask=blocks2.to(torch.int8).cuda()).backward(do.cuda())
    dq, dk, dv = R.softmax_attention_grads(q, k, v, do, scale=scale)
    _check(qd.grad, dq, "dq", case + ("all",))
    _check(kd.grad, dk, "dk", case + ("all",))


@pytest.mark.parametrize("mask_name", ["causal", "window", "plus_one", "head_dependent"])
def test_backward_masks_are_bit_exact(cuda_device, mask_name):
    """One-hot probes of the masks the two backward launches apply (tiles skipped by index or by their tile-class
    tables, elements tested where a tile is partly visible), at 4300 positions -- more than 64 streamed items per
    resident tile, so the tables are read in several chunks of ballots, ragged last tiles in both launches -- and
    two q heads per kv head.  Integers, compared exactly:
      * dk / dv launch: the graph out = sum_kv f(s) v with f = 1 on every finite score and 0 on a masked one;
        dO holds one-hot rows (q -> column q mod DV), so dv[kv, j] = dO^T p counts the queries of residue class j
        that see key kv (summed over the group's q heads);
      * dq launch: f(s) = s, so ds = dp on visible scores and 0 on masked ones; with v and dO all equal to the
        first unit vector dp = 1, and K one-hot rows make dq[q, j] = ds K count the visible keys of class j."""
    mask_mod = {"causal": C.causal_mask, "window": C.make_sliding_window_mask(100),
                "plus_one": C.causal_plus_one_mask, "head_dependent": C.head_dependent_mask}[mask_name]
    B, H, Hkv, S, D = 1, 2, 1, 4300, 64
    dtype = torch.float16
    print(f"case bwd mask probe {mask_name}", flush=True)
    dense = torch.from_numpy(M.dense_mask_grid(mask_mod, B, H, S, S)).float()        # [B,H,S,S]
    onehot = torch.zeros(S, D)
    onehot[torch.arange(S), torch.arange(S) % D] = 1.0
    meta = (meta_tensor(B, H, S, D, dtype=dtype), meta_tensor(B, Hkv, S, D, dtype=dtype),
            meta_tensor(B, Hkv, S, D, dtype=dtype))

    def ones_score_mod(score, custom_fwd_inputs, b, h, q_idx, kv_idx):
        return ((score * 0.001 + 50.0).tanh() + 1.0) * 0.5

    def plain_score_mod(score, custom_fwd_inputs, b, h, q_idx, kv_idx):
        return score * 1.0

    q, k, v = C.make_inputs(B, S, S, H, Hkv, D, D, dtype)
    # dk / dv launch
    mod = AttentionEngine(meta, CustomIO({}), score_mod=ones_score_mod, mask_mod=mask_mod, online_func=C.OnlineIdentity())
    bwd = mod._op.backward_op()
    assert bwd.kind == 1
    do = onehot.to(dtype).view(1, S, 1, D).expand(B, S, H, D).contiguous()
    out = torch.zeros(B, S, H, D, dtype=dtype)
    _, _, dv = bwd(q.cuda(), k.cuda(), v.cuda(), out.cuda(), None, do.cuda())
    expect = torch.einsum("bhqk,qd->bkd", dense, onehot).view(B, S, Hkv, D)
    assert expect.max().item() >= {"causal": 100, "plus_one": 100, "window": 4, "head_dependent": 5}[mask_name]
    assert torch.equal(dv.float().cpu(), expect), mask_name
    # dq launch
    mod = AttentionEngine(meta, CustomIO({}), score_mod=plain_score_mod, mask_mod=mask_mod, online_func=C.OnlineIdentity())
    bwd = mod._op.backward_op()
    e0 = torch.zeros(D, dtype=dtype)
    e0[0] = 1.0
    kk = onehot.to(dtype).view(1, S, 1, D).expand(B, S, Hkv, D).contiguous()
    vv = e0.view(1, 1, 1, D).expand(B, S, Hkv, D).contiguous()
    do = e0.view(1, 1, 1, D).expand(B, S, H, D).contiguous()
    dq, _, _ = bwd(q.cuda(), kk.cuda(), vv.cuda(), out.cuda(), None, do.cuda())
    expect = torch.einsum("bhqk,kd->bqhd", dense, onehot)
    assert torch.equal(dq.float().cpu(), expect), mask_name


@pytest.mark.parametrize("B,H,Hkv,S,D,dtype,causal", [
    (1, 2, 2, 256, 64, torch.float16, False),
    (2, 4, 2, 333, 128, torch.bfloat16, True),      # grouped heads, ragged tiles, causal
    (1, 3, 1, 200, 64, torch.float16, True),
])
def test_traced_backward_with_two_final_row_scales(cuda_device, B, H, Hkv, S, D, dtype, causal):
    """An online function with TWO final row scales whose forward() / backward() rules read both: the rules are
    traced (no fixed gradient applies), the backward launches carry both row scales per q row, and since the
    function is softmax attention written differently its gradients must be those of the oracle
    (softmax_attention_grads, pinned by float64 autograd).  The exported scales themselves: m + log r = lse."""
    print(f"case two row scales B{B} H{H} Hkv{Hkv} S{S} D{D} {dtype} causal={causal}", flush=True)
    scale = 1 / math.sqrt(D)
    q, k, v = C.make_inputs(B, S, S, H, Hkv, D, D, dtype, seed=13)
    do = torch.randn(B, S, H, D, generator=torch.Generator().manual_seed(113)).to(dtype)
    meta = (meta_tensor(B, H, S, D, dtype=dtype), meta_tensor(B, Hkv, S, D, dtype=dtype),
            meta_tensor(B, Hkv, S, D, dtype=dtype))
    mod = AttentionEngine(meta, CustomIO({}), score_mod=C.make_scale_score_mod(scale),
                          mask_mod=C.causal_mask if causal else None, online_func=OnlineSoftmaxTwoScales())
    bwd = mod._op.backward_op()
    assert bwd.kind == 2 and bwd.rowscale_names == ["m", "r"] and bwd.n_rs == 2
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    out = mod(qd, kd, vd)
    out.backward(do.cuda())
    ref_out, lse = R.softmax_attention(q, k, v, scale=scale, causal=causal)
    assert (out.detach().float().cpu() - ref_out).abs().max().item() <= 2e-2
    m, r = mod.final_rowscales["m"].cpu(), mod.final_rowscales["r"].cpu()
    assert (m + r.log() - lse).abs().max().item() <= 1e-3
    dq, dk, dv = R.softmax_attention_grads(q, k, v, do, scale=scale, causal=causal)
    case = (B, H, Hkv, S, D, dtype, causal)
    _check(qd.grad, dq, "dq", case)
    _check(kd.grad, dk, "dk", case)
    _check(vd.grad, dv, "dv", case)


@pytest.mark.parametrize("B,H,Hkv,S,D", [(2, 9, 3, 33, 64), (1, 17, 17, 31, 64), (3, 8, 8, 64, 64), (2, 5, 5, 65, 128), (1, 1, 1, 1, 64)])
def test_row_sums_at_the_edges_of_their_workgroups(cuda_device, B, H, Hkv, S, D):
    """ae_bwd_delta_kernel: 32 positions of 8 heads (D 64) or 4 a workgroup, heads and positions past the end among them."""
    test_traced_backward_with_two_final_row_scales(cuda_device, B, H, Hkv, S, D, torch.float16, True)


def test_backward_of_other_graphs_is_refused(cuda_device):
    """An online function that keeps row scales of its own but defines no forward() / backward() rules
    (here: the running sum of |s| without them) has no backward.  Its forward still runs on tensors that
    require gradients, with the result of the plain call; the missing rule is reported by .backward(), where the
    reference reports it."""
    B, H, S, D = 1, 2, 128, 64
    meta = (meta_tensor(B, H, S, D, dtype=torch.float16),) * 3
    mod = AttentionEngine(meta, CustomIO({}), score_mod=C.make_scale_score_mod(0.125), mask_mod=None,
                          online_func=C.OnlineAbsNorm())
    q, k, v = (t.cuda() for t in C.make_inputs(B, S, S, H, H, D, D, torch.float16))
    plain = mod(q, k, v)
    qg, kg, vg = (t.clone().requires_grad_(True) for t in (q, k, v))
    out = mod(qg, kg, vg)
    assert out.requires_grad and torch.equal(out.detach(), plain)
    with pytest.raises(NotImplementedError, match="no backward for this engine"):
        out.sum().backward()
    assert qg.grad is None


@pytest.mark.parametrize("B,H,Hkv,Sq,Skv,D,dtype,causal,parts", [
    (1, 8, 2, 333, 333, 128, torch.bfloat16, True, 3),      # ragged; the last kv tile has 4 heads x 2 items
    (2, 4, 1, 700, 700, 64, torch.float16, True, 6),
    (1, 2, 2, 130, 130, 128, torch.float16, True, 4),       # the second kv tile has one item: three parts without any
    (1, 4, 2, 200, 520, 64, torch.bfloat16, False, 2),      # no mask, unequal lengths
    (1, 4, 4, 65, 1, 128, torch.bfloat16, False, 2),        # one key
])
def test_backward_kv_tiles_shared_by_workgroups(cuda_device, monkeypatch, B, H, Hkv, Sq, Skv, D, dtype, causal, parts):
    """dk/dv launches that share a kv tile out (AE_BWD_SPLIT): gradients as the oracle's, the same bits on every call (the
    parts are added in their order, whoever finishes last) and on every replay of a graph, with eager calls in between."""
    scale = 1 / math.sqrt(D)
    print(f"case shared kv tiles B{B} H{H}/{Hkv} {Sq}x{Skv} D{D} {dtype} causal={causal} parts={parts}", flush=True)
    q, k, v = C.make_inputs(B, Sq, Skv, H, Hkv, D, D, dtype, seed=31)
    dout = torch.randn(B, Sq, H, D, generator=torch.Generator().manual_seed(32)).to(dtype)
    mod = _engine(B, H, Hkv, Sq, D, D, dtype, C.causal_mask if causal else None, scale)
    op = mod._op.backward_op()
    monkeypatch.setattr(op, "dkv_parts", lambda *a: parts)
    ref = R.softmax_attention_grads(q, k, v, dout, scale=scale, causal=causal)
    leaves = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    do = dout.cuda()

    def step():
        return torch.autograd.grad(mod(*leaves), leaves, do)
    first = step()                                   # through Python
    for got, want, what in zip(first, ref, ("dq", "dk", "dv")):
        _check(got, want, what, (B, H, Hkv, Sq, Skv, D, parts))
    for _ in range(3):                               # through the native host path
        assert all(torch.equal(a, b) for a, b in zip(step(), first))
    torch.cuda.synchronize()
    qd, kd, vd = (t.detach() for t in leaves)
    out, rs = mod.forward_with_rowscales(qd, kd, vd)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        grads = op(qd, kd, vd, out, rs["lse"], do)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(grads, first))
        step()


@pytest.mark.parametrize("S,rows", [(1000, 128), (6000, 256)])
def test_backward_rows_of_the_dq_launch_follow_the_problem(cuda_device, S, rows):
    """Few 256-row q tiles are halved; an engine whose caller chose keeps that choice."""
    B, H, D, dtype = 1, 16, 128, torch.bfloat16
    mod = _engine(B, H, H, S, D, D, dtype, C.causal_mask, 1 / math.sqrt(D))
    op = mod._op.backward_op()
    assert op.rows_of_dq(B, H, S, True, True) == rows
    from core.lower.prefill_bwd_op import PrefillBwdOp
    assert PrefillBwdOp(mod._op, *op._graph, dq_rows=256).rows_of_dq(B, H, S, True, True) == 256
    q, k, v = C.make_inputs(B, S, S, H, H, D, D, dtype, seed=5)
    dout = torch.randn(B, S, H, D, generator=torch.Generator().manual_seed(6)).to(dtype)
    leaves = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    got = torch.autograd.grad(mod(*leaves), leaves, dout.cuda())
    one = [t[:, :, 3:4] for t in (q, k, v, dout)]
    ref = R.softmax_attention_grads(*one, scale=1 / math.sqrt(D), causal=True)
    for g, want, what in zip(got, ref, ("dq", "dk", "dv")):
        _check(g[:, :, 3:4], want, what, (S, rows))


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,H,Hkv,Sq,Skv,dtype", [
    (1, 2, 2, 1, 1, torch.float16),
    (2, 3, 3, 64, 64, torch.bfloat16),
    (1, 4, 2, 65, 65, torch.float16),         # a q tile of one row; grouped heads
    (2, 2, 1, 129, 129, torch.bfloat16),      # a key tile of one key
    (1, 3, 3, 300, 300, torch.float16),       # two workgroups, the second's last waves without rows
    (1, 9, 3, 577, 577, torch.bfloat16),
    (1, 2, 2, 100, 300, torch.float16),       # unequal lengths: every block of ds exists
    (2, 2, 2, 390, 70, torch.bfloat16),
])
def test_backward_with_ds_kept_in_memory(cuda_device, monkeypatch, B, H, Hkv, Sq, Skv, dtype, causal):
    """AE_BWD_KEEP_DS and ae_bwd_dq.hip at sizes where the plan would not take them: against the oracle, and against the launches
    that form ds twice."""
    from core.lower.prefill_bwd_op import PrefillBwdOp
    print(f"case ds kept B{B} H{H} Hkv{Hkv} Sq{Sq} Skv{Skv} {dtype} causal={causal}", flush=True)
    D, scale = 128, 1 / math.sqrt(128)
    q, k, v = C.make_inputs(B, Sq, Skv, H, Hkv, D, D, dtype, seed=Sq)
    do = torch.randn(B, Sq, H, D, generator=torch.Generator().manual_seed(5)).to(dtype)
    monkeypatch.setattr(PrefillBwdOp, "dkv_parts", lambda self, *a: 1)
    grads = []
    for keep in (False, True):
        monkeypatch.setattr(PrefillBwdOp, "keeps_ds", lambda self, *a: keep and a[4] != 2)      # (unequal lengths: a mask table)
        mod = _engine(B, H, Hkv, Sq, D, D, dtype, C.causal_mask if causal else None, scale)
        for _ in range(2):                    # through Python, then through the native host path
            leaves = [t.cuda().requires_grad_(True) for t in (q, k, v)]
            mod(*leaves).backward(do.cuda())
        grads.append([t.grad.float().cpu() for t in leaves])
        assert any(key[-1] for key in mod.attention.backward_op()._variants) == (keep and (Sq == Skv or not causal))
    case = (B, H, Hkv, Sq, Skv, dtype, causal)
    ref = R.softmax_attention_grads(q, k, v, do, scale=scale, causal=causal)
    for got, want, what in zip(grads[1], ref, ("dq", "dk", "dv")):
        _check(got, want, what, case)
    # the row sums rowsum(do * o) come from another order of 128 fp32 terms: within e = 128 * 2^-24 sum |do o| of a row, which moves
    # its ds by p e (and perhaps to the next value of the input type), dq by scale e p |k| and dk by scale (p e)^T |q| at most;
    # dv does not use them
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    out, _ = R.softmax_attention(q, k, v, scale=scale, causal=causal)
    e = (128 * 2.0 ** -24 * (out * do.float()).abs().sum(-1)).transpose(1, 2)                   # [B, H, Sq]
    heads = [t.double().transpose(1, 2) for t in (q, k.repeat_interleave(H // Hkv, 2))]
    sc = heads[0] @ heads[1].transpose(-1, -2) * scale
    if causal:
        sc = sc.masked_fill(torch.arange(Sq)[:, None] < torch.arange(Skv)[None, :], float("-inf"))
    pe = torch.softmax(sc, -1).nan_to_num(0.0) * e.double()[..., None]
    moved = (scale * (pe @ heads[1].abs()), scale * (pe.transpose(-1, -2) @ heads[0].abs()).unflatten(1, (Hkv, H // Hkv)).sum(2))
    for got, want, by in zip(grads[1], grads[0], moved):
        assert (got - want).norm().item() <= eps * want.norm().item() + by.norm().item()
    assert torch.equal(grads[1][2], grads[0][2])


def test_when_ds_is_kept(cuda_device):
    """By the visible pairs and the size of its buffer; not for other graphs, masks by table or a caller's own dq rows."""
    op = _engine(4, 32, 32, 2048, 128, 128, torch.bfloat16, C.causal_mask, 0.1).attention
    bwd = op.backward_op()
    assert bwd.keeps_ds(4, 32, 2048, 2048, 1, False) and not bwd.keeps_ds(4, 32, 2048, 2048, 2, False)
    assert not bwd.keeps_ds(1, 32, 1024, 1024, 1, False) and not bwd.keeps_ds(64, 32, 8192, 8192, 1, False)
    # q tiles t of 64 rows see the 128-key tiles 0 .. t / 2
    assert bwd.ds_floats(1, 1, 300, 300, 1) == sum(t // 2 + 1 for t in range(5)) * 64 * 128 // 2
    assert bwd.ds_floats(2, 3, 300, 300, 0) == 6 * 5 * 3 * 64 * 128 // 2
    assert bwd.keeps_ds(1, 32, 8192, 8192, 1, False)
    op.work_limit = 100 << 20
    assert not bwd.keeps_ds(4, 32, 2048, 2048, 1, False)


def test_a_backward_keeps_no_work_buffer(cuda_device):
    """The first backward of a shape, through Python, and later native ones leave their gradients allocated and no more: not
    ds (71 MB here), nor the row sums, nor what they were called with."""
    B, H, S, D = 1, 16, 2048, 128
    mod = _engine(B, H, H, S, D, D, torch.bfloat16, C.causal_mask, 1 / math.sqrt(D))
    bwd = mod.attention.backward_op()
    bwd.dkv_parts = lambda *a: 1
    assert bwd.keeps_ds(B, H, S, S, 1, False)
    q, k, v = (t.cuda().requires_grad_(True) for t in C.make_inputs(B, S, S, H, H, D, D, torch.bfloat16, seed=9))
    for _ in range(3):
        out = mod(q, k, v)
        before = torch.cuda.memory_allocated()
        dout = torch.ones_like(out)
        grads = torch.autograd.grad(out, (q, k, v), dout)
        del dout
        kept = torch.cuda.memory_allocated() - before - sum(g.numel() * g.element_size() for g in grads)
        assert kept <= 0, kept
        del grads, out


@pytest.mark.gpu
def test_no_memory_for_ds(cuda_device, monkeypatch):
    """A backward whose ds cannot be had takes the two launches, as one that may not keep it does."""
    B, H, S = 1, 16, 2048
    q, k, v = (t.cuda().requires_grad_(True) for t in C.make_inputs(B, S, S, H, H, 128, 128, torch.bfloat16, seed=3))
    dout = torch.randn(B, S, H, 128, device="cuda", dtype=torch.bfloat16)
    grads = []
    for limit in (0, None):
        op = _engine(B, H, H, S, 128, 128, torch.bfloat16, C.causal_mask, 0.1).attention
        op.work_limit = limit
        bwd = op.backward_op()
        assert bwd.keeps_ds(B, H, S, S, 1, False) == (limit is None)
        bwd.dkv_parts = lambda *a: 1
        empty, refused = torch.empty, []

        def short(*a, **kw):
            if a and isinstance(a[0], int) and a[0] > 1 << 24:
                refused.append(a[0])
                raise torch.OutOfMemoryError("no memory")
            return empty(*a, **kw)
        monkeypatch.setattr(torch, "empty", short)
        grads.append(torch.autograd.grad(op(q, k, v), (q, k, v), dout))
        monkeypatch.setattr(torch, "empty", empty)
        assert len(refused) == (limit is None)
    assert all(torch.equal(a, b) for a, b in zip(*grads))
    # natively, from the second call of a shape on: the allocator may take less than ds (284 MB) needs
    S = 4096
    q, k, v = (t.cuda().requires_grad_(True) for t in C.make_inputs(B, S, S, H, H, 128, 128, torch.bfloat16, seed=4))
    dout = torch.randn(B, S, H, 128, device="cuda", dtype=torch.bfloat16)
    for limit in (0, None):
        op.work_limit = limit
        want = [torch.autograd.grad(op(q, k, v), (q, k, v), dout) for _ in range(2)]
        if limit == 0:
            grads = want[1]
    assert bwd.keeps_ds(B, H, S, S, 1, False) and not torch.equal(grads[0], want[1][0])
    del want
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (160 << 20)) / total)
    try:
        again = torch.autograd.grad(op(q, k, v), (q, k, v), dout)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert all(torch.equal(a, b) for a, b in zip(grads, again))


class _MemoryLeft:
    """Inside, torch's allocator has ``mib`` MiB beyond what it holds."""

    def __init__(self, mib):
        self.mib = mib

    def __enter__(self):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (self.mib << 20)) / total)

    def __exit__(self, *exc):
        torch.cuda.set_per_process_memory_fraction(1.0)


def _ds_engine(S, limit=None, B=1, H=16):
    mod = _engine(B, H, H, S, 128, 128, torch.bfloat16, C.causal_mask, 0.1)
    mod.attention.work_limit = limit
    bwd = mod.attention.backward_op()
    bwd.dkv_parts = lambda *a: 1
    assert bwd.keeps_ds(B, H, S, S, 1, False) == (limit is None)
    q, k, v = (t.cuda().requires_grad_(True) for t in C.make_inputs(B, S, S, H, H, 128, 128, torch.bfloat16, seed=4))
    dout = torch.randn(B, S, H, 128, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16).cuda()
    return mod, lambda: mod(q, k, v), lambda out: torch.autograd.grad(out, (q, k, v), dout)


def _same(a, b):
    return all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("natively", [False, True])
def test_memory_for_ds_but_not_for_the_gradients_beside_it(cuda_device, natively):
    """264 MiB of ds and 48 MiB of gradients where 290 are left: the launches that need no ds run, as they did before."""
    _, forward, backward = _ds_engine(4096, limit=0)
    two = backward(forward())
    _, forward, backward = _ds_engine(4096)
    if natively:
        assert not _same(backward(forward()), two)
    out = forward()
    with _MemoryLeft(290):
        got = backward(out)
    assert _same(got, two)


@pytest.mark.parametrize("natively", [False, True])
def test_a_refused_ds_is_asked_for_again(cuda_device, monkeypatch, natively):
    """A moment without memory does not leave a shape with the slower launches: after DS_RETRY calls ds is tried again."""
    from core.lower import prefill_bwd_op as B
    monkeypatch.setattr(B, "DS_RETRY", 2, raising=False)
    _, forward, backward = _ds_engine(4096, limit=0)
    two = backward(forward())
    _, forward, backward = _ds_engine(4096)
    if natively:
        backward(forward())
    out = forward()
    with _MemoryLeft(160):
        assert _same(backward(out), two)
    assert _same(backward(forward()), two) and _same(backward(forward()), two)
    kept = backward(forward())
    assert not _same(kept, two) and _same(kept, backward(forward()))
