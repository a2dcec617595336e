"""Prefill tiles whose waves share the kv axis (AE_KW of csrc/kernels/ae_prefill.hip): every tile shape of
core/lower/lower.py kv_group_tiles against the oracle, where groups run out of tiles, rows and keys end inside a tile,
and rows see nothing."""
import math

import pytest
import torch

import attn_cases as C
from attn_engine import AttentionEngine
from core import CustomIO, meta_tensor
from core.lower.lower import PrefillTiles, kv_group_tiles, kv_group_tiles_split
from core.lower.prefill_op import PrefillOp
from oracle import attention_ref as R
from oracle import masks as OM

TILES = [PrefillTiles(n_waves=1, kv_groups=4, block_n=32), PrefillTiles(n_waves=2, kv_groups=4, block_n=32),
         PrefillTiles(n_waves=2, kv_groups=2, block_n=32), PrefillTiles(kv_groups=2)]


def test_the_choice_follows_the_number_of_workgroups():
    assert kv_group_tiles(128, 128, 32, 8, 8, True) == TILES[0]
    assert kv_group_tiles(128, 128, 32, 333, 333, True) == TILES[1]
    assert kv_group_tiles(64, 64, 32, 333, 333, True) == TILES[0]
    assert kv_group_tiles(128, 128, 32, 1000, 1000, True) == TILES[2]
    assert kv_group_tiles(128, 128, 32, 1500, 1500, True) == TILES[3]
    assert kv_group_tiles(128, 128, 16, 1200, 1200, False) == TILES[3]
    assert kv_group_tiles(128, 128, 64, 4096, 4096, True) is None
    assert kv_group_tiles_split(32) == TILES[0] and kv_group_tiles_split(64) == TILES[2]
    assert kv_group_tiles_split(128) is None


@pytest.mark.gpu
@pytest.mark.parametrize("tiles", TILES, ids=lambda t: f"{t.block_m}x{t.kv_groups}x{t.block_n}")
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16)])
@pytest.mark.parametrize("mask", ["none", "causal", "window", "shifted"])
def test_kv_groups_against_the_oracle(cuda_device, tiles, D, dtype, mask):
    mod = {"none": None, "causal": C.causal_mask, "window": C.make_sliding_window_mask(50),
           "shifted": C.causal_shifted_mask}[mask]
    for B, H, Hkv, S in ((1, 2, 2, 1), (1, 2, 1, 31), (2, 2, 2, 65), (1, 4, 2, 129), (2, 3, 3, 300)):
        print(f"case kv groups {tiles.block_m}x{tiles.kv_groups}x{tiles.block_n} D{D} {mask} B{B} H{H} S{S}", flush=True)
        if mask == "shifted" and S <= 128:
            continue                                             # (nothing is visible)
        q, k, v = C.make_inputs(B, S, S, H, Hkv, D, D, dtype, seed=S)
        meta = (meta_tensor(B, H, S, D, dtype=dtype), meta_tensor(B, Hkv, S, D, dtype=dtype), meta_tensor(B, Hkv, S, D, dtype=dtype))
        op = PrefillOp(meta, CustomIO({}), C.make_scale_score_mod(1 / math.sqrt(D)), mod, C.OnlineSoftmax(), "-inf", tiles=tiles)
        assert op.tiles == tiles and "#define AE_KW " in op.source
        out = op(q.cuda(), k.cuda(), v.cuda()).float().cpu()
        lse = op.final_rowscales["lse"].cpu()
        vis = None if mod is None else torch.from_numpy(OM.dense_mask_grid(mod, B, H, S, S))
        ref, rlse = R.softmax_attention(q, k, v, causal=False, mask=vis)
        seen = torch.isfinite(rlse)
        assert (out - ref.nan_to_num(0.0)).abs().max().item() <= 2e-2
        assert torch.equal(torch.isfinite(lse), seen)
        assert (lse[seen] - rlse[seen]).abs().max().item() <= 1e-3
        assert (lse[~seen] == float("-inf")).all()


def test_the_choice_of_wide_key_launches():
    def choice(H, S, B=1):
        return kv_group_tiles(192, 128, B * H, S, S, True)
    assert choice(16, 485, 2) == choice(16, 1428) == TILES[1]
    assert choice(16, 343) == choice(16, 1014, 2) == choice(32, 899) == TILES[2]
    assert choice(16, 2979) == choice(32, 1514) == TILES[3]
    assert choice(16, 986, 3) is None and choice(128, 433) is None and choice(16, 5334) is None and choice(32, 262, 3) is None


def test_the_choice_of_windows_and_short_keys():
    """Windows at head dim 64: two groups while 128-row tiles do not fill the chip twice, then 64-key tiles unless the window is
    narrow; short unmasked calls at head dim 128: 32-key tiles where three workgroups a CU or less padding pay."""
    def window(B, S, w, D=64):
        return _engine(S, C.make_sliding_window_mask(w), H=16, Hkv=16, D=D, B=B)._op.tiles_for(B, 16, S, S)
    assert window(3, 755, 121) == TILES[2] and window(1, 6102, 655) == PrefillTiles()
    assert window(3, 2719, 133) == PrefillTiles(block_n=32) == window(3, 4096, 655, D=128)
    def full(B, H, S):
        return _engine(S, None, H=H, Hkv=H, B=B)._op.tiles_for(B, H, S, S)
    assert full(24, 32, 73) == full(21, 32, 216) == full(17, 8, 387) == PrefillTiles(block_n=32)
    assert full(5, 32, 1328) == full(16, 16, 256) == PrefillTiles()
    op = _engine(73, None, H=32, Hkv=32, B=24)._op
    assert op.tiles_for(16, 16, 256, 256) == PrefillTiles() and op.tiles_for(8, 32, 349, 349) == PrefillTiles(block_n=32)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,S", [(24, 32, 73), (17, 8, 387), (21, 32, 216)])
def test_short_unmasked_calls(cuda_device, B, H, S):
    """... computed with those tiles: the oracle's results on the first and the last (batch, head)."""
    D, dtype = 128, torch.bfloat16
    mod = _engine(S, None, H=H, Hkv=H, B=B)
    q, k, v = C.make_inputs(B, S, S, H, H, D, D, dtype, seed=S)
    out = mod(q.cuda(), k.cuda(), v.cuda()).float().cpu()
    for b, h in ((0, 0), (B - 1, H - 1)):
        ref, rlse = R.softmax_attention(*(t[b:b + 1, :, h:h + 1] for t in (q, k, v)), causal=False)
        assert (out[b:b + 1, :, h:h + 1] - ref).abs().max().item() <= 2e-2
        assert (mod.final_rowscales["lse"].cpu()[b, h] - rlse[0, 0]).abs().max().item() <= 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("tiles", TILES[1:], ids=lambda t: f"{t.block_m}x{t.kv_groups}x{t.block_n}")
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_kv_groups_of_wide_keys(cuda_device, tiles, dtype):
    """Head dims 192 / 128: one key, tiles and groups that end inside each other, more tiles than two per group."""
    D, DV = 192, 128
    for B, H, Hkv, S in ((1, 2, 2, 1), (1, 2, 1, 33), (2, 3, 3, 129), (1, 4, 2, 390), (1, 2, 2, 1000)):
        print(f"case wide key groups {tiles.block_m}x{tiles.kv_groups}x{tiles.block_n} B{B} H{H} S{S} {dtype}", flush=True)
        q, k, v = C.make_inputs(B, S, S, H, Hkv, D, DV, dtype, seed=S)
        meta = (meta_tensor(B, H, S, D, dtype=dtype), meta_tensor(B, Hkv, S, D, dtype=dtype), meta_tensor(B, Hkv, S, DV, dtype=dtype))
        op = PrefillOp(meta, CustomIO({}), C.make_scale_score_mod(1 / math.sqrt(D)), C.causal_mask, C.OnlineSoftmax(), "-inf",
                       tiles=tiles)
        assert op.tiles == tiles and "#define AE_KW " in op.source
        out = op(q.cuda(), k.cuda(), v.cuda()).float().cpu()
        ref, rlse = R.softmax_attention(q, k, v, causal=True)
        assert (out - ref).abs().max().item() <= 2e-2
        assert (op.final_rowscales["lse"].cpu() - rlse).abs().max().item() <= 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("Sq,Skv", [(1, 40), (1, 1000), (31, 129), (33, 700), (64, 2100)])
def test_kv_groups_of_split_launches(cuda_device, Sq, Skv):
    B, H, D, dtype = 1, 3, 128, torch.float16
    q, k, v = C.make_inputs(B, Sq, Skv, H, H, D, D, dtype, seed=7)
    meta = (meta_tensor(B, H, Sq, D, dtype=dtype), meta_tensor(B, H, Skv, D, dtype=dtype), meta_tensor(B, H, Skv, D, dtype=dtype))
    mod = AttentionEngine(meta, CustomIO({}), C.make_scale_score_mod(1 / math.sqrt(D)), None, C.OnlineSoftmax())
    assert mod._op.tiles == kv_group_tiles_split(Sq)
    out = mod(q.cuda(), k.cuda(), v.cuda()).float().cpu()
    ref, lse = R.softmax_attention(q, k, v, causal=False)
    assert (out - ref).abs().max().item() <= 2e-2
    assert (mod.final_rowscales["lse"].cpu() - lse).abs().max().item() <= 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 3, 65, 700), (2, 5, 127, 1000), (1, 2, 193, 2100), (1, 3, 256, 1030), (8, 16, 200, 500), (1, 1, 300, 2000)])
def test_partial_results_of_split_launches(cuda_device, B, H, Sq, Skv, D):
    """Rows that end inside a wave, a wave without rows, 256-row workgroups (two passes over the columns), a row's columns
    of 64 and 128; through Python, then natively."""
    dtype = torch.float16
    print(f"case partial results B{B} H{H} {Sq}x{Skv} D{D}", flush=True)
    q, k, v = C.make_inputs(B, Sq, Skv, H, H, D, D, dtype, seed=9)
    meta = (meta_tensor(B, H, Sq, D, dtype=dtype), meta_tensor(B, H, Skv, D, dtype=dtype), meta_tensor(B, H, Skv, D, dtype=dtype))
    mod = AttentionEngine(meta, CustomIO({}), C.make_scale_score_mod(1 / math.sqrt(D)), None, C.OnlineSoftmax())
    assert mod._op.tiles.block_m == (256 if 192 < Sq <= 256 and B * H <= 64 else 128)
    assert mod._op.tiles_for(B, H, 100, Skv) == PrefillTiles()
    ref, lse = R.softmax_attention(q, k, v, causal=False)
    for _ in range(2):
        out = mod(q.cuda(), k.cuda(), v.cuda()).float().cpu()
        assert (out - ref).abs().max().item() <= 2e-2
        assert (mod.final_rowscales["lse"].cpu() - lse).abs().max().item() <= 1e-3


@pytest.mark.gpu
def test_kv_groups_of_graphs_without_row_state(cuda_device):
    B, H, S, D, dtype = 1, 2, 200, 64, torch.float16
    q, k, v = C.make_inputs(B, S, S, H, H, D, D, dtype, seed=3)
    meta = (meta_tensor(B, H, S, D, dtype=dtype),) * 3
    mod = AttentionEngine(meta, CustomIO({"softmax_bias": (1,)}), C.make_sigmoid_score_mod(1 / math.sqrt(D)), None,
                          C.OnlineIdentity())
    assert mod._op.tiles.kv_groups == 4
    out = mod(q.cuda(), k.cuda(), v.cuda(), torch.tensor([-2.0], device="cuda"))
    ref = R.sigmoid_attention(q, k, v, bias=-2.0)
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2


@pytest.mark.gpu
@pytest.mark.parametrize("tiles", TILES, ids=lambda t: f"{t.block_m}x{t.kv_groups}x{t.block_n}")
@pytest.mark.parametrize("what", ["key", "tile", "value", "infinite_key"])
@pytest.mark.parametrize("causal", [False, True])
def test_a_nan_reaches_every_row_that_sees_it(cuda_device, tiles, what, causal):
    """... also where it is all that a kv group sees of a row; rows that do not see it are as without it.  (An infinite
    score makes its row NaN: inf - inf.)"""
    B, H, S, D, dtype = 1, 2, 200, 64, torch.float16
    print(f"case nan {tiles.block_m}x{tiles.kv_groups}x{tiles.block_n} {what} causal={causal}", flush=True)
    q, k, v = C.make_inputs(B, S, S, H, H, D, D, dtype, seed=13)
    q = q.abs() + 2 ** -6                                         # (an infinite key scores +inf with every row)
    meta = (meta_tensor(B, H, S, D, dtype=dtype),) * 3
    op = PrefillOp(meta, CustomIO({}), C.make_scale_score_mod(1 / math.sqrt(D)), C.causal_mask if causal else None,
                   C.OnlineSoftmax(), "-inf", tiles=tiles)
    ref, _ = R.softmax_attention(q, k, v, causal=causal)
    lo, hi = (64, 96) if what == "tile" else (70, 71)
    bad = (v if what == "value" else k).clone()
    bad[:, lo:hi] = math.nan if what != "infinite_key" else 0.0
    if what == "infinite_key":
        bad[:, lo:hi, :, 0] = math.inf
    out = op(q.cuda(), (k if what == "value" else bad).cuda(), (bad if what == "value" else v).cuda()).float().cpu()
    sees = torch.arange(S) >= lo if causal else torch.ones(S, dtype=torch.bool)
    assert torch.isnan(out[:, sees]).all()
    if causal and what != "value":                                # (0 * NaN: a masked key's value still spoils its tile)
        assert (out[:, ~sees] - ref[:, ~sees]).abs().max().item() <= 2e-2


def _engine(S, mask, split=False, H=32, Hkv=8, D=128, B=1, Skv=None, dtype=torch.bfloat16):
    meta = (meta_tensor(B, H, S, D, dtype=dtype),) + (meta_tensor(B, Hkv, Skv or S, D, dtype=dtype),) * 2
    return AttentionEngine(meta, CustomIO({}), C.make_scale_score_mod(1 / math.sqrt(D)), mask, C.OnlineSoftmax())


def test_the_tiles_follow_the_shape_of_the_call():
    """An engine declared for a short prompt keeps nothing of it at other lengths; one declared large does not change."""
    op = _engine(333, C.causal_mask)._op
    assert op.tiles == TILES[1] and op.tiles_for(1, 32, 333, 333) == TILES[1]
    assert op.tiles_for(1, 32, 4096, 4096) == PrefillTiles() == op.tiles_for(8, 32, 333, 333)
    assert op.tiles_for(1, 32, 1000, 1000) == kv_group_tiles(128, 128, 32, 1000, 1000, True) == TILES[2]
    assert op._plan(1, 32, 4096, 4096, None).block_m == 128 and op.tiles == TILES[1]
    # no table reaches the tiles that share the kv axis: a mask that is a band at the declared length only
    odd = _engine(333, lambda b, h, q, kv: (q >= kv) & ((q < 400) | (kv % 2 == 0)))._op
    assert odd.tiles == TILES[1] and odd.tiles_for(1, 32, 500, 500) == PrefillTiles()
    large = _engine(4096, C.causal_mask, H=16)._op
    assert large.tiles.kv_groups == 1 and large.tiles_for(1, 16, 100, 100) == large.tiles
    few = _engine(8, None, H=8, Hkv=8, Skv=4096)._op
    assert few.split_kv and few.tiles == TILES[0] and few.tiles_for(1, 8, 64, 4096) == TILES[2]
    assert few.tiles_for(1, 8, 128, 4096) == PrefillTiles() and few.plan_splits(1, 8, 128, 4096)[1] % 64 == 0


@pytest.mark.gpu
def test_an_engine_for_short_prompts_at_other_lengths(cuda_device):
    H, Hkv, D = 32, 8, 128
    mod = _engine(333, C.causal_mask)
    op = mod._op

    def check(S, B=1):
        print(f"case B{B} S{S}", flush=True)
        q, k, v = C.make_inputs(B, S, S, H, Hkv, D, D, torch.bfloat16, seed=S)
        ref, rlse = R.softmax_attention(q, k, v, causal=True)
        for _ in range(2):                       # through Python, then natively
            out = mod(q.cuda(), k.cuda(), v.cuda()).float().cpu()
            assert (out - ref).abs().max().item() <= 2e-2
            assert (mod.final_rowscales["lse"].cpu() - rlse).abs().max().item() <= 1e-3
    for S, B in ((333, 1), (1100, 1), (333, 4), (70, 1), (333, 1)):
        check(S, B)
    built = {src.count("#define AE_KW ") for _, _, src in op._variants.values()}
    assert built == {0, 1} and op.tiles == TILES[1]
    # a block mask of the caller's, once: it takes the tiles that read tables, the declared shape keeps its own
    q, k, v = C.make_inputs(1, 333, 333, H, Hkv, D, D, torch.bfloat16, seed=1)
    blocks = torch.zeros(1, 1, 3, 3, dtype=torch.int8)
    blocks[..., 0] = 1
    out = mod(q.cuda(), k.cuda(), v.cuda(), blocks.cuda()).float().cpu()
    ref, _ = R.softmax_attention(q, k, v, causal=False, mask=torch.from_numpy(
        OM.dense_mask_grid(lambda b, h, qi, ki: (qi >= ki) & (ki < 128), 1, H, 333, 333)))
    assert (out - ref).abs().max().item() <= 2e-2
    assert op.tiles == TILES[1]
    check(333)


def test_split_launches_take_the_cheapest_tiles():
    """Head dim 128: tiles and splits of a launch by one cost, splits that cover the cache with none empty; other engines
    and launches that fill the chip keep the tiles they had."""
    op = _engine(8, None, H=8, Hkv=8, Skv=4096)._op
    for B, H in ((1, 8), (3, 16), (7, 32), (40, 32)):
        for Sq in (1, 32, 33, 64, 65, 128, 129, 256, 257):
            for Skv in (1, 31, 33, 522, 16001):
                own = op.tiles_for(B, H, Sq, Skv)
                tiles = op._launch_tiles(B, H, Sq, Skv, own)
                n, per = op.plan_splits(B, H, Sq, Skv, tiles)
                assert per % tiles.block_n == 0 and n * per >= Skv > (n - 1) * per
                assert tiles.lds_bytes(128, 128) <= 160 * 1024
                assert (Sq <= 256 and (Sq <= 64 or B * H <= 256)) or tiles == own
    three = [PrefillTiles(**f[0]) for f in op.SPLIT_FORMS.values()]
    assert op._launch_tiles(1, 8, 8, 4096, None) == three[0] and op._launch_tiles(1, 8, 64, 4096, None) == three[1]
    assert op._launch_tiles(1, 32, 128, 8192, None) == three[2] and op._launch_tiles(5, 32, 216, 3498, None) == three[3]
    assert op._launch_tiles(8, 8, 115, 521, None) == three[1]                    # 128 workgroups, not three splits of 64
    # short caches, and more heads than CUs: the engine's own tiles, unsplit; a long cache that one split reads best
    for B, Sq, Skv, tiles in ((3, 30, 704, TILES[0]), (3, 37, 651, TILES[2]), (9, 61, 521, TILES[2]), (16, 40, 2000, TILES[2]),
                              (5, 61, 15254, three[1]), (5, 45, 500, three[1]), (3, 30, 1100, three[0]), (9, 61, 8000, three[1])):
        got = op._launch_tiles(B, 32, Sq, Skv, op.tiles_for(B, 32, Sq, Skv))
        assert got == tiles, (B, Sq, Skv, got)
        if (B, Skv) != (9, 8000) and Skv != 1100:
            assert op.plan_splits(B, 32, Sq, Skv, got)[0] == 1, (B, Sq, Skv)
    narrow = _engine(8, None, H=8, Hkv=8, Skv=4096, D=64)._op
    assert narrow._launch_tiles(1, 8, 8, 4096, TILES[0]) == TILES[0]


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["32", "64", "128", "256"])
@pytest.mark.parametrize("Sq", [1, 33, 128, 150])
def test_three_tile_stages(cuda_device, form, Sq):
    """AE_KV_STAGES 3: none to seven tiles of a kv group, ragged last tiles, with and without a split; through Python, then
    natively."""
    B, H, D, dtype = 2, 3, 128, torch.float16
    for Skv, n in ((1, 1), (31, 1), (33, 1), (64, 1), (65, 2), (129, 1), (200, 1), (300, 2), (449, 1), (700, 3)):
        print(f"case three stages {form} Sq{Sq} Skv{Skv} splits {n}", flush=True)
        q, k, v = C.make_inputs(B, Sq, Skv, H, H, D, D, dtype, seed=Skv)
        op = _engine(Sq, None, H=H, Hkv=H, B=B, Skv=4096, dtype=dtype)._op
        assert op.split_kv
        tiles = PrefillTiles(**op.SPLIT_FORMS[form][0])
        op._launch_tiles = lambda *a: tiles
        op.plan_splits = lambda *a: (n, -(-Skv // (64 * n)) * 64)
        ref, lse = R.softmax_attention(q, k, v, causal=False)
        for _ in range(2):
            out = op(q.cuda(), k.cuda(), v.cuda()).float().cpu()
            assert (out - ref).abs().max().item() <= 2e-2
            assert (op.final_rowscales["lse"].cpu() - lse).abs().max().item() <= 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form,Sq", [("32", 5), ("32", 32), ("64", 61), ("64", 200)])
def test_the_first_tile_leaves_no_rounding_of_weights(cuda_device, form, Sq, dtype):
    """AE_FIRST_REST: where only the first 32 keys count, the result is as good as its own rounding, at every edge of the cache;
    with one split and with two."""
    B, H, D = 2, 3, 128
    for Skv, n in ((31, 1), (32, 1), (300, 1), (700, 2)):
        print(f"case first tile {form} Sq{Sq} Skv{Skv} splits {n} {dtype}", flush=True)
        q, k, v = C.make_inputs(B, Sq, Skv, H, H, D, D, dtype, seed=Skv + Sq)
        q[..., 0] = 40.0
        k[..., 0] = 0.0
        k[:, 32:, :, 0] = -20.0                       # 70 nats below
        op = _engine(Sq, None, H=H, Hkv=H, B=B, Skv=4096, dtype=dtype)._op
        tiles = PrefillTiles(**op.SPLIT_FORMS[form][0])
        op._launch_tiles = lambda *a: tiles
        op.plan_splits = lambda *a: (n, -(-Skv // (64 * n)) * 64)
        p = torch.softmax(torch.einsum("bqhd,bkhd->bhqk", q.double(), k.double()) / math.sqrt(D), -1)
        ref = torch.einsum("bhqk,bkhd->bqhd", p, v.double())
        # u = 2^-8 or 2^-11 (8 or 11 significant bits): the result's rounding is within u |result|, a weight's and then its rest's
        # within u^2 of it, and the weights sum to 1; 2^-18 for fp32 scores of at most 2^4, exponentials and sums
        u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        bound = u * ref.abs() + (u * u + 2.0 ** -18) * v.abs().max().item()
        for _ in range(2):
            err = (op(q.cuda(), k.cuda(), v.cuda()).cpu().double() - ref).abs()
            assert (err <= bound).all(), (err - bound).max().item()


def test_which_split_launches_merge_in_their_last_workgroup():
    op = _engine(8, None, H=8, Hkv=8, Skv=4096)._op
    forms = {n: PrefillTiles(**f[0]) for n, f in op.SPLIT_FORMS.items()}
    assert op._merges_in_last(8, 8, forms["32"], 8) and op._merges_in_last(8, 32, forms["32"], 2)
    assert not op._merges_in_last(8, 9, forms["32"], 8) and not op._merges_in_last(8, 1, forms["32"], 9)
    assert not op._merges_in_last(8, 8, forms["32"], 1) and not op._merges_in_last(8, 8, forms["64"], 2)
    assert not op._merges_in_last(1 << 14, 8, forms["32"], 8)                    # 2 GiB between a tile's results
    op._merges.any_order = False                                                  # (another combine() counts its places)
    assert not op._merges_in_last(8, 8, forms["32"], 8)


@pytest.mark.gpu
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16)])
@pytest.mark.parametrize("Sq,n", [(1, 2), (1, 8), (3, 5), (4, 8), (5, 7), (8, 8), (16, 4), (17, 3), (21, 3), (32, 2)])
def test_the_last_workgroup_merges(cuda_device, D, dtype, Sq, n):
    """AE_MERGE_LAST against the same splits merged by a second launch, bit for bit: passes that the rows fill, exceed by one
    and do not fill, every capacity; on two streams in turn, and in a graph (two launches again) between eager calls."""
    H, Skv, B = 3, 64 * n - 5, 2
    tiles = TILES[0] if D == 64 else PrefillTiles(**PrefillOp.SPLIT_FORMS["32"][0])
    print(f"case last workgroup merges D{D} Sq{Sq} splits {n}", flush=True)
    q, k, v = (t.cuda() for t in C.make_inputs(B, Sq, Skv, H, H, D, D, dtype, seed=Sq * 8 + n))
    ops = []
    for most in (0, 8192):
        op = _engine(Sq, None, H=H, Hkv=H, B=B, Skv=4096, D=D, dtype=dtype)._op
        op.MERGED_VALUES = most
        op._launch_tiles = lambda *a: tiles
        op.plan_splits = lambda *a: (n, 64)
        assert op.split_kv and op._merges_in_last(H, Sq, tiles, n) == (most > 0)
        ops.append(op)
    two = ops[0](q, k, v).float()
    two_lse = ops[0].final_rowscales["lse"]

    def check(out, lse):
        assert torch.equal(out.float(), two) and torch.equal(lse, two_lse)

    ref, rlse = R.softmax_attention(q.cpu(), k.cpu(), v.cpu(), causal=False)
    assert (two.cpu() - ref).abs().max().item() <= 2e-2 and (two_lse.cpu() - rlse).abs().max().item() <= 1e-3
    streams = [torch.cuda.current_stream(), torch.cuda.Stream()]
    for i in range(6):                                                # through Python, then natively; two streams in turn
        s = streams[i % 2]
        s.wait_stream(streams[1 - i % 2])
        with torch.cuda.stream(s):
            out = ops[1](q, k, v)
            lse = ops[1].final_rowscales["lse"]
        s.synchronize()
        check(out, lse)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops[1](q, k, v)
        lse = ops[1].final_rowscales["lse"]
    for _ in range(3):
        out.zero_(), lse.zero_()
        graph.replay()
        check(ops[1](q, k, v), ops[1].final_rowscales["lse"])
        torch.cuda.synchronize()
        check(out, lse)
