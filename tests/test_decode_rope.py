"""Decode attention that rotates, norms and writes the cache itself, against the kernel that does so first: the same pages,
outputs within the rounding of one bfloat16 query; at block and page edges, with and without each option."""
import pytest
import torch

from test_kernels import DEV, PagedKV, ops, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,hd,ps", [(5, 1, 64, 32), (8, 2, 128, 64), (40, 8, 128, 64), (16, 1, 128, 32)])
@pytest.mark.parametrize("rope,norm,temp", [(True, True, False), (False, False, True), (True, False, True), (False, True, False)])
@pytest.mark.parametrize("n_splits", [1, 3])
def test_against_the_two_kernels(H, G, hd, ps, rope, norm, temp, n_splits):
    lens = [1, 32, 33, 64, 300, 161]
    T = len(lens)
    kv = PagedKV(lens, G, hd, ps, torch.bfloat16)
    kp, vp = ops().kv_operand_order(kv.kp.to(DEV), kv.vp.to(DEV))
    qkv = rnd(T, (H + 2 * G) * hd, dtype=torch.bfloat16, seed=4)
    positions = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV)
    slots = torch.tensor([kv.tables[s][(n - 1) // ps] * ps + (n - 1) % ps for s, n in enumerate(lens)], dtype=torch.int32, device=DEV)
    seq, bt = torch.arange(T, dtype=torch.int32, device=DEV), kv.bt.to(DEV)
    inv = (10000.0 ** (-torch.arange(hd // 2, dtype=torch.float64) / (hd // 2))).float().to(DEV)
    scratch = torch.empty(ops().attn_decode_workspace(T, H, hd, n_splits) // 4, dtype=torch.float32, device=DEV)
    q, want, got = (torch.zeros(T, H * hd, dtype=torch.bfloat16, device=DEV) for _ in range(3))
    kp2, vp2 = kp.clone(), vp.clone()
    ops().rope_kvwrite(qkv, q, kp, vp, positions, slots, inv, H, G, hd, ps, use_rope=rope, adjacent=False, use_norm=norm, norm_eps=1e-5,
                       use_temp=temp, floor_scale=16, attn_scale=0.1, kv_tiled=True)
    args = (positions, seq, bt, T, H, G, hd, ps, "full", 0, hd ** -0.5, n_splits)
    ops().attn_decode(q, kp, vp, want, scratch, *args)
    ops().attn_decode_rope(qkv, kp2, vp2, got, scratch, positions, slots, *args[1:], inv_freq=inv if rope else None,
                           norm_eps=1e-5 if norm else 0.0, temperature=(16, 0.1) if temp else None)
    assert torch.equal(vp, vp2)
    # the sum of squares runs in another order: now and then an element rounds to the next bfloat16 (2^-8 apart at most)
    off = (kp.float() - kp2.float()).abs()
    assert float((off / kp.float().abs().clamp_min(1e-3)).max()) <= 2 ** -7 and float((off > 0).float().mean()) < 1e-3
    # a query or key element that rounds the other way moves a score by 2^-8 of one of hd products; the output rounds once more
    assert (got.float() - want.float()).abs().max() <= 1.5e-2 * max(1.0, float(want.float().abs().max()))


def test_refuses_what_it_cannot_do():
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=DEV)
    i32 = lambda *s: torch.zeros(*s, dtype=torch.int32, device=DEV)
    f = torch.zeros(4096, device=DEV)
    with pytest.raises(ops().KernelError):          # a head size that the kernel does not have
        ops().attn_decode_rope(z(1, 6 * 32), z(1, 1, 32, 32), z(1, 1, 32, 32), z(1, 4 * 32), f, i32(1), i32(1), i32(1), i32(1, 4), 1, 4, 1, 32,
                               32, "full", 0, 1.0, 1)
    with pytest.raises(ops().KernelError):          # no cache row
        ops().attn_decode_rope(z(1, 6 * 64), z(1, 1, 32, 64), z(1, 1, 64, 32), z(1, 4 * 64), f, i32(1), i32(0), i32(1), i32(1, 4), 1, 4, 1, 64,
                               32, "full", 0, 1.0, 1)


@pytest.mark.parametrize("vis,span", [("full", 0), ("chunk", 64), ("window", 45), ("window", 1)])
@pytest.mark.parametrize("softcap,sloped", [(0.0, False), (4.0, False), (0.0, True), (3.0, True)])
@pytest.mark.parametrize("n_splits", [1, 2, 13])
@pytest.mark.parametrize("hd", [64, 128])
def test_what_a_query_sees_caps_slopes_and_rows_without_a_place(vis, span, softcap, sloped, n_splits, hd):
    """Queries that open a chunk or a block, windows whose first key lies inside a block, more splits than blocks (the one
    that holds the last block writes the row), and a token without a cache row, which leaves the pages alone."""
    lens, H, G, ps = [1, 32, 33, 65, 64, 300, 129, 97], 6, 2, 32
    T = len(lens)
    kv = PagedKV(lens, G, hd, ps, torch.bfloat16)
    kp, vp = ops().kv_operand_order(kv.kp.to(DEV), kv.vp.to(DEV))
    before = kp.clone(), vp.clone()
    qkv = rnd(T, (H + 2 * G) * hd, dtype=torch.bfloat16, seed=9)
    positions = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV)
    slots = torch.tensor([kv.tables[s][(n - 1) // ps] * ps + (n - 1) % ps for s, n in enumerate(lens)], dtype=torch.int32, device=DEV)
    slots[5] = -1
    seq, bt = torch.arange(T, dtype=torch.int32, device=DEV), kv.bt.to(DEV)
    inv = (10000.0 ** (-torch.arange(hd // 2, dtype=torch.float64) / (hd // 2))).float().to(DEV)
    slopes = (0.02 * (1 + torch.arange(H))).float().to(DEV) if sloped else None
    scratch = torch.empty(ops().attn_decode_workspace(T, H, hd, n_splits) // 4, dtype=torch.float32, device=DEV)
    q, want, got = (torch.zeros(T, H * hd, dtype=torch.bfloat16, device=DEV) for _ in range(3))
    kp2, vp2 = kp.clone(), vp.clone()
    ops().rope_kvwrite(qkv, q, kp, vp, positions, slots, inv, H, G, hd, ps, use_rope=True, adjacent=False, use_norm=False, norm_eps=0.0,
                       use_temp=False, floor_scale=0, attn_scale=0.0, kv_tiled=True)
    args = (positions, seq, bt, T, H, G, hd, ps, vis, span, hd ** -0.5, n_splits)
    ops().attn_decode(q, kp, vp, want, scratch, *args, softcap=softcap, slopes=slopes)
    ops().attn_decode_rope(qkv, kp2, vp2, got, scratch, positions, slots, *args[1:], inv_freq=inv, softcap=softcap, slopes=slopes)
    assert torch.equal(kp, kp2) and torch.equal(vp, vp2)         # (without a norm: no sum whose order could differ)
    page = kv.tables[5][299 // ps]
    assert torch.equal(kp2[page], before[0][page]) and torch.equal(vp2[page], before[1][page])
    assert not torch.equal(kp2, before[0])
    assert torch.equal(got, want)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("n_splits", [1, 2, 9, 17, 40])
def test_own_key_at_every_place_of_a_block_and_any_number_of_splits(hd, n_splits):
    """The token's own key and value never pass through memory on their way to the scores: a token at each of the 32 places of a
    block gives what the two kernels give, bit for bit (without a norm the query is the same), behind one block and behind
    two; the pages keep NaN where no key has been written; the splits' records are joined 8, 16 or 32 at a time."""
    lens, H, G, ps = list(range(1, 65)), 6, 2, 32
    T = len(lens)
    kv = PagedKV(lens, G, hd, ps, torch.bfloat16)
    kv.vp[kv.vp == -70.0] = float("nan")
    kp, vp = ops().kv_operand_order(kv.kp.to(DEV), kv.vp.to(DEV))
    qkv = rnd(T, (H + 2 * G) * hd, dtype=torch.bfloat16, seed=11)
    positions = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV)
    slots = torch.tensor([kv.tables[s][(n - 1) // ps] * ps + (n - 1) % ps for s, n in enumerate(lens)], dtype=torch.int32, device=DEV)
    seq, bt = torch.arange(T, dtype=torch.int32, device=DEV), kv.bt.to(DEV)
    inv = (10000.0 ** (-torch.arange(hd // 2, dtype=torch.float64) / (hd // 2))).float().to(DEV)
    scratch = torch.empty(ops().attn_decode_workspace(T, H, hd, n_splits) // 4, dtype=torch.float32, device=DEV)
    q, want, got = (torch.zeros(T, H * hd, dtype=torch.bfloat16, device=DEV) for _ in range(3))
    kp2, vp2 = kp.clone(), vp.clone()
    ops().rope_kvwrite(qkv, q, kp, vp, positions, slots, inv, H, G, hd, ps, use_rope=True, adjacent=False, use_norm=False, norm_eps=0.0,
                       use_temp=False, floor_scale=0, attn_scale=0.0, kv_tiled=True)
    args = (positions, seq, bt, T, H, G, hd, ps, "full", 0, hd ** -0.5, n_splits)
    ops().attn_decode(q, kp, vp, want, scratch, *args)
    ops().attn_decode_rope(qkv, kp2, vp2, got, scratch, positions, slots, *args[1:], inv_freq=inv)
    bits = lambda t: t.view(torch.int16)
    assert torch.equal(bits(kp), bits(kp2)) and torch.equal(bits(vp), bits(vp2))
    assert torch.equal(bits(got), bits(want)) and bool(torch.isfinite(want.float()).all())


@pytest.mark.parametrize("H,G,hd", [(4, 4, 64), (4, 4, 128), (16, 1, 128)])
@pytest.mark.parametrize("vis,span", [("full", 0), ("window", 40), ("chunk", 48)])
@pytest.mark.parametrize("n_splits", [1, 3, 64])
def test_waves_and_splits_without_a_block(H, G, hd, vis, span, n_splits):
    """One to sixteen query heads a kv head (the records' room), contexts of one block and of five, splits that have none: the two
    kernels' bits, and pages whose other places hold NaN."""
    lens, ps = [1, 2, 31, 32, 33, 64, 65, 97, 129, 160], 64
    T = len(lens)
    kv = PagedKV(lens, G, hd, ps, torch.bfloat16)
    kv.vp[kv.vp == -70.0] = float("nan")
    kp, vp = ops().kv_operand_order(kv.kp.to(DEV), kv.vp.to(DEV))
    qkv = rnd(T, (H + 2 * G) * hd, dtype=torch.bfloat16, seed=5)
    positions = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV)
    slots = torch.tensor([kv.tables[s][(n - 1) // ps] * ps + (n - 1) % ps for s, n in enumerate(lens)], dtype=torch.int32, device=DEV)
    seq, bt = torch.arange(T, dtype=torch.int32, device=DEV), kv.bt.to(DEV)
    scratch = torch.empty(ops().attn_decode_workspace(T, H, hd, n_splits) // 4, dtype=torch.float32, device=DEV)
    q, want, got = (torch.zeros(T, H * hd, dtype=torch.bfloat16, device=DEV) for _ in range(3))
    kp2, vp2 = kp.clone(), vp.clone()
    ops().rope_kvwrite(qkv, q, kp, vp, positions, slots, None, H, G, hd, ps, use_rope=False, adjacent=False, use_norm=False, norm_eps=0.0,
                       use_temp=False, floor_scale=0, attn_scale=0.0, kv_tiled=True)
    args = (positions, seq, bt, T, H, G, hd, ps, vis, span, hd ** -0.5, n_splits)
    ops().attn_decode(q, kp, vp, want, scratch, *args)
    ops().attn_decode_rope(qkv, kp2, vp2, got, scratch, positions, slots, *args[1:])
    bits = lambda t: t.view(torch.int16)
    assert torch.equal(bits(kp), bits(kp2)) and torch.equal(bits(vp), bits(vp2))
    assert torch.equal(bits(got), bits(want)) and bool(torch.isfinite(want.float()).all())
