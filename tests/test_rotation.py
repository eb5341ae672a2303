"""A pair's rotation, bit for bit: (a cos - b sin, b cos + a sin) with one rounded product and one fused multiply-add each, in the
kernel that rotates a prompt's rows and in the decode attention that rotates its own, from the 32-bit kernel's sines and cosines."""
import pytest
import torch

from test_kernels import DEV, ops, rnd

pytestmark = pytest.mark.gpu


def _sines(positions, inv, hd):
    """The kernels' own cosines and sines: rows (1, 0) rotated in 32 bits."""
    T, half = positions.numel(), hd // 2
    rows = torch.cat([torch.ones(T, half), torch.zeros(T, half), torch.zeros(T, 2 * hd)], 1).to(DEV)
    out = torch.empty(T, hd, device=DEV)
    ops().rope_kvwrite(rows, out, None, None, positions, None, inv, 1, 1, hd, 32, use_rope=True, adjacent=False, use_norm=False,
                       norm_eps=0.0, use_temp=False, floor_scale=1, attn_scale=0.0, write_kv=False)
    return out[:, :half].cpu(), out[:, half:].cpu()


def _rotated(x, cs, sn, adjacent):
    """x [T, heads, hd] in bfloat16, on the CPU: a fused product is exact in 64 bits."""
    half = x.shape[-1] // 2
    x = x.cpu().float()
    a, b = (x[..., 0::2], x[..., 1::2]) if adjacent else (x[..., :half], x[..., half:])
    cs, sn = cs[:, None], sn[:, None]
    ra = (a.double() * cs.double() - (b * sn).double()).float().bfloat16()
    rb = (b.double() * cs.double() + (a * sn).double()).float().bfloat16()
    return torch.stack([ra, rb], -1).flatten(-2) if adjacent else torch.cat([ra, rb], -1)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("adjacent", [False, True])
@pytest.mark.parametrize("T", [200, 2048])
def test_prompt_rows(hd, adjacent, T):
    H, G, ps = 1024 // hd, 2, 32
    qkv = rnd(T, (H + 2 * G) * hd, dtype=torch.bfloat16)
    positions = torch.randperm(3 * T, generator=torch.Generator().manual_seed(1))[:T].to(torch.int32).to(DEV)
    inv = (10000.0 ** (-torch.arange(hd // 2, dtype=torch.float64) * 2 / hd)).float().to(DEV)
    slots = torch.arange(T, dtype=torch.int32, device=DEV)
    q = torch.empty(T, H * hd, dtype=torch.bfloat16, device=DEV)
    pages = -(-T // ps)
    k, v = torch.zeros(pages, G, ps, hd, dtype=torch.bfloat16, device=DEV), torch.zeros(pages, G, hd, ps, dtype=torch.bfloat16, device=DEV)
    ops().rope_kvwrite(qkv, q, k, v, positions, slots, inv, H, G, hd, ps, use_rope=True, adjacent=adjacent, use_norm=False, norm_eps=0.0,
                       use_temp=False, floor_scale=1, attn_scale=0.0)
    rows = qkv.view(T, H + 2 * G, hd)
    want = _rotated(rows[:, :H + G], *_sines(positions, inv, hd), adjacent)
    keys = k.transpose(1, 2).reshape(pages * ps, G, hd)[:T]
    values = v.permute(0, 3, 1, 2).reshape(pages * ps, G, hd)[:T]
    assert torch.equal(q.view(T, H, hd).cpu(), want[:, :H]) and torch.equal(keys.cpu(), want[:, H:])
    assert torch.equal(values, rows[:, H + G:])


def test_decoded_rows():
    T, H, G, hd, ps = 1024, 8, 8, 128, 32
    qkv = rnd(T, (H + 2 * G) * hd, dtype=torch.bfloat16)
    positions = torch.randint(0, ps, (T,), generator=torch.Generator().manual_seed(1)).to(torch.int32).to(DEV)
    inv = (31.0 * 10000.0 ** (-torch.arange(hd // 2, dtype=torch.float64) * 2 / hd)).float().to(DEV)
    own = torch.arange(T, dtype=torch.int32, device=DEV)                 # a request and a page a token
    k, v = torch.zeros(T, G, ps, hd, dtype=torch.bfloat16, device=DEV), torch.zeros(T, G, hd, ps, dtype=torch.bfloat16, device=DEV)
    out = torch.empty(T, H * hd, dtype=torch.bfloat16, device=DEV)
    scratch = torch.empty(max(ops().attn_decode_workspace(T, H, hd, 1) // 4, 4), dtype=torch.float32, device=DEV)
    ops().attn_decode_rope(qkv, k, v, out, scratch, positions, own * ps + positions, own, own[:, None].contiguous(), T, H, G, hd, ps,
                           "full", 0, hd ** -0.5, 1, inv_freq=inv)
    plain = torch.zeros_like(k)
    want = _rotated(qkv.view(T, H + 2 * G, hd)[:, H:H + G], *_sines(positions, inv, hd), False)
    plain[own.long(), :, positions.long()] = want.to(DEV)
    assert torch.equal(k, ops().kv_operand_order(plain, v)[0])
