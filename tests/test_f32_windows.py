"""32-bit attention behind short windows and chunks: as many waves as there are tiles to see, small heads without padding."""
import pytest
import torch

from test_f32_kernels import test_attention_over_tiles_of_32_keys as over_tiles
from test_kernels import DEV, PagedKV, ops, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,hd,ps,vis,span", [(6, 3, 48, 8, "window", 8), (4, 2, 16, 4, "window", 9), (4, 4, 32, 16, "window", 34),
                                                (2, 1, 16, 4, "chunk", 16), (3, 1, 96, 32, "window", 98), (4, 2, 16, 16, "window", 99),
                                                (2, 2, 32, 16, "full", 0), (2, 1, 128, 32, "chunk", 96)])
def test_waves_and_head_sizes(H, G, hd, ps, vis, span):
    over_tiles(H, G, hd, ps, vis, span)


@pytest.mark.parametrize("H,G,hd", [(8, 2, 128), (16, 8, 64), (8, 1, 32), (12, 4, 16), (40, 8, 48), (4, 4, 128), (8, 2, 96)])
@pytest.mark.parametrize("vis,span", [("full", 0), ("window", 60), ("window", 120), ("chunk", 96)])
def test_a_token_has_the_same_bits_alone_and_among_many(H, G, hd, vis, span):
    """Prompts' workgroups serve one, two or four query heads of a key head, a token alone one: the same order of every sum."""
    T, ps = 700, 16
    kv = PagedKV([T], G, hd, ps, torch.float32)
    kp, vp, bt = kv.kp.to(DEV), kv.vp.to(DEV), kv.bt.to(DEV)
    q = rnd(T, H * hd, seed=3)
    pos, seq = torch.arange(T, dtype=torch.int32, device=DEV), torch.zeros(T, dtype=torch.int32, device=DEV)
    slopes = (0.03 * (1 + torch.arange(H))).float().to(DEV)
    outs = []
    for each in (T, 96, 1):
        out = torch.zeros(T, H * hd, device=DEV)
        for a in range(0, T, each) if each > 1 else (0, 31, 32, 95, 96, 300, 699):
            n = min(each, T - a)
            ops().attn_generic(q[a:a + n], kp, vp, out[a:a + n], pos[a:a + n], seq[a:a + n], bt, n, H, G, hd, ps, vis, span, hd ** -0.5,
                               softcap=20.0, slopes=slopes)
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    for t in (0, 31, 32, 95, 96, 300, 699):
        assert torch.equal(outs[0][t], outs[2][t])


@pytest.mark.parametrize("H,G,T", [(8, 2, 300), (4, 4, 2)])
@pytest.mark.parametrize("first", [0, 3])
def test_keys_of_a_page_that_was_given_back_poison_every_query_that_sees_them(H, G, T, first):
    """A wave whose every tile lies in such pages has no maximum; its NaN must not be taken for a wave without tiles."""
    hd, ps, n = 64, 32, 400
    kv = PagedKV([n], G, hd, ps, torch.float32)
    bt = kv.bt.clone()
    bt[0, first] = -1
    q, out = rnd(T, H * hd, seed=3), torch.zeros(T, H * hd, device=DEV)
    pos, seq = torch.arange(n - T, n, dtype=torch.int32, device=DEV), torch.zeros(T, dtype=torch.int32, device=DEV)
    ops().attn_generic(q, kv.kp.to(DEV), kv.vp.to(DEV), out, pos, seq, bt.to(DEV), T, H, G, hd, ps, "full", 0, hd ** -0.5)
    sees = pos >= first * ps
    assert bool(torch.isnan(out[sees]).all()) and bool(torch.isfinite(out[~sees]).all())


@pytest.mark.parametrize("H,G,hd", [(5, 1, 128), (12, 4, 96), (6, 2, 80), (4, 4, 64), (8, 2, 128), (4, 2, 48)])
@pytest.mark.parametrize("vis,span", [("window", 1), ("window", 8), ("chunk", 8), ("window", 9)])
def test_windows_of_a_few_keys(H, G, hd, vis, span):
    """Which kernel takes them depends on the layer alone: a token has the same bits alone and among many, on both sides of the lines."""
    over_tiles(H, G, hd, 32, vis, span)
    test_a_token_has_the_same_bits_alone_and_among_many(H, G, hd, vis, span)
