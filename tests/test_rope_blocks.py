"""Rotation and cache write of many tokens: values that go to their pages eight keys at a time, against the same rows written a few
tokens a call, over runs of places that begin and end anywhere."""
import pytest
import torch

from test_kernels import DEV, ops, rnd

pytestmark = pytest.mark.gpu


def _slots(T, ps, starts):
    """Runs of consecutive places from each start on, in pages of their own; places missing and exchanged here and there."""
    each, out = -(-T // len(starts)), []
    pages = -(-(each + 32) // ps)
    for r, first in enumerate(starts):
        out += [r * pages * ps + first + i for i in range(min(each, T - len(out)))]
    if T > 140:
        out[50] = out[131] = -1
        out[90], out[91] = out[91], out[90]
    return torch.tensor(out, dtype=torch.int32, device=DEV), len(starts) * pages


@pytest.mark.parametrize("H,G,hd", [(4, 2, 128), (3, 1, 8), (5, 3, 64), (2, 2, 512)])
@pytest.mark.parametrize("T", [256, 287, 289, 330, 1037])
@pytest.mark.parametrize("ps,tiled", [(32, True), (32, False), (8, False), (64, True)])
def test_many_tokens_write_what_few_write(H, G, hd, T, ps, tiled):
    if tiled and hd % 32:
        pytest.skip("operand order takes head sizes of 32 and multiples")
    slots, n_pages = _slots(T, ps, (0, 5, 8, 23))
    qkv = rnd(T, (H + 2 * G) * hd, dtype=torch.bfloat16)
    pos = (torch.arange(T, dtype=torch.int32, device=DEV) * 7) % 1000
    inv = (10000.0 ** (-torch.arange(hd // 2, dtype=torch.float64) * 2 / hd)).float().to(DEV)

    def run(step):
        q = torch.zeros(T, H * hd, dtype=torch.bfloat16, device=DEV)
        k, v = (torch.zeros(n_pages * G * ps * hd, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        kp, vp = k.view(n_pages, G, ps, hd), v.view(n_pages, G, hd, ps)
        for t in range(0, T, step):
            e = min(T, t + step)
            ops().rope_kvwrite(qkv[t:e], q[t:e], kp, vp, pos[t:e], slots[t:e], inv, H, G, hd, ps, use_rope=True, adjacent=False, use_norm=True,
                               norm_eps=1e-5, use_temp=True, floor_scale=64, attn_scale=0.1, kv_tiled=tiled)
        return q, kp, vp

    for got, want in zip(run(T), run(100)):
        assert torch.equal(got, want)
