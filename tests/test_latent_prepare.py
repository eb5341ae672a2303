"""Latent attention's preparation: pairs turned from the table of a token's angles and past it, elements that pass, the cache row."""
import pytest
import torch

from test_kernels import DEV, ops, rnd


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,n,r,R,rot", [(1, 1, 2, 2, 3, 2), (3, 5, 8, 7, 300, 6), (2, 40, 16, 64, 512, 64), (2, 3, 8, 9, 33, 0), (2, 2, 4, 512, 64, 512), (2, 2, 4, 530, 64, 516)])
@pytest.mark.parametrize("own", [False, True])
def test_against_64_bits(T, H, n, r, R, rot, own):
    qd, dkv, w = rnd(T, H * (n + r)), rnd(T, R + r, seed=1), rnd(R, seed=2)
    inv = 10000.0 ** (-torch.arange(max(rot // 2, 1), device=DEV).float() / max(rot // 2, 1))
    pos = torch.tensor([0, 4999, 17][:T], dtype=torch.int32, device=DEV)
    slots = torch.tensor([3, -1, 0][:T], dtype=torch.int32, device=DEV)
    qa, kv = torch.zeros(T * H, R + r, device=DEV), torch.full((1, 1, 4, R + r), 7.0, device=DEV)
    rows, off = torch.zeros(H * T, dtype=torch.int32, device=DEV), torch.zeros(H + 1, dtype=torch.int32, device=DEV)
    ops().latent_prepare(qd, dkv, qa, kv, pos, slots, inv, w, 1e-6, H, n, r, R, rot, own, rows, off)
    ang = (pos.float()[:, None] * inv[:rot // 2]).double()              # the angle is a product of 32 bits
    c, s = torch.cos(ang), torch.sin(ang)

    def turned(x):                                                      # [T, heads, r]
        y, c_, s_ = x.double().clone(), c[:, None], s[:, None]
        a, b = x[..., 0:rot:2].double(), x[..., 1:rot:2].double()
        y[..., 0:rot:2], y[..., 1:rot:2] = a * c_ - b * s_, b * c_ + a * s_
        return y
    q = qd.view(T, H, n + r)[..., n:]
    # two products and a sum, sine and cosine within 2 units in the last place: 6 of them of the pair's length
    bound = 6 * 2.0 ** -24 * 2 * q.abs().max()
    assert (qa.view(T, H, R + r)[..., R:] - turned(q)).abs().max() <= bound
    assert (qa.view(T, H, R + r)[..., :R] == 0).all()
    assert rows.tolist() == [t * H + h for h in range(H) for t in range(T)] and off.tolist() == [h * T for h in range(H + 1)]
    if not own:
        assert (kv == 7.0).all()
        return
    lat = dkv[:, :R].double()
    lat = lat / torch.sqrt((lat * lat).mean(1, keepdim=True) + 1e-6) * w.double()
    part = turned(dkv[:, None, R:])[:, 0]
    for t, slot in enumerate(slots.tolist()):
        if slot >= 0:
            assert (kv[0, 0, slot, :R] - lat[t]).abs().max() <= (R + 8) * 2.0 ** -24 * lat[t].abs().max()      # a sum of R squares, a root, two products
            assert (kv[0, 0, slot, R:] - part[t]).abs().max() <= 6 * 2.0 ** -24 * 2 * dkv[:, R:].abs().max()
    free = [i for i in range(4) if i not in slots.tolist()]
    assert (kv[0, 0, free] == 7.0).all()
