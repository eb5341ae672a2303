"""The choice of experts among equals, infinities and what is no number: the lowest index first, whatever lanes hold them, and the weight of the
expert that was taken."""
import pytest
import torch

from test_kernels import DEV, ops

SIZES = [(1, 1), (16, 4), (63, 3), (64, 64), (65, 5), (128, 8), (300, 70), (512, 8)]


def taken(row, top, groups=None):
    """The experts by value, the lowest index among equals; a taken one falls to minus infinity, where what is no number is, too."""
    row = torch.where(row.isnan(), torch.full_like(row, float("-inf")), row)
    first = lambda x: int((x == x.max()).nonzero()[0])
    if groups:
        size, open_ = row.numel() // groups[0], torch.zeros(row.numel(), dtype=torch.bool)
        for _ in range(groups[1]):
            left = torch.where(open_, torch.full_like(row, float("-inf")), row)
            e = first(left)
            open_[e // size * size:(e // size + 1) * size] = True
        row = torch.where(open_, row, torch.full_like(row, float("-inf")))
    out, row = [], row.clone()
    for _ in range(top):
        out.append(first(row))
        row[out[-1]] = float("-inf")
    return out


def choose(z, bias, top, **kw):
    expert, weight = torch.full((z.shape[0] * top,), -1, dtype=torch.int32, device=DEV), torch.full((z.shape[0] * top,), -1.0, device=DEV)
    ops().router_topk(z.to(DEV), None if bias is None else bias.to(DEV), expert, weight, top, **kw)
    return expert.view(-1, top).tolist(), weight.view(-1, top).cpu().double()


@pytest.mark.gpu
@pytest.mark.parametrize("E,top", SIZES)
@pytest.mark.parametrize("kind", ["equal", "steps", "infinite", "nan", "last"])
def test_lowest_index_among_equals(E, top, kind):
    T = 9
    g = torch.Generator().manual_seed(E + top)
    z = torch.randn(T, E, generator=g)
    if kind == "equal":
        z = torch.zeros(T, E)
    elif kind == "steps":
        z = z.round()
    elif kind == "infinite":
        z[:, ::2] = float("-inf")
    elif kind == "nan":
        z[:, ::3] = float("nan")
    else:
        z[:, -1] = z.max() + 1.0
    expert, weight = choose(z, None, top, scoring="softmax_taken")
    for t in range(T):
        assert expert[t] == taken(z[t], top)
        if not z[t][expert[t]].isfinite().any() or z[t][expert[t]].isnan().any():
            continue                                        # no weights among what has no finite value
        # a softmax of 32 bits: an exponential (2 units), a product, and a sum that `top` rescaled terms have gone into
        assert (weight[t] - torch.softmax(z[t][expert[t]].double(), 0)).abs().max() <= (top + 4) * 2.0 ** -23


@pytest.mark.gpu
@pytest.mark.parametrize("E,top,groups", [(E, top, None) for E, top in SIZES] + [(E, top, (8, 3)) for E, top in SIZES if E % 8 == 0 and 8 * top <= 3 * E])
@pytest.mark.parametrize("renorm", [False, True])
def test_equals_by_score_and_bias_weighed_without_it(E, top, renorm, groups):
    T = 9
    g = torch.Generator().manual_seed(E * 3 + top)
    # scores of exactly 0, one half and 1, and biases that make them equal across experts
    z = torch.tensor([-200.0, 0.0, 40.0])[torch.randint(0, 3, (T, E), generator=g)]
    bias = torch.tensor([0.0, 0.5, -0.5, 0.25])[torch.randint(0, 4, (E,), generator=g)]
    score = torch.sigmoid(z.double())
    score = torch.where(z > 1, torch.ones_like(score), torch.where(z < -1, torch.zeros_like(score), score))
    expert, weight = choose(z, bias, top, renorm=renorm, scoring="sigmoid", **({"groups": groups} if groups else {}))
    for t in range(T):
        assert expert[t] == taken((score[t] + bias).float(), top, groups)
        want = score[t][expert[t]]
        if renorm:
            want = want / (want.sum() + 1e-20)
        assert (weight[t] - want).abs().max() <= 4 * 2.0 ** -24       # halves are summed exactly; a reciprocal and a product
