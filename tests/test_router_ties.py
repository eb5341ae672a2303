"""The choice of experts among equals, infinities and what is no number: the lowest index first, whatever lanes hold them."""
import pytest
import torch

from test_kernels import DEV, ops


@pytest.mark.gpu
@pytest.mark.parametrize("E,top", [(1, 1), (16, 4), (63, 3), (64, 64), (65, 5), (128, 8), (300, 70), (512, 8)])
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
    expert, weight = torch.zeros(T * top, dtype=torch.int32, device=DEV), torch.zeros(T * top, device=DEV)
    ops().router_topk(z.to(DEV), None, expert, weight, top, scoring="softmax_taken")
    value = torch.where(z.isnan(), torch.full_like(z, float("-inf")), z)
    for t in range(T):
        row, got = value[t].clone(), expert[t * top:(t + 1) * top].tolist()
        for e in got:
            if row.max() == float("-inf"):
                break                                   # nothing but what is never preferred is left
            assert e == int((row == row.max()).nonzero()[0])
            row[e] = float("-inf")
