"""The row list of many tokens at the edges of its workgroups (256 tokens, 1,024 threads) and of an expert's number of bits, with
entries that belong to no expert, against a stable sort."""
import pytest
import torch

from test_kernels import DEV, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [257, 512, 1023, 1025, 2050])
@pytest.mark.parametrize("E", [1, 2, 5, 64, 65, 2048])
@pytest.mark.parametrize("kind", ["spread", "one", "some of none"])
def test_many_tokens_in_order_inside_their_groups(T, E, kind):
    g = torch.Generator().manual_seed(T + E)
    expert = torch.randint(0, E, (T,), generator=g, dtype=torch.int32)
    if kind == "one":
        expert[:] = E - 1
    elif kind == "some of none":
        expert[::7], expert[3::11] = -1, E
    weight = torch.rand(T, generator=g)
    src, dst = (torch.full((2 * T,), -7, dtype=torch.int32, device=DEV) for _ in range(2))
    scale, offsets = torch.full((2 * T,), -7.0, device=DEV), torch.empty(E + 2, dtype=torch.int32, device=DEV)
    ops().moe_plan(expert.to(DEV), weight.to(DEV), src, scale, dst, offsets, T, E, True)
    of_one = (expert >= 0) & (expert < E)
    order = torch.nonzero(of_one).flatten()
    order = order[torch.sort(expert[order], stable=True).indices]
    n = len(order)
    assert src[:n].tolist() == order.tolist() and dst[:n].tolist() == order.tolist()
    assert torch.equal(scale[:n].cpu(), weight[order])
    counts = torch.bincount(expert[of_one].long(), minlength=E)
    assert offsets.tolist() == [0] + torch.cumsum(counts, 0).tolist() + [2 * T]
    shared = torch.nonzero(of_one).flatten()                       # a shared expert's row is written by its token's entry
    assert src[T + shared.to(DEV)].tolist() == shared.tolist() and dst[T + shared.to(DEV)].tolist() == (T + shared).tolist()
