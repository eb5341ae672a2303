"""The choice of several experts and the row list in one call against the two calls it stands for, with groups that every
token visits; on both sides of the size up to which one workgroup does it."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,E,top,shared", [(1, 4, 1, 0), (1, 16, 4, 2), (2, 70, 2, 1), (128, 16, 4, 2), (129, 16, 4, 2), (7, 300, 70, 1),
                                            (300, 512, 2, 4), (64, 8, 8, 3)])
@pytest.mark.parametrize("scoring,groups", [("sigmoid", None), ("softmax_taken", None), ("softmax", (2, 2))])
def test_router_plan(T, E, top, shared, scoring, groups):
    from spite_amd.csrc import hipops
    g = torch.Generator().manual_seed(T + E)
    z = torch.randn(T, E, generator=g).round(decimals=1).to(DEV)          # (equal logits among them)
    bias = (0.1 * torch.randn(E, generator=g)).to(DEV)
    i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device=DEV)
    n, rows = T * top, T * (top + shared)
    want_e, want_w = i32(n), torch.empty(n, device=DEV)
    hipops.router_topk(z, bias, want_e, want_w, top, scoring=scoring, groups=groups)
    expert, weight = i32(n), torch.empty(n, device=DEV)
    src, dst, scale, offsets = i32(rows), i32(rows), torch.empty(rows, device=DEV), i32(E + shared + 1)
    hipops.router_plan(z, bias, expert, weight, top, src, scale, dst, offsets, shared, scoring=scoring, groups=groups)
    assert torch.equal(expert, want_e) and torch.equal(weight, want_w)
    e = want_e.cpu().numpy()
    order = np.argsort(e, kind="stable")
    tail = np.arange(shared * T)
    assert np.array_equal(dst.cpu().numpy(), np.concatenate([order, n + tail]))
    assert np.array_equal(src.cpu().numpy(), np.concatenate([order // top, tail % T if T else tail]))
    assert torch.equal(scale.cpu(), torch.cat([want_w.cpu()[torch.from_numpy(order)], torch.ones(shared * T)]))
    first = [int((e < x).sum()) for x in range(E + 1)] + [n + (j + 1) * T for j in range(shared)]
    assert offsets.cpu().tolist() == first


@pytest.mark.parametrize("parts", [1, 3])
@pytest.mark.parametrize("d", [64, 30])
def test_combine_adds_the_parts_of_the_extra_row(parts, d):
    from spite_amd.csrc import hipops
    T, top = 5, 3
    g = torch.Generator().manual_seed(d)
    y, w, ex = torch.randn(T * top, d, generator=g), torch.rand(T * top, generator=g), torch.randn(parts * T, d, generator=g)
    out = torch.empty(T, d, device=DEV)
    hipops.moe_combine(y.to(DEV), w.to(DEV), ex.to(DEV), out, T, top, n_extra=parts)
    ref = (y.double().view(T, top, d) * w.double().view(T, top, 1)).sum(1) + ex.double().view(parts, T, d).sum(0)
    assert (out.cpu().double() - ref).abs().max() < 1e-5 * float(ref.abs().max())      # a few fp32 roundings


@pytest.mark.parametrize("T,fan", [(7, 2), (1, 4), (601, 3)])
def test_plan_of_entries_that_end_inside_a_token(T, fan):
    """Without groups that every token visits, the last token may bring fewer entries than the others."""
    from spite_amd.csrc import hipops
    E = 5
    expert = torch.randint(0, E, (T,), generator=torch.Generator().manual_seed(T), dtype=torch.int32)
    weight = torch.rand(T, generator=torch.Generator().manual_seed(1))
    src, dst, offsets = (torch.full((n,), -7, dtype=torch.int32, device=DEV) for n in (T, T, E + 1))
    scale = torch.empty(T, device=DEV)
    hipops.moe_plan(expert.to(DEV), weight.to(DEV), src, scale, dst, offsets, T, E, False, fan=fan)
    order = torch.argsort(expert, stable=True)
    assert torch.equal(dst.cpu().long(), order) and torch.equal(src.cpu().long(), order // fan) and torch.equal(scale.cpu(), weight[order])
    assert offsets.cpu().tolist() == [int((expert < e).sum()) for e in range(E + 1)]
    with pytest.raises(hipops.KernelError):                # (a group of whole tokens has no row list then)
        hipops.moe_plan(expert.to(DEV), weight.to(DEV), torch.cat([src] * 2), torch.cat([scale] * 2), torch.cat([dst] * 2),
                        torch.cat([offsets] * 2), T, E, True, fan=fan)


@pytest.mark.parametrize("T,E,top,shared", [(8, 512, 64, 1), (8, 4, 1, 2), (9, 16, 4, 1), (10, 64, 50, 0)])
def test_on_both_sides_of_a_token_a_wave(T, E, top, shared):
    test_router_plan(T, E, top, shared, "sigmoid", None)
