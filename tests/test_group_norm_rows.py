"""The gated norm of wide groups: both ends of each number of elements a thread, weights that wrap, against 64 bits."""
import pytest
import torch

from test_kernels import DEV, ops, rnd


@pytest.mark.gpu
@pytest.mark.parametrize("group", [512, 513, 2048, 2049, 5120, 5121, 8192, 8193])
@pytest.mark.parametrize("act", [None, "silu", "sigmoid"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_wide_groups(group, act, dtype):
    T, n = 3, 2 * group
    o, gate = rnd(T, n), rnd(T, n + 8, seed=1).to(dtype)[:, :n]
    for n_w in (n, group):
        w = rnd(n_w, seed=2)
        y = torch.empty(T, n, dtype=dtype, device=DEV)
        ops().gated_group_norm(o, w, y, group, 1e-6, gate=gate if act else None, act=act)
        x = o.double().view(T, 2, group)
        x = (x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)).view(T, n) * w.double().repeat(n // n_w)
        if act:
            z = gate.double()
            x = x * (torch.nn.functional.silu(z) if act == "silu" else torch.sigmoid(z))
        # a sum of `group` squares by a thread's 32 and a tree, a root, and some eight roundings behind it; then the result's own
        bound = (48 * 2.0 ** -24 + (2.0 ** -8 if dtype == torch.bfloat16 else 0)) * x.abs() + 1e-7
        assert ((y.double() - x).abs() <= bound).all()
