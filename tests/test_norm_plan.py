"""One row: the norm that forms a router's logits also leaves the row list of the grouped products."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("d,E", [(64, 1), (66, 3), (5120, 16), (2048, 130), (12032, 250)])
@pytest.mark.parametrize("shared", [0, 1])
@pytest.mark.parametrize("kind", ["plain", "ties", "nan first", "nan later", "low"])
def test_plan_of_one_row_is_moe_plans(d, E, shared, kind):
    """Every array equals what ``moe_plan`` makes of the same logits, whichever expert wins: the last one, the first of
    equals, logits that are not numbers, and all of them below anything a float holds."""
    from spite_amd.csrc import hipops
    torch.manual_seed(d + E)
    h, w = torch.randn(1, d, device="cuda"), torch.rand(d, device="cuda") + 0.5
    proj = torch.randn(E, d, device="cuda")
    if kind == "plain":
        proj[-1] = h[0]
    elif kind == "ties":
        proj[E // 2:] = h[0]
    elif kind == "nan first":
        proj[0] = float("nan")
    elif kind == "nan later":
        proj[-1] = float("nan")
    else:
        proj[:] = -h[0].sign() * float("inf")
    n = 1 + shared
    def arrays():
        i = lambda k: torch.full((k,), -7, dtype=torch.int32, device="cuda")
        f = lambda k: torch.full((k,), -7.0, device="cuda")
        return i(1), f(1), i(n), f(n), i(n), i(E + 1 + shared)
    logits, out = torch.empty(1, E, device="cuda"), torch.empty(1, d, device="cuda", dtype=torch.bfloat16)
    got = arrays()
    hipops.add_rmsnorm(h, w, 1e-5, out=out, proj=proj, proj_out=logits, plan=got + (shared,))
    want = arrays()
    hipops.moe_plan(*want, 1, E, shared, logits=logits)
    for a, b in zip(got, want):
        assert torch.equal(torch.nan_to_num(a.float(), nan=-9.0), torch.nan_to_num(b.float(), nan=-9.0))


@pytest.mark.gpu
def test_plan_is_refused_for_more_rows_and_rows_that_do_not_fit():
    from spite_amd.csrc import hipops
    for rows, d, E in ((2, 64, 4), (1, 12288, 4)):
        h, proj = torch.randn(rows, d, device="cuda"), torch.randn(E, d, device="cuda")
        i = torch.zeros(8, dtype=torch.int32, device="cuda")
        f = torch.zeros(8, device="cuda")
        with pytest.raises(hipops.KernelError):
            hipops.add_rmsnorm(h, torch.ones(d, device="cuda"), 1e-5, out=torch.empty_like(h), proj=proj,
                               proj_out=torch.empty(rows, E, device="cuda"), plan=(i, f, i, f, i, i, 1))
