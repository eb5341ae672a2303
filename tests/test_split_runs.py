"""The tiled product with its sum over k cut into runs: any number of runs, partial sums anywhere a float may lie."""
import pytest
import torch

from test_kernels import DEV, ops, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,runs", [(70, 64, 4096, r) for r in (2, 4, 7, 8, 11, 16, 32)] + [(129, 528, 2112, r) for r in (2, 3, 5, 6, 9, 11)])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_the_runs_sums_added_in_their_order(M, N, K, runs, off, out_dtype):
    a, w = rnd(M, K, dtype=torch.bfloat16), ops().operand_order(rnd(N, K, dtype=torch.bfloat16, seed=1))
    part = torch.empty(runs * M * N + off, device=DEV)[off:].view(runs, M, N)
    y = torch.empty(M, N, dtype=out_dtype, device=DEV)
    ops().gemm_tiled(a, w, y, M, N, K, part=part)
    total = torch.zeros(M, N, device=DEV)
    for r in range(runs):
        total += part[r]
    assert torch.equal(y, total.to(out_dtype))
    want = a.double() @ rnd(N, K, dtype=torch.bfloat16, seed=1).double().T
    assert (y.double() - want).abs().max() <= 2e-2 * max(1.0, float(want.abs().max()))      # as the product in one run
