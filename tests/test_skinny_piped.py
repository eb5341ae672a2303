"""The weight stream of one or two rows, and over groups, against the one of three rows: the same bits for every number of a
wave's blocks, and against 64 bits."""
import pytest
import torch

from test_kernels import DEV, ops, rnd


@pytest.mark.gpu
@pytest.mark.parametrize("variant,waves", [(5, 4), (6, 8), (8, 8)])
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("N", [16, 48, 272])
def test_a_row_alone_in_pairs_and_in_groups(variant, waves, glu, N):
    # up to five and a half blocks of 64 a wave: none, one, and every remainder of the loop over pairs
    for K in [64 * b for b in (1, waves - 1, waves, waves + 1, 2 * waves, 3 * waves - 1, 3 * waves, 4 * waves + 1, 5 * waves + 3)]:
        x, w = rnd(3, K).bfloat16(), rnd((2 if glu else 1) * N, K, seed=1).bfloat16()
        wt = ops().operand_order(w)
        three, one, two = (torch.empty(n, N, device=DEV) for n in (3, 1, 2))
        run = lambda a, y, n: ops().gemm_skinny(a, wt, y, n, N, K, glu=glu, tiled=True, variant=variant)
        run(x, three, 3)
        run(x[:1].contiguous(), one, 1)
        run(x[1:].contiguous(), two, 2)
        assert torch.equal(one, three[:1]) and torch.equal(two, three[1:]), K
        exact = x.double() @ w.double().T
        if glu:
            exact = torch.nn.functional.silu(exact[:, :N]) * exact[:, N:]
        # fp32 sums of K exact products, the gate's silu (2^-20) beside them
        assert (three - exact).abs().max() <= (K * 2.0 ** -23 + 2.0 ** -20) * exact.abs().max() + 1e-30, K

        # groups of 2, 0, 17 and 1 rows through a row list, scaled, to rows in another order
        sizes = [2, 0, 17, 1]
        src = torch.tensor([i % 3 for i in range(20)], dtype=torch.int32, device=DEV)
        dst = torch.arange(19, -1, -1, dtype=torch.int32, device=DEV)
        scale = torch.tensor([1.0, 0.5, 2.0, 4.0] * 5, device=DEV)          # powers of two: exact in any order
        off = torch.tensor([0, 2, 2, 19, 20], dtype=torch.int32, device=DEV)
        ws = ops().operand_order(torch.stack([w] * len(sizes)))
        got = torch.full((20, N), float("nan"), device=DEV)
        ops().gemm_skinny(x, ws, got, 20, N, K, offsets=off, n_groups=4, a_rows=src, a_scale=None if glu else scale, y_rows=dst, glu=glu,
                          max_rows=17 if variant != 5 else 16, tiled=True, variant=variant)
        want = three[src.long()] * (1.0 if glu else scale[:, None])
        assert torch.equal(got[dst.long()], want), K
