"""The 32-bit stream of few rows over sums of every number of pieces a run: the bits of a tile's rows."""
import pytest
import torch

from test_kernels import DEV, ops, rnd


@pytest.mark.gpu
@pytest.mark.parametrize("K", [32, 96, 512, 544, 1020, 1024, 1028, 1540, 2048, 2112, 2564, 3584, 4612])
@pytest.mark.parametrize("glu", [False, True])
def test_every_number_of_pieces_a_run(K, glu):
    # a run is K / 8 rounded up to 64: none to eighteen pieces of 32, the last run's end inside a piece
    N = 33000                                        # tall enough for tiles from nine rows on
    a, w = rnd(70, K), rnd((2 if glu else 1) * 64, K, seed=1)
    tall = torch.cat([w[:64].repeat(516, 1)[:N], w[64:].repeat(516, 1)[:N]]) if glu else w.repeat(516, 1)[:N]
    tile = torch.empty(70, N, device=DEV)
    ops().gemm_generic(a, tall, tile, 70, N, K, glu=glu)
    for rows in (1, 2, 16, 17, 40):
        y = torch.empty(rows, 64, device=DEV)
        ops().gemm_generic(a[:rows].contiguous(), w, y, rows, 64, K, glu=glu)
        assert torch.equal(y, tile[:rows, :64]), rows
