"""The 32-bit stream of few rows over sums of every kind of run: the bits of a tile's rows."""
import pytest
import torch

from test_kernels import DEV, ops, rnd


def operands(K, glu):
    """70 rows of X, 64 rows of W (of either half), and these repeated to a W of N rows."""
    a, w = rnd(70, K), rnd((2 if glu else 1) * 64, K, seed=1)
    tall = lambda N: torch.cat([half.repeat(-(-N // 64), 1)[:N] for half in w.split(64)])
    tile = torch.empty(70, 33000, device=DEV)              # tall enough for tiles from nine rows on
    ops().gemm_generic(a, tall(33000), tile, 70, 33000, K, glu=glu)
    return a, w, tall, tile[:, :64]


@pytest.mark.gpu
@pytest.mark.parametrize("K", [32, 96, 512, 544, 1020, 1024, 1028, 1540, 1700, 1764, 2048, 2112, 2564, 3584, 4612])
@pytest.mark.parametrize("glu", [False, True])
def test_every_number_of_pieces_a_run(K, glu):
    # a run is K / 8 rounded up to 64: an even number of pieces of 32 up to twenty, the last run any (1,700 five and 1,764 seven, then an end inside a piece)
    a, w, _, tile = operands(K, glu)
    for rows in (1, 2, 16, 17, 40):
        y = torch.empty(rows, 64, device=DEV)
        ops().gemm_generic(a[:rows].contiguous(), w, y, rows, 64, K, glu=glu)
        assert torch.equal(y, tile[:rows]), rows


@pytest.mark.gpu
@pytest.mark.parametrize("K", [32, 544, 1028, 1700, 1764, 2048])
@pytest.mark.parametrize("rows,variant", [(17, 32), (32, 32), (33, 64), (64, 64)])
@pytest.mark.parametrize("glu", [False, True])
def test_32_and_64_rows_a_workgroup(K, rows, variant, glu):
    N = 3072
    assert ops().lib().spite_gemm_f32_choice(rows, N, K, 0, int(glu)) == variant
    a, _, tall, tile = operands(K, glu)
    y = torch.empty(rows, N, device=DEV)
    ops().gemm_generic(a[:rows].contiguous(), tall(N), y, rows, N, K, glu=glu)
    assert torch.equal(y, tile[:rows].repeat(1, N // 64))
