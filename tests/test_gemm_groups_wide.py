"""The product over groups in tiles of 320 columns, and the order in which these and four waves' tiles over many groups go to the XCDs: every
height, groups of up to four tiles and larger ones, among many groups; bit for bit against the tiled product."""
import pytest
import torch

from test_gemm_groups import HEIGHTS
from test_kernels import DEV, ops, rnd, run_gemm


@pytest.mark.gpu
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N", [16, 304, 320, 336, 656])
@pytest.mark.parametrize("K", [64, 192, 320, 448])
@pytest.mark.parametrize("cap", [128, 160])
def test_every_height_row_lists_and_scales(out_dtype, N, K, cap):
    M, G = sum(HEIGHTS), len(HEIGHTS)
    g = torch.Generator().manual_seed(3)
    a, w = rnd(M + 3, K, dtype=torch.bfloat16), ops().operand_order(rnd(G, N, K, dtype=torch.bfloat16, seed=1))
    kw = dict(offsets=torch.tensor([sum(HEIGHTS[:g]) for g in range(G + 1)], dtype=torch.int32, device=DEV), n_groups=G,
              a_rows=torch.randint(0, M + 3, (M,), generator=g).to(torch.int32).to(DEV), a_scale=(torch.rand(M, generator=g) + 0.5).to(DEV),
              y_rows=torch.randperm(M + 2, generator=g)[:M].to(torch.int32).to(DEV))
    y, z = torch.zeros(M + 2, N, dtype=out_dtype, device=DEV), torch.zeros(M + 2, N, dtype=out_dtype, device=DEV)
    ops().gemm_tiled(a, w, y, M, N, K, shape=1, **kw)
    ops().gemm_groups(torch.full_like(a, float("nan")), w, z, M, N, K, waves=5, cap=cap, **kw)      # what the local memory held must not show
    ops().gemm_groups(a, w, z, M, N, K, waves=5, cap=cap, **kw)
    assert torch.equal(y, z)


@pytest.mark.gpu
@pytest.mark.parametrize("waves", [4, 5])
@pytest.mark.parametrize("rows", [[512, 513, 0, 700, 1], [3] * 70 + [900] + [129] * 60, [1300, 600], [0] * 63 + [641, 2, 640], [20] * 9, [30] * 62 + [200], [30] * 63 + [200]])
def test_small_and_large_groups_among_each_other(waves, rows):
    M, N, K, G = sum(rows), 1296, 128, len(rows)
    a, w = rnd(M, K, dtype=torch.bfloat16), ops().operand_order(rnd(G, N, K, dtype=torch.bfloat16, seed=1))
    offsets = torch.tensor([sum(rows[:g]) for g in range(G + 1)], dtype=torch.int32, device=DEV)
    y, z = torch.full((M + 9, N), 7.0, device=DEV), torch.full((M + 9, N), 7.0, device=DEV)
    ops().gemm_tiled(a, w, y, M, N, K, offsets=offsets, n_groups=G, shape=1)
    ops().gemm_groups(a, w, z, M, N, K, offsets=offsets, n_groups=G, waves=waves, cap=128)
    assert torch.equal(y, z) and (z[M:] == 7.0).all()


@pytest.mark.gpu
def test_against_64_bits_and_refusals():
    def fn(a, w, y, M, N, K, **kw):
        ops().gemm_groups(a, ops().operand_order(w), y, M, N, K, waves=5, cap=160, **kw)
    run_gemm(fn, torch.bfloat16, torch.float32, 400, 336, 192, False, True, 5)
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ops().KernelError):
        ops().gemm_groups(z(4, 64), z(1, 32, 64), z(4, 16), 4, 16, 64, offsets=torch.tensor([0, 4], dtype=torch.int32, device=DEV), n_groups=1, glu=True, waves=5)


def test_choice_where_they_fit_the_chip():
    """16 experts: sixteen tiles of 320 columns are one a compute unit (2,048 tokens 273 / 237 us, 1,547 236 / 219); a gated product and an
    expert more than fits keep what they had."""
    from spite_amd.csrc.hipops import gemm_groups_wide_choice
    at = lambda T, E, top, whole, N, K: gemm_groups_wide_choice(T, E, T * top / E, whole, N, K, 3)
    assert at(2048, 16, 1, 0, 5120, 8192)[0] == 5 and at(1547, 16, 1, 0, 5120, 8192)[0] == 5 and at(2077, 16, 1, 0, 5120, 4096) == (5, 160)
    assert at(940, 32, 4, 0, 2048, 5120) is None and at(330, 16, 1, 1, 5120, 8192) is None and at(0, 16, 1, 0, 64, 64) is None
