"""The product over groups in tiles of several heights: every height and both ends of it, one step of K and a last round that K
does not fill, against float64 and, bit for bit, against the tiled product (both add k in the same order)."""
import pytest
import torch

from test_kernels import DEV, ops, rnd, run_gemm

HEIGHTS = [0, 1, 32, 33, 64, 65, 80, 81, 96, 97, 112, 113, 128, 129, 144, 145, 160, 161, 0, 257, 321]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,groups", [(70, 48, 64, 5), (400, 272, 128, 3), (900, 528, 192, 4), (90, 16, 320, 70), (300, 144, 448, 130)])
@pytest.mark.parametrize("glu,out_dtype", [(False, torch.float32), (False, torch.bfloat16), (True, torch.bfloat16), (True, torch.float32)])
@pytest.mark.parametrize("waves,cap", [(4, 128), (4, 160), (8, 128), (8, 160)])
def test_groups_with_row_lists(M, N, K, groups, glu, out_dtype, waves, cap):
    def fn(a, w, y, M, N, K, **kw):
        ops().gemm_groups(a, ops().operand_order(w), y, M, N, K, waves=waves, cap=cap, **kw)
    run_gemm(fn, torch.bfloat16, out_dtype, M, N, K, glu, True, groups)


@pytest.mark.gpu
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("waves,cap", [(4, 128), (4, 160), (8, 128), (8, 160)])
@pytest.mark.parametrize("K", [64, 192, 320])
def test_groups_of_every_height_equal_the_tiled_product(glu, waves, cap, K):
    """What the local memory held before must not show: a product whose rows are not numbers runs first."""
    M, N, G = sum(HEIGHTS), 272, len(HEIGHTS)
    a, w = rnd(M, K, dtype=torch.bfloat16), ops().operand_order(rnd(G, 2 * N if glu else N, K, dtype=torch.bfloat16, seed=1))
    offsets = torch.tensor([sum(HEIGHTS[:g]) for g in range(G + 1)], dtype=torch.int32, device=DEV)
    y, z = torch.zeros(M, N, device=DEV), torch.ones(M, N, device=DEV)
    ops().gemm_tiled(a, w, y, M, N, K, offsets=offsets, n_groups=G, glu=glu, shape=1)
    ops().gemm_groups(torch.full_like(a, float("nan")), w, z, M, N, K, offsets=offsets, n_groups=G, glu=glu, waves=waves, cap=cap)
    ops().gemm_groups(a, w, z, M, N, K, offsets=offsets, n_groups=G, glu=glu, waves=waves, cap=cap)
    assert torch.equal(y, z)


@pytest.mark.gpu
def test_refuses_what_it_cannot_do():
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=DEV)
    o = torch.tensor([0, 4], dtype=torch.int32, device=DEV)
    call = lambda a, w, y, K=64, **kw: ops().gemm_groups(a, w, y, 4, y.shape[1], K, offsets=o, n_groups=1, **kw)
    for a, w, y, kw in ((z(4, 96), z(1, 16, 96), z(4, 16), dict(K=96)), (z(4, 64), z(1, 24, 64), z(4, 24), {}),
                        (z(4, 64), z(1, 16, 64), z(4, 18)[:, :16], {}), (z(4, 64), z(1, 16, 64), z(4, 16), dict(waves=6)),
                        (z(4, 64), z(1, 16, 64), z(4, 16), dict(cap=96))):
        with pytest.raises(ops().KernelError):
            call(a, w, y, **kw)
    assert not ops().gemm_groups_ok(z(4, 64), z(4, 16), 4, 16, 64, ops().gate_code("relu")[0])
    assert not ops().gemm_groups_ok(z(4, 64), z(4, 18)[:, :16], 4, 16, 64, 0) and ops().gemm_groups_ok(z(4, 64), z(4, 16), 4, 16, 64, 1)


def test_choice_of_waves_and_height():
    """Sizes that were timed: long prompts and short ones, narrow experts, and streams of W that the tiled product keeps."""
    from spite_amd.csrc.hipops import gemm_groups_choice
    at = lambda T, E, top, whole, N, K, glu: gemm_groups_choice(T, E, T * top / E, whole, N, K, glu)
    assert at(2048, 16, 1, 1, 8192, 5120, True) == (8, 160) and at(1547, 16, 1, 1, 8192, 5120, True) == (8, 128)
    assert at(330, 16, 1, 1, 8192, 5120, True)[0] == 4 and at(1531, 16, 4, 2, 1024, 2048, True) == (4, 128)
    assert at(1200, 16, 1, 1, 2048, 3072, False)[0] == 4
    for T in (69, 228, 425):
        assert at(T, 16, 1, 1, 5120, 8192, False) is None
    assert at(300, 4, 1, 0, 1216, 4416, False) == (4, 128) and gemm_groups_choice(0, 16, 0.0, 0, 64, 64, False) is None


@pytest.mark.gpu
@pytest.mark.parametrize("waves,cap", [(4, 128), (8, 160)])
@pytest.mark.parametrize("G,rows", [(1, [300]), (9, [0] * 8 + [5]), (64, [0, 0, 161] + [0] * 60 + [40]), (65, [1] * 65), (200, [0] * 70 + [3] + [0] * 128 + [170]),
                                    (129, [0] * 129)])
def test_groups_of_which_few_hold_rows(waves, cap, G, rows):
    """The launch is sized by the rows and the number of groups; what holds rows is found among them, and nothing else is written."""
    M, N, K = sum(rows), 272, 128
    a, w = rnd(max(M, 1), K, dtype=torch.bfloat16), ops().operand_order(rnd(G, N, K, dtype=torch.bfloat16, seed=1))
    offsets = torch.tensor([sum(rows[:g]) for g in range(G + 1)], dtype=torch.int32, device=DEV)
    M = M + 200                                                  # room for more rows than the offsets name
    a = torch.cat([a, rnd(200, K, dtype=torch.bfloat16, seed=2)])
    y, z = torch.full((M, N), 7.0, device=DEV), torch.full((M, N), 7.0, device=DEV)
    ops().gemm_tiled(a, w, y, M, N, K, offsets=offsets, n_groups=G, shape=1)
    ops().gemm_groups(a, w, z, M, N, K, offsets=offsets, n_groups=G, waves=waves, cap=cap)
    assert torch.equal(y, z) and (z[sum(rows):] == 7.0).all()


def test_choice_against_the_product_that_would_run_otherwise():
    """Sizes at which every kernel was timed: the tiled product with its own tile, or both operands in LDS, was 6 to 26 % faster than the
    tiles that an estimate without it had taken; and sizes that stay with them."""
    from spite_amd.csrc.hipops import gemm_groups_choice
    from spite_amd.parts.linear import grouped_tile_shape

    def at(T, E, top, whole, N, K, glu, lds=False):
        shape = grouped_tile_shape(T, E, whole, col_tiles=-(-N // (256 if glu else 512))) if top == 1 else 0
        return gemm_groups_choice(T, E, T * top / E, whole, N, K, glu, shape, lds)

    for tiled in ((1237, 16, 1, 1, 3072, 2048, False), (1512, 16, 1, 1, 3072, 2048, False), (1042, 16, 1, 1, 3072, 8192, False),
                  (2189, 32, 1, 1, 768, 14336, True), (1040, 64, 2, 1, 512, 8192, True), (686, 32, 1, 1, 1024, 16384, True),
                  (88, 16, 1, 1, 3072, 4096, True), (897, 16, 1, 1, 4096, 14336, False)):
        assert at(*tiled) is None, tiled
    for in_lds in ((838, 8, 2, 1, 1536, 16384, True), (212, 4, 4, 2, 6144, 16384, False), (402, 16, 8, 2, 1024, 8192, True),
                   (1376, 64, 8, 2, 512, 16384, False)):
        assert at(*in_lds, lds=True) is None, in_lds
    assert at(2048, 16, 1, 1, 8192, 5120, True) == (8, 160) and at(1531, 16, 4, 2, 1024, 2048, True) == (4, 128)
    assert at(126, 4, 4, 1, 5120, 16384, True) == (4, 128) and at(1483, 32, 8, 1, 768, 16384, False) == (8, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("waves,cap", [(4, 128), (4, 160), (8, 128), (8, 160)])
def test_row_lists_scales_and_scattered_rows_equal_the_tiled_product(glu, out_dtype, waves, cap):
    M, N, K, G = sum(HEIGHTS), 272, 192, len(HEIGHTS)
    g = torch.Generator().manual_seed(3)
    a, w = rnd(M + 3, K, dtype=torch.bfloat16), ops().operand_order(rnd(G, 2 * N if glu else N, K, dtype=torch.bfloat16, seed=1))
    kw = dict(offsets=torch.tensor([sum(HEIGHTS[:g]) for g in range(G + 1)], dtype=torch.int32, device=DEV), n_groups=G, glu=glu,
              a_rows=torch.randint(0, M + 3, (M,), generator=g).to(torch.int32).to(DEV), a_scale=(torch.rand(M, generator=g) + 0.5).to(DEV),
              y_rows=torch.randperm(M + 2, generator=g)[:M].to(torch.int32).to(DEV))
    y, z = torch.zeros(M + 2, N, dtype=out_dtype, device=DEV), torch.zeros(M + 2, N, dtype=out_dtype, device=DEV)
    ops().gemm_tiled(a, w, y, M, N, K, shape=1, **kw)
    ops().gemm_groups(a, w, z, M, N, K, waves=waves, cap=cap, **kw)
    assert torch.equal(y, z)
