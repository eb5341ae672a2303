"""Which of the 32-bit products a call takes, and the same bits from each of them."""
import pytest
import torch

from test_kernels import DEV, ops, rnd, run_gemm


def test_lines_lie_where_both_sides_were_timed():
    from spite_amd.csrc.hipops import lib
    at = lib().spite_gemm_f32_variant
    assert [at(2 * t, 3072, 17) for t in (1, 16, 32, 64, 68, 150, 200)] == [16, 16, 16, 16, 16, -32, -64]
    assert [at(m, 32768, 0) for m in (1, 8, 9, 64, 65, 100)] == [16, 16, -32, -32, -64, -64]
    assert [at(m, 3072, 0) for m in (16, 17, 64, 65, 301)] == [16, 32, 64, -32, -32]
    assert at(400000, 64, 50000) == -64 and at(64, 64, 2) == 64

    at = lib().spite_gemm_f32_choice             # 8: a workgroup takes eight columns of each half
    assert [at(2 * t, 2048, k, 129, 0) for t in (107, 267) for k in (768, 1024, 1536, 2048)] == [-32, -32, -32, 16] * 2
    assert [at(120, 1024, k, 33, 1) for k in (512, 768)] == [-32, 16] and at(20, 256, 512, 4, 1) == 8
    assert [at(m, 16384, 2048, 0, 1) for m in (64, 65, 166)] == [-32, -64, -64]
    assert [at(m, 16384, 2048, 0, 0) for m in (65, 96, 97, 186)] == [-32, -32, -64, -64]
    assert [at(m, 6144, 2048, 0, 1) for m in (158, 161)] == [-32, -64]
    assert [at(1908, 512, 2048, 9, g) for g in (0, 1)] == [-32, -32] and at(3000, 1536, 2048, 65, 1) == -64
    assert [at(1, 6144, k, 0, 1) for k in (512, 2047, 2048)] == [16, 16, 8] and at(1, 4096, 128, 0, 1) == 8 and at(1, 4100, 2048, 0, 1) == 16


def test_lines_of_17_to_64_rows():
    """Both sides timed with the tiles as they are: the stream of 16 rows up to four workgroups a compute unit, without groups three and
    a half and below one; then tiles of 32 (48 rows of 5 groups x 3,072 x 2,048: 30 us, 64 rows a workgroup of the stream 63)."""
    from spite_amd.csrc.hipops import lib
    at = lib().spite_gemm_f32_choice
    assert [at(48, n, 2048, 5, 0) for n in (1024, 2048, 3072)] == [16, 16, -32] and [at(m, 3072, 2048, 5, 1) for m in (40, 48, 64)] == [16, -32, -32]
    assert [at(m, 5120, 5120, 3, 0) for m in (25, 34, 64)] == [16, -32, -32] and at(64, 6144, 768, 5, 1) == -32 and at(64, 768, 512, 5, 0) == 16
    assert [at(m, 1024, 1024, 0, 0) for m in (17, 64)] == [16, 16] and [at(m, 5120, 5120, 0, 0) for m in (32, 33, 64)] == [32, -32, -32]
    assert [at(m, 3072, 2048, 0, 0) for m in (17, 33, 64)] == [32, 64, 64] and at(64, 200, 2048, 5, 0) == 64


@pytest.mark.gpu
@pytest.mark.parametrize("M,groups", [(200, 40), (70, 5), (300, 5), (40, 3)])
@pytest.mark.parametrize("N,K,glu", [(80, 292, False), (80, 292, True), (16400, 36, False)])
def test_groups(M, groups, N, K, glu):
    run_gemm(ops().gemm_generic, torch.float32, torch.float32, M, N, K, glu, True, groups)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17, 32, 33, 48, 49, 64, 65, 100])
def test_a_row_of_a_tall_matrix_has_the_same_bits_in_every_variant(rows):
    N, K = 16400 * 2, 132
    a, w = rnd(130, K), rnd(N, K, seed=1)
    whole, part = torch.empty(130, N, device=DEV), torch.empty(rows, N, device=DEV)
    ops().gemm_generic(a, w, whole, 130, N, K)
    ops().gemm_generic(a[:rows].contiguous(), w, part, rows, N, K)
    narrow = torch.empty(rows, 48, device=DEV)
    ops().gemm_generic(a[:rows].contiguous(), w[:48].contiguous(), narrow, rows, 48, K)
    assert torch.equal(part, whole[:rows]) and torch.equal(narrow, whole[:rows, :48])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 36), (5, 24, 516), (16, 2056, 260), (3, 20, 64)])
@pytest.mark.parametrize("groups", [0, 4])
def test_gated_rows_with_both_halves_in_one_operand(M, N, K, groups):
    """Eight columns a workgroup (N a multiple of 8) and sixteen, the last ones part of their tile."""
    run_gemm(ops().gemm_generic, torch.float32, torch.float32, M, N, K, True, groups > 0, max(groups, 1))
    a, w = rnd(M, K), rnd(2 * N, K, seed=1)
    y, many = torch.empty(M, N, device=DEV), torch.empty(M + 100, N, device=DEV)
    ops().gemm_generic(a, w, y, M, N, K, glu=True)
    ops().gemm_generic(torch.cat([a, rnd(100, K, seed=3)]), w, many, M + 100, N, K, glu=True)
    assert torch.equal(y, many[:M])


@pytest.mark.gpu
@pytest.mark.parametrize("K", [4, 60, 64, 68, 128, 188, 192, 256, 260, 320, 384, 388, 448, 516, 580, 772])
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("M,N", [(90, 200), (75, 33000)])
def test_tiles_add_up_in_the_streams_order_wherever_the_sum_ends(K, glu, M, N):
    """Sums that end inside a step, with one, with the steps whose loads would pass the end: a row of a tile (of 32 rows, of
    64) has the bits that the stream gives it alone, and a row of a tile of 32 among groups of one to forty rows."""
    a, w = rnd(M, K), rnd((2 if glu else 1) * N, K, seed=1)
    whole, one = torch.empty(M, N, device=DEV), torch.empty(1, N, device=DEV)
    ops().gemm_generic(a, w, whole, M, N, K, glu=glu)
    for r in (0, 15, 16, 63, 64, M - 1):
        ops().gemm_generic(a[r:r + 1].contiguous(), w, one, 1, N, K, glu=glu)
        assert torch.equal(one[0], whole[r])
    N = min(N, 1024)
    sizes = [1, 17, 33, 0, 16, 40, 8, 3]
    offsets = torch.tensor([0] + list(torch.tensor(sizes).cumsum(0)), dtype=torch.int32, device=DEV)
    n = sum(sizes)
    x, ws = rnd(n, K, seed=5), rnd(len(sizes), (2 if glu else 1) * N, K, seed=6)
    y = torch.empty(n, N, device=DEV)
    ops().gemm_generic(x, ws, y, n, N, K, glu=glu, offsets=offsets, n_groups=len(sizes))
    at = 0
    for g, size in enumerate(sizes):
        for r in {at, at + size - 1} if size else ():
            alone = torch.empty(1, N, device=DEV)
            ops().gemm_generic(x[r:r + 1].contiguous(), ws[g].contiguous(), alone, 1, N, K, glu=glu)
            assert torch.equal(alone[0], y[r])
        at += size


@pytest.mark.gpu
@pytest.mark.parametrize("K", [4, 60, 64, 68, 128, 188, 192, 256, 260, 320, 384, 388, 448, 516, 580, 772])
@pytest.mark.parametrize("glu,N,sizes", [(True, 3000, [1, 17, 33, 0, 49, 64, 40, 60, 65]), (False, 2100, [1, 17, 33, 49, 1000])])
def test_groups_in_tiles_of_64_rows_wherever_the_sum_ends(K, glu, N, sizes):
    """Tiles of 64 rows over groups: one to four live quarters, both loops over k, sums that end anywhere in a step; the choice is
    asserted, so that the case stays on the kernel that it is for.  A row has the bits that the stream gives it alone."""
    from spite_amd.csrc.hipops import lib
    n, ng = sum(sizes), len(sizes)
    assert lib().spite_gemm_f32_choice(n, N, K, ng, int(glu)) == -64
    offsets = torch.tensor([0] + list(torch.tensor(sizes).cumsum(0)), dtype=torch.int32, device=DEV)
    x, ws = rnd(n, K, seed=5), rnd(ng, (2 if glu else 1) * N, K, seed=6)
    y = torch.empty(n, N, device=DEV)
    ops().gemm_generic(x, ws, y, n, N, K, glu=glu, offsets=offsets, n_groups=ng)
    at = 0
    for g, size in enumerate(sizes):
        for r in {at, at + size // 2, at + size - 1} if size else ():
            alone = torch.empty(1, N, device=DEV)
            ops().gemm_generic(x[r:r + 1].contiguous(), ws[g].contiguous(), alone, 1, N, K, glu=glu)
            assert torch.equal(alone[0], y[r]), (g, r - at)
        at += size
