"""Tiles of 320 columns over groups whose sizes the host knows on average alone: the device makes the product where the tiles that there are
fit the rounds that were reckoned with, and leaves the groups to the next product where they do not."""
import pytest
import torch

from test_kernels import DEV, ops, rnd


def fits(rows, cap, cols, rounds, per_xcd=32):
    """Groups of few tiles and larger ones, an eighth of each kind (rounded up) to each of eight dies of 32 compute units."""
    tiles = [-(-r // cap) for r in rows]
    live = sum(t > 0 for t in tiles)
    limit = min(4, 2 * sum(tiles) // live) if live else 0
    few = sum(t for t in tiles if t <= limit) * cols
    return -(-few // 8) + -(-(sum(tiles) * cols - few) // 8) <= rounds * per_xcd


@pytest.mark.gpu
@pytest.mark.parametrize("cap", [128, 160])
@pytest.mark.parametrize("rows,N,rounds", [
    ([20] * 16, 5120, 1), ([20] * 15 + [130], 5120, 1), ([20] * 15 + [170], 5120, 1), ([20] * 17, 5120, 1), ([20] * 17, 5120, 2),
    ([0] * 16, 5120, 1), ([3] * 130, 640, 1), ([3] * 129, 640, 1), ([0] * 100 + [3] * 28, 640, 1), ([1300] + [5] * 20, 2240, 1), ([1300] + [5] * 30, 2240, 1), ([70] * 35, 2240, 1), ([70] * 37, 2240, 1)])
def test_the_tiles_that_there_are_decide(rows, N, rounds, cap):
    M, G, K = max(sum(rows), 1), len(rows), 64
    a, w = rnd(M, K, dtype=torch.bfloat16), ops().operand_order(rnd(G, N, K, dtype=torch.bfloat16, seed=1))
    offsets = torch.tensor([sum(rows[:g]) for g in range(G + 1)], dtype=torch.int32, device=DEV)
    y, z = torch.full((M, N), 7.0, device=DEV), torch.full((M, N), 7.0, device=DEV)
    others = torch.full((G + 2,), -5, dtype=torch.int32, device=DEV)
    ops().gemm_tiled(a, w, y, M, N, K, offsets=offsets, n_groups=G, shape=1)
    ops().gemm_groups(a, w, z, M, N, K, offsets=offsets, n_groups=G, waves=5, cap=cap, rounds=rounds, others=others)
    cus = ops().cu_count()
    taken = fits(rows, cap, -(-N // 320), rounds, cus // 8)
    assert torch.equal(z, y if taken else torch.full_like(y, 7.0))
    assert torch.equal(others[:-1], torch.zeros_like(offsets) if taken else offsets) and others[-1] == -5
    if not taken:
        ops().gemm_tiled(a, w, z, M, N, K, offsets=others, n_groups=G, shape=1)
        assert torch.equal(y, z)


@pytest.mark.gpu
@pytest.mark.parametrize("other", [(8, 128), (4, 160), None])
def test_a_captured_product_follows_the_groups(monkeypatch, other):
    """One graph, replayed with groups that fit, that do not, and none: the bits of the tiled product each time."""
    from spite_amd.csrc import hipops
    from spite_amd.parts.linear import Weight, linear
    M, G, N, K = 400, 16, 5120, 128
    monkeypatch.setattr(hipops, "gemm_groups_wide_estimate", lambda *a: ((5, 160), 1))
    monkeypatch.setattr(hipops, "gemm_groups_choice", lambda *a: other)
    x, w = rnd(M, K, dtype=torch.bfloat16), Weight(rnd(G, N, K, dtype=torch.bfloat16, seed=1))
    assert w.tiled
    sets = [[25] * 16, [200, 200] + [0] * 14, [10] * 15 + [250], [0] * 16, [160] + [16] * 15, [161] + [15] * 14 + [29]]
    at = lambda s: torch.tensor([sum(s[:g]) for g in range(G + 1)], dtype=torch.int32, device=DEV)
    offsets, y = at(sets[0]), torch.zeros(M, N, device=DEV)
    dst = torch.randperm(M, generator=torch.Generator().manual_seed(2)).to(torch.int32).to(DEV)
    run = lambda: linear(x, w, y, offsets=offsets, n_groups=G, max_rows=300, group_rows=25, y_rows=dst)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for s in sets * 2:
        offsets.copy_(at(s))
        y.fill_(7.0)
        graph.replay()
        z = torch.full_like(y, 7.0)
        ops().gemm_tiled(x, w.data, z, M, N, K, offsets=at(s), n_groups=G, y_rows=dst, shape=1)
        assert torch.equal(y, z), s


@pytest.mark.gpu
def test_refusals():
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=DEV)
    o = torch.tensor([0, 4], dtype=torch.int32, device=DEV)
    call = lambda **kw: ops().gemm_groups(z(4, 64), z(1, 32, 64), z(4, 32), 4, 32, 64, offsets=o, n_groups=1, **kw)
    for kw in (dict(waves=8, rounds=1, others=o.clone()), dict(waves=5, others=o.clone()), dict(waves=5, rounds=1, others=o[:1].clone()),
               dict(waves=5, rounds=1, others=o), dict(waves=5, rounds=1, others=o.clone().long())):
        with pytest.raises(ops().KernelError):
            call(**kw)


def test_choice_at_the_edge():
    """16 experts of which an expected one has no more rows than a tile: by chance alone the tiles fit 97 times of 100 at 2,048 tokens, two of three at
    2,200 and less than every other at 2,250; and products too short for a second launch."""
    from spite_amd.csrc.hipops import gemm_groups_wide_estimate
    at = lambda T, E, top, whole, N, K, shape=3: gemm_groups_wide_estimate(T, E, T * top / E, whole, N, K, shape)
    for T in (1441, 1547, 2048, 2200):
        assert at(T, 16, 1, 0, 5120, 8192) == ((5, 160), 1), T
    for T in (2250, 2272, 2300):
        assert at(T, 16, 1, 0, 5120, 8192) == (None, 0), T
    assert at(1350, 16, 2, 0, 5120, 4096, 0) == ((5, 128), 2)           # groups of 169 rows: two tiles, nearly all of them
    for short in ((514, 16, 2, 1, 7168, 768, 0), (211, 32, 8, 0, 5120, 768, 0), (1675, 16, 1, 0, 5120, 1024, 3)):
        assert at(*short) == (None, 0), short
    assert gemm_groups_wide_estimate(0, 16, 0.0, 0, 5120, 8192) == (None, 0)
