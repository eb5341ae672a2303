"""The 32-bit product on the matrix units and the 32-bit attention over tiles of keys, at the edges of their tiles."""
import math

import pytest
import torch

from test_kernels import DEV, PagedKV, attention_reference, ops, plain_first, rnd, run_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 16, 4), (16, 17, 36), (17, 64, 260), (33, 100, 2048), (64, 30, 1028), (65, 64, 288),
                                   (130, 129, 36), (301, 80, 2052)])
@pytest.mark.parametrize("glu,grouped", [(False, False), (True, False), (True, True)])
def test_product_at_the_edges_of_its_tiles(M, N, K, glu, grouped):
    run_gemm(ops().gemm_generic, torch.float32, torch.float32, M, N, K, glu, grouped)


@pytest.mark.parametrize("K", [36, 2048, 3072])
@pytest.mark.parametrize("glu", [False, True])
def test_a_row_has_the_same_bits_alone_and_among_many(K, glu):
    M, N = 150, 96
    a, w = rnd(M, K), rnd(2 * N if glu else N, K, seed=1)
    whole = torch.empty(M, N, device=DEV)
    ops().gemm_generic(a, w, whole, M, N, K, glu=glu)
    for first, rows in ((0, 1), (3, 16), (20, 40), (70, 64), (85, 65)):
        part = torch.empty(rows, N, device=DEV)
        ops().gemm_generic(a[first:first + rows].contiguous(), w, part, rows, N, K, glu=glu)
        assert torch.equal(part, whole[first:first + rows]), (first, rows)


def test_the_sum_is_no_less_exact_than_an_ascending_chain():
    """Against 64 bits, beside a chain of FMAs over k in ascending order (each step rounded once, formed in float64)."""
    M, N, K = 70, 64, 2048
    a, w = rnd(M, K), rnd(N, K, seed=1)
    y = torch.empty(M, N, device=DEV)
    ops().gemm_generic(a, w, y, M, N, K)
    ref = a.double() @ w.double().T
    chain = torch.zeros(M, N, device=DEV)
    for k in range(K):
        chain = (chain.double() + a[:, k:k + 1].double() * w[:, k].double()).float()
    off = lambda z: float((z.double() - ref).pow(2).mean().sqrt())
    assert off(y) <= off(chain)


@pytest.mark.parametrize("H,G,hd,ps,vis,span", [(4, 2, 16, 4, "full", 0), (6, 3, 48, 8, "window", 70), (8, 2, 128, 64, "chunk", 128),
                                                (3, 1, 64, 32, "window", 1), (4, 4, 128, 64, "window", 300)])
def test_attention_over_tiles_of_32_keys(H, G, hd, ps, vis, span):
    lens = [330, 64, 1]
    queries = [(0, 329), (0, 63), (0, 64), (0, 127), (0, 128), (0, 255), (0, 256), (0, 300), (1, 63), (1, 0), (2, 0)]
    kv = PagedKV(lens, G, hd, ps, torch.float32)
    qs = torch.randn(len(queries), H, hd, generator=torch.Generator().manual_seed(2))
    ref = attention_reference(kv, queries, qs, H, vis, span)
    scale = 1.0 / math.sqrt(hd)

    def attend(which, kp, vp):
        out = torch.zeros(len(which), H * hd, device=DEV)
        pos = torch.tensor([queries[i][1] for i in which], dtype=torch.int32, device=DEV)
        seq = torch.tensor([queries[i][0] for i in which], dtype=torch.int32, device=DEV)
        ops().attn_generic(qs[which].reshape(len(which), H * hd).to(DEV), kp.to(DEV), vp.to(DEV), out, pos, seq, kv.bt.to(DEV),
                           len(which), H, G, hd, ps, vis, span, scale)
        return out

    every = list(range(len(queries)))
    got = attend(every, kv.kp, kv.vp)
    assert (got.double().cpu().view(len(queries), H, hd) - ref).abs().max() < 2e-5 * max(1.0, float(ref.abs().max()))
    for i in every:
        # the same bits alone, with NaN in every row that the query does not see
        s, p = queries[i]
        kp, vp = torch.full_like(kv.kp, float("nan")), torch.full_like(kv.vp, float("nan"))
        for j in range(plain_first(vis, span, p), p + 1):
            pg, off = kv.tables[s][j // ps], j % ps
            kp[pg, :, off], vp[pg, :, :, off] = kv.kp[pg, :, off], kv.vp[pg, :, :, off]
        assert torch.equal(attend([i], kp, vp)[0], got[i]), queries[i]
