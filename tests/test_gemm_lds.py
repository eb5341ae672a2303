"""The product with both operands in LDS: tile edges in every direction, groups of every tile height, against float64 and,
bit for bit, against the tiled product (both add k in the same order)."""
import pytest
import torch

from test_kernels import DEV, ops, rnd, run_gemm

pytestmark = pytest.mark.gpu


def lds(a, w, y, M, N, K, **kw):
    ops().gemm_lds(a, ops().operand_order(w), y, M, N, K, **kw)


@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (96, 272, 128), (129, 256, 192), (161, 528, 64), (257, 48, 320), (300, 144, 512)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("glu,nb", [(False, 0), (True, 0), (False, 4), (False, 5), (True, 6), (False, 8)])
def test_plain(M, N, K, out_dtype, glu, nb):
    run_gemm(lds, torch.bfloat16, out_dtype, M, N, K, glu, False, nb=nb)


@pytest.mark.parametrize("M,N,K,groups", [(70, 48, 64, 5), (400, 272, 128, 3), (900, 144, 192, 4), (9, 16, 64, 70)])
@pytest.mark.parametrize("glu", [False, True])
def test_groups_with_row_lists(M, N, K, groups, glu):
    run_gemm(lds, torch.bfloat16, torch.float32, M, N, K, glu, True, groups)


@pytest.mark.parametrize("glu", [False, True])
def test_groups_of_every_tile_height_equal_the_tiled_product(glu):
    rows = [0, 1, 96, 97, 128, 129, 160, 161, 192, 193, 256, 257, 0, 520]
    M, N, K, G = sum(rows), 272, 192, len(rows)
    a, w = rnd(M, K, dtype=torch.bfloat16), ops().operand_order(rnd(G, 2 * N if glu else N, K, dtype=torch.bfloat16, seed=1))
    offsets = torch.tensor([sum(rows[:g]) for g in range(G + 1)], dtype=torch.int32, device=DEV)
    y, z = torch.zeros(M, N, device=DEV), torch.ones(M, N, device=DEV)
    ops().gemm_tiled(a, w, y, M, N, K, offsets=offsets, n_groups=G, glu=glu, shape=1)
    ops().gemm_lds(a, w, z, M, N, K, offsets=offsets, n_groups=G, glu=glu)
    assert torch.equal(y, z)


@pytest.mark.parametrize("act", ["gelu", "silu"])
def test_activation_and_rows_apart(act):
    M, N, K = 150, 64, 128
    wide = rnd(M, K + 64, dtype=torch.bfloat16)
    a, w = wide[:, :K], ops().operand_order(rnd(N, K, dtype=torch.bfloat16, seed=1))
    out = torch.zeros(2, M, N + 3, device=DEV)                   # rows that no 16-byte store can take
    ops().gemm_tiled(a, w, out[0, :, :N], M, N, K, act=act)
    ops().gemm_lds(a, w, out[1, :, :N], M, N, K, act=act)
    assert torch.equal(out[0], out[1])


def test_refuses_what_it_cannot_do():
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ops().KernelError):
        ops().gemm_lds(z(4, 96), z(16, 96), z(4, 16), 4, 16, 96)           # K no multiple of 64
    with pytest.raises(ops().KernelError):
        ops().gemm_lds(z(4, 64), z(24, 64), z(4, 24), 4, 24, 64)           # N no multiple of 16
    with pytest.raises(ops().KernelError):
        ops().gemm_lds(z(4, 64), z(16, 64), z(4, 16), 4, 16, 64, nb=7)     # no such tile


def test_shared_expert_apart_gives_the_same_logits(monkeypatch):
    """The down product as two (the routed groups, the shared expert with both operands in LDS): the same sums."""
    from spite_amd import Engine, StepEntry
    from spite_amd.parts import feed_forward
    cfg = dict(architectures=["Llama4ForCausalLM"], num_hidden_layers=2, hidden_size=256, num_attention_heads=4, num_key_value_heads=2,
               head_dim=64, rms_norm_eps=1e-5, num_local_experts=4, num_experts_per_tok=1, intermediate_size=512,
               intermediate_size_mlp=1024, interleave_moe_layer_step=1, vocab_size=512, rope_theta=1e4, torch_dtype="bfloat16")
    tokens = torch.randint(0, 512, (300,), generator=torch.Generator().manual_seed(0)).tolist()
    out, calls = [], []
    for shape in (0, 1, 3):
        monkeypatch.setattr(feed_forward, "whole_group_apart", lambda *a: shape)
        eng = Engine(cfg, random_weights=True, seed=3, cache_tokens=512, max_requests=1)
        seen = ops().gemm_lds
        monkeypatch.setattr(ops(), "gemm_lds", lambda *a, **kw: (calls.append(shape), seen(*a, **kw))[1])
        monkeypatch.setattr(ops(), "lds_suits", lambda M, N, K, glu, runs: True)
        out.append(eng.step([StepEntry(eng.admit(), tokens, list(range(300)))]).clone())
        monkeypatch.setattr(ops(), "gemm_lds", seen)
    assert calls.count(1) == calls.count(0) + 2
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
