"""The product of some tens to hundreds of rows with its sum over k in runs: tile edges in every direction, runs of one step and of
unequal length, against float64; one run bit for bit against the tiled product."""
import pytest
import torch

from test_kernels import DEV, ops, rnd, run_gemm


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (33, 272, 128), (64, 528, 320), (97, 48, 448), (161, 256, 576), (330, 144, 192)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("nb", [2, 4, 5, 6, 7, 8, 9, 10])
def test_plain(M, N, K, out_dtype, nb):
    steps = K // 64
    for runs in {1, 2, 3, steps}:
        if -(-steps // runs) * (runs - 1) >= steps and runs > 1:
            continue

        def fn(a, w, y, M, N, K, **kw):
            part = torch.full((runs, M, N), float("nan"), device=DEV) if runs > 1 else None
            ops().gemm_runs(a, ops().operand_order(w), y, M, N, K, runs=runs, nb=nb, part=part)
        run_gemm(fn, torch.bfloat16, out_dtype, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("nb", [2, 7, 10])
def test_one_run_equals_the_tiled_product_and_rows_lie_apart(nb):
    M, N, K = 170, 272, 320
    wide = rnd(M, K + 64, dtype=torch.bfloat16)
    a, w = wide[:, :K], ops().operand_order(rnd(N, K, dtype=torch.bfloat16, seed=1))
    y, z, odd = torch.zeros(M, N, device=DEV), torch.ones(M, N + 4, device=DEV)[:, :N], torch.ones(M, N + 3, device=DEV)[:, :N]
    ops().gemm_tiled(a, w, y, M, N, K, shape=1)
    ops().gemm_runs(torch.full_like(wide, float("nan"))[:, :K], w, z, M, N, K, runs=1, nb=nb)        # what LDS held must not show
    ops().gemm_runs(a, w, z, M, N, K, runs=1, nb=nb)
    assert torch.equal(y, z)
    ops().gemm_runs(a, w, odd, M, N, K, runs=2, nb=nb, part=torch.empty(2, M, N, device=DEV))
    assert (odd - y).abs().max() < 1e-5 * float(y.abs().max()) * K ** 0.5
    with pytest.raises(ops().KernelError):
        ops().gemm_runs(a, w, odd, M, N, K, runs=1, nb=nb)              # rows that no 16-byte store can take
    for kw in (dict(runs=2, nb=nb), dict(runs=4, nb=nb, part=torch.empty(4, M, N, device=DEV)), dict(runs=1, nb=3)):
        with pytest.raises(ops().KernelError):
            ops().gemm_runs(a, w, y, M, N, K, **kw)


def test_choice_where_both_sides_were_timed():
    from spite_amd.csrc.hipops import gemm_runs_choice as at
    assert at(32, 32768, 5120) is None and at(64, 3072, 2048) is None and at(64, 32768, 5120) == (2, 4) and at(64, 5120, 8192) == (12, 4)
    assert at(330, 7168, 5120) == (3, 7) and at(330, 5120, 5120) == (4, 7) and at(500, 5120, 5120) == (3, 8)
    assert at(2048, 5120, 5120) is None and at(2048, 7168, 5120) is None and at(2048, 2048, 16384) is None
    for M, N, K in ((65, 16, 64), (100, 512, 128), (800, 20000, 12000), (1531, 576, 5120)):
        got = at(M, N, K)
        if got is not None:
            steps = K // 64
            assert -(-M // (16 * got[1])) * -(-N // 256) * got[0] <= 256 and (got[0] == 1 or -(-steps // got[0]) * (got[0] - 1) < steps)


@pytest.mark.gpu
def test_tokens_between_the_streams_and_the_prompts():
    """Steps of 33 to 64 rows and of a short prompt through the engine's layers: each row as in a step of its own."""
    from spite_amd import Engine, StepEntry
    cfg = dict(architectures=["Llama4ForCausalLM"], num_hidden_layers=2, hidden_size=256, num_attention_heads=4, num_key_value_heads=2,
               head_dim=64, rms_norm_eps=1e-5, num_local_experts=16, num_experts_per_tok=1, intermediate_size=512,
               intermediate_size_mlp=1024, interleave_moe_layer_step=1, vocab_size=512, rope_theta=1e4, torch_dtype="bfloat16")
    eng = Engine(cfg, random_weights=True, seed=3, cache_tokens=64 * 64, max_requests=64)
    tokens = torch.randint(0, 512, (40, 3), generator=torch.Generator().manual_seed(0)).tolist()
    slots = [eng.admit() for _ in tokens]
    prompt = eng.step([StepEntry(s, t[:2], [1]) for s, t in zip(slots, tokens)]).clone()           # 80 rows
    decode = eng.step([StepEntry(s, t[2:], [0]) for s, t in zip(slots, tokens)]).clone()           # 40 rows
    for s in slots:
        eng.release(s)
    scale = float(decode.float().abs().max())
    for i in (0, 17, 39):
        s = eng.admit()
        one = eng.step([StepEntry(s, tokens[i][:2], [1])]).clone()
        two = eng.step([StepEntry(s, tokens[i][2:], [0])]).clone()
        eng.release(s)
        assert (one[0] - prompt[i]).float().abs().max() < 0.05 * scale and (two[0] - decode[i]).float().abs().max() < 0.05 * scale


def test_many_rows_take_runs_where_that_was_faster():
    """Above 800 rows one run of small tiles was 5 to 26 % slower than the large tiles of the other products, several runs 16 % faster."""
    from spite_amd.csrc.hipops import gemm_runs_choice as at
    for M, N, K in ((1922, 3072, 14336), (2829, 2048, 6144), (1041, 5120, 8192), (1547, 5120, 8192), (1036, 5120, 5120), (2427, 1536, 8192), (1783, 2048, 14336)):
        assert at(M, N, K) is None, (M, N, K)
    for M, N, K, runs in ((900, 1024, 5120, 5), (1531, 576, 5120, 5), (1200, 2048, 4096, 4), (800, 5120, 5120, 2)):
        assert at(M, N, K)[0] == runs, (M, N, K, at(M, N, K))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 64, 768), (40, 32768, 832), (40, 5184, 5120), (100, 272, 1472)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_linear_takes_the_runs(M, N, K, out_dtype, monkeypatch):
    """One run and several, with the partial sums from a workspace and without one, against float64."""
    from spite_amd.parts import linear as parts
    seen, inner = [], ops().gemm_runs
    monkeypatch.setattr(parts.hipops, "gemm_runs", lambda *a, **kw: (seen.append((kw["runs"], kw["part"])), inner(*a, **kw)))

    class Taken(list):
        def take(self, shape, dtype):
            self.append(torch.full(shape, float("nan"), dtype=dtype, device=DEV))
            return self[-1]
    x, w = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, dtype=torch.bfloat16, seed=1)
    y, z, ws = torch.empty(M, N, dtype=out_dtype, device=DEV), torch.empty(M, N, dtype=out_dtype, device=DEV), Taken()
    parts.linear(x, parts.Weight(w), y, ws=ws)
    parts.linear(x, parts.Weight(w), z)
    runs = ops().gemm_runs_choice(M, N, K)[0]
    assert [r for r, _ in seen] == [runs] * 2 and (runs == 1) == (N == 32768) and [tuple(t.shape) for t in ws] == [(runs, M, N)] * (runs > 1)
    assert torch.equal(y, z) and (runs == 1 or seen[0][1] is ws[0])
    exact, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    last = 2.0 ** -8 if out_dtype == torch.bfloat16 else 0.0
    assert ((y.double() - exact).abs() <= size * K * 2.0 ** -24 + exact.abs() * last).all()
