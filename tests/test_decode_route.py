"""Which of the two ways a step of decoded tokens goes through its attention."""
import pytest
import torch


def test_the_rule():
    from spite_amd.csrc.hipops import attn_decode_rope_suits, cu_count
    cus = cu_count()
    assert attn_decode_rope_suits(1) and attn_decode_rope_suits(2 * cus) and not attn_decode_rope_suits(2 * cus + 1)


@pytest.mark.gpu
def test_both_ways_give_the_same_logits(monkeypatch):
    """A batch on either side of the rule's line: the pages are the same, the logits differ by the rounding of a query."""
    from spite_amd import Engine, StepEntry
    from spite_amd.csrc import hipops
    cfg = dict(architectures=["Llama4ForCausalLM"], num_hidden_layers=2, hidden_size=256, num_attention_heads=4, num_key_value_heads=2,
               head_dim=64, rms_norm_eps=1e-5, num_local_experts=4, num_experts_per_tok=1, intermediate_size=512,
               intermediate_size_mlp=1024, interleave_moe_layer_step=2, vocab_size=512, rope_theta=1e4, torch_dtype="bfloat16")
    out, fused = [], []
    run = hipops.attn_decode_rope
    for suits in (True, False):
        calls = []
        monkeypatch.setattr(hipops, "attn_decode_rope_suits", lambda heads: suits)
        monkeypatch.setattr(hipops, "attn_decode_rope", lambda *a, **kw: (calls.append(1), run(*a, **kw))[1])
        eng = Engine(cfg, random_weights=True, seed=3, cache_tokens=512, max_requests=3)
        slots = [eng.admit() for _ in range(3)]
        g = torch.Generator().manual_seed(1)
        eng.step([StepEntry(s, torch.randint(0, 512, (n,), generator=g).tolist(), [n - 1]) for s, n in zip(slots, (5, 33, 70))])
        out.append(eng.step([StepEntry(s, [7 + s], [0]) for s in slots]).clone())
        fused.append(len(calls))
    assert fused == [2, 0]
    assert (out[0].float() - out[1].float()).abs().max() <= 2e-2 * out[1].float().abs().max()
