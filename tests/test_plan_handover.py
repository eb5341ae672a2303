"""The row list that a norm may make for the feed-forward behind it: handed over only between parts whose ``forward`` takes it."""
import pytest
import torch

from spite_amd.engine.context import Env, HostBatch, StepContext, Workspace
from spite_amd.parts.block import PreNormBlock, takes_plan
from spite_amd.parts.feed_forward import DenseGLU, MoeTop1Sigmoid
from spite_amd.parts.norm import RMSNorm

CPU = torch.device("cpu")


class OwnNorm(RMSNorm):
    """A norm with the ``forward`` that a norm had before there were plans."""

    def forward(self, h, out, *, d1=None, d2=None, out32=None, rows=None, write_h=True, proj=None, proj_out=None):
        proj_out.copy_(h @ proj.T)


class OwnMoe(MoeTop1Sigmoid):
    """Experts chosen its own way from the logits."""

    def forward(self, x, x32, ctx, projected=None):
        self.seen = projected
        return (torch.zeros(x.shape),)


class Recorder(RMSNorm):
    def forward(self, h, out, *, d1=None, proj=None, proj_out=None, plan=None):
        self.plan = plan
        proj_out.copy_(h @ proj.T)


class RecorderMoe(MoeTop1Sigmoid):
    def forward(self, x, x32, ctx, projected=None, plan=None):
        self.plan, self.seen = plan, projected
        return (torch.zeros(x.shape),)


def step(norm_kind, ffn_kind, T):
    env = Env(torch.float32, CPU)
    block = object.__new__(PreNormBlock)
    block.env, block.norm2 = env, norm_kind(env, 8, 1e-5)
    block.ffn = ffn_kind(env, hidden_size=8, intermediate_size=16, n_experts=4)
    block.ffn.w_router = torch.randn(4, 8, generator=torch.Generator().manual_seed(0))
    block._plans = takes_plan(block.norm2, block.ffn)
    ctx = StepContext(T=T, n_seqs=1, token_ids=None, positions=None, seq_of_token=None, cu_seqlens=None, seq_slots=None,
                      seq_starts=None, logit_rows=None, n_out=0, host=HostBatch(None, None, None, None), ws=Workspace(CPU, 1 << 16))
    h = torch.randn(T, 8)
    block._stage_ffn({"h": h, "mixed": torch.zeros(T, 8)}, ctx, None)
    assert torch.equal(block.ffn.seen, h @ block.ffn.w_router.T)
    return block


@pytest.mark.parametrize("T", [1, 2])
@pytest.mark.parametrize("norm,ffn", [(OwnNorm, OwnMoe), (OwnNorm, RecorderMoe), (Recorder, OwnMoe), (Recorder, RecorderMoe)])
def test_parts_with_a_forward_of_their_own(norm, ffn, T):
    block = step(norm, ffn, T)
    both = norm is Recorder and ffn is RecorderMoe and T == 1
    for part in (block.norm2, block.ffn):
        assert (getattr(part, "plan", None) is not None) == both


def test_which_parts_take_a_plan():
    env = Env(torch.float32, CPU)
    norm = RMSNorm(env, 8, 1e-5)
    assert takes_plan(norm, MoeTop1Sigmoid(env, 8, 16, 4)) and not takes_plan(norm, DenseGLU(env, 8, 16))
