"""When a shared expert becomes groups of the routed experts' products, and when it keeps products of its own."""
import pytest
import torch

from spite_amd.engine.context import Env
from spite_amd.parts.feed_forward import MoeTopKSigmoid


def groups_of(F, Fs, dtype=torch.bfloat16):
    d, E = 64, 3
    part = MoeTopKSigmoid(Env(dtype, torch.device("cpu")), d, F, E, 2, Fs, score_bias=False)
    t = {"router": torch.zeros(E, d)}
    for e in [f"e{e}" for e in range(E)] + ["shared"]:
        n = Fs if e == "shared" else F
        t[f"{e}.gate"], t[f"{e}.up"], t[f"{e}.down"] = (torch.zeros(s, dtype=dtype) for s in ((n, d), (n, d), (d, n)))
    part.load(t)
    assert (part.ws_down is None) == (part.shared_groups > 0) and part.w_down.shape[0] == E + part.shared_groups
    return part.shared_groups


@pytest.mark.parametrize("F,Fs,m", [(64, 64, 1), (64, 128, 2), (64, 192, 0), (64, 256, 0), (64, 96, 0)])
def test_up_to_two_groups(F, Fs, m):
    """From three on the rows that the product back writes for each cost long prompts more than the launches they save."""
    assert groups_of(F, Fs) == m


@pytest.mark.parametrize("F,Fs,m", [(20, 40, 0), (24, 48, 0), (32, 64, 0), (96, 192, 0), (40, 80, 0), (48, 96, 2), (12, 24, 0), (10, 20, 0), (16, 32, 2), (10, 10, 1)])
def test_no_groups_that_lose_the_matrix_units_or_the_operand_order(F, Fs, m):
    """The whole width is a multiple of 8, 16 or 64 where the groups' width is not: their products would run on plain FMAs,
    or read rows where tiles were."""
    assert groups_of(F, Fs) == m
