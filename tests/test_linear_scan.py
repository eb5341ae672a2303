"""The linear recurrence: a request's tokens taken in blocks give the bits of the same tokens taken one by one."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["channel", "head", "bonus"])
@pytest.mark.parametrize("H,D,V,dtype", [(2, 6, 10, torch.float32), (2, 64, 40, torch.bfloat16), (1, 128, 128, torch.bfloat16),
                                         (1, 130, 20, torch.bfloat16), (1, 256, 72, torch.bfloat16)])
@pytest.mark.parametrize("lens", [[1, 7, 16], [8, 9, 15], [17, 33]])
def test_blocks_of_tokens_match_single_tokens(kind, H, D, V, dtype, lens):
    """Blocks hold 16 tokens (8 for the widest heads): lengths below, at and above them.  Each token's sums run over the
    same pairs of lanes whichever of the two kernels takes them, so results and states are equal, not close."""
    from spite_amd.csrc import hipops
    torch.manual_seed(D + V)
    n, T = len(lens), sum(lens)
    row = (torch.randn(T, H * (2 * D + V), device="cuda") * 0.5).to(dtype)
    q, k, v = row[:, :H * D], row[:, H * D:2 * H * D], row[:, 2 * H * D:]
    opt = dict(decay=torch.rand(T, H * D, device="cuda")) if kind != "head" else dict(head_decay=torch.rand(H, device="cuda"))
    if kind == "bonus":
        opt["bonus"] = torch.randn(H, D, device="cuda")
    start = torch.randn(n, H, D, V, device="cuda")
    slots = torch.arange(n, dtype=torch.int32, device="cuda")
    first = [sum(lens[:i]) for i in range(n + 1)]
    whole, s_whole = torch.empty(T, H * V, device="cuda"), start.clone()
    hipops.linear_attn_scan(q, k, v, whole, s_whole, torch.tensor(first, dtype=torch.int32, device="cuda"), slots, n, H, D, V, **opt)
    single, s_single = torch.empty(T, H * V, device="cuda"), start.clone()
    one = torch.tensor([0, 1], dtype=torch.int32, device="cuda")
    for i in range(n):
        for t in range(first[i], first[i + 1]):
            cut = dict(opt, decay=opt["decay"][t:t + 1]) if "decay" in opt else opt
            hipops.linear_attn_scan(q[t:t + 1], k[t:t + 1], v[t:t + 1], single[t:t + 1], s_single, one, slots[i:i + 1], 1, H, D, V,
                                    longest=1, **cut)
    assert torch.equal(whole, single) and torch.equal(s_whole, s_single)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["channel", "head"])
@pytest.mark.parametrize("D,V,dtype", [(6, 10, torch.float32), (24, 40, torch.bfloat16), (72, 24, torch.bfloat16), (130, 20, torch.bfloat16)])
@pytest.mark.parametrize("T", [1, 16, 37])
def test_a_head_takes_nothing_from_its_neighbours(kind, D, V, dtype, T):
    """Heads that fill no whole row of lanes: what lies beside a head in q, k, v and the decay, and beyond the last token, is
    not a number, and neither the head's results nor its state may differ from those of a batch that holds only numbers."""
    from spite_amd.csrc import hipops
    torch.manual_seed(D * T)
    H, pad = 3, 20
    numbers = (torch.randn(T + pad, H * (2 * D + V), device="cuda") * 0.5).to(dtype)
    decay = torch.rand(T + pad, H * D, device="cuda")
    start = torch.randn(1, H, D, V, device="cuda")
    cu, slot = torch.tensor([0, T], dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    got = []
    for spoil in (False, True):
        row, a = numbers.clone(), decay.clone()
        if spoil:                                   # heads 0 and 2, and every row past the request's last
            for part, w in ((row[:, :H * D], D), (row[:, H * D:2 * H * D], D), (row[:, 2 * H * D:], V), (a, D)):
                part[:, :w] = part[:, 2 * w:] = float("nan")
                part[T:] = float("nan")
        opt = dict(decay=a[:T]) if kind == "channel" else dict(head_decay=torch.full((H,), 0.75, device="cuda"))
        out, state = torch.zeros(T, H * V, device="cuda"), start.clone()
        hipops.linear_attn_scan(row[:T, :H * D], row[:T, H * D:2 * H * D], row[:T, 2 * H * D:], out, state, cu, slot, 1, H, D, V, **opt)
        got.append((out[:, V:2 * V].clone(), state[:, 1].clone()))
    assert torch.isfinite(got[0][0]).all() and torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["channel", "head", "bonus"])
@pytest.mark.parametrize("H,D,V,lens", [(4, 64, 64, [1, 7, 16, 17, 0, 40] * 7), (4, 24, 40, [33, 2, 16, 15, 5] * 9), (40, 8, 8, [16, 1, 3, 0, 9] * 3),
                                        (3, 56, 24, [1, 7, 16, 3])])
def test_narrow_heads_of_many_or_short_entries(kind, H, D, V, lens):
    """Heads of up to 64 take their blocks another way where workgroups are many or entries short: the bits of the same requests one
    at a time, with factors on the values and q and k heads shared, and nothing from rows that no entry has."""
    from spite_amd.csrc import hipops
    torch.manual_seed(D + V)
    n, T, pad, share = len(lens), sum(lens), 20, 1 if H % 2 else 2
    first = [sum(lens[:i]) for i in range(n + 1)]
    row = (torch.randn(T + pad, H // share * 2 * D + H * V, device="cuda") * 0.5).bfloat16()
    decay, vs = torch.rand(T + pad, H * D, device="cuda"), torch.rand(T + pad, H, device="cuda")
    row[T:] = decay[T:] = vs[T:] = float("nan")
    w = H // share * D
    q, k, v = row[:, :w], row[:, w:2 * w], row[:, 2 * w:]
    opt = dict(qk_heads=H // share)
    if kind == "bonus":
        opt["bonus"] = torch.randn(H, D, device="cuda")
    each = dict(head_decay=torch.rand(H, device="cuda")) if kind == "head" else None
    start = torch.randn(n, H, D, V, device="cuda")
    slots = torch.randperm(n, device="cuda").int()
    whole, s_whole = torch.empty(T, H * V, device="cuda"), start.clone()
    hipops.linear_attn_scan(q[:T], k[:T], v[:T], whole, s_whole, torch.tensor(first, dtype=torch.int32, device="cuda"), slots, n, H, D, V,
                            longest=max(lens), v_scale=vs[:T], **(each or dict(decay=decay[:T])), **opt)
    alone, s_alone = torch.empty(T, H * V, device="cuda"), start.clone()
    for i in range(n):
        a, b = first[i], first[i + 1]
        if a < b:                                    # (a length that is not known: the scan)
            hipops.linear_attn_scan(q[a:b], k[a:b], v[a:b], alone[a:b], s_alone, torch.tensor([0, b - a], dtype=torch.int32, device="cuda"),
                                    slots[i:i + 1], 1, H, D, V, v_scale=vs[a:b], **(each or dict(decay=decay[a:b])), **opt)
    assert torch.isfinite(whole).all() and torch.equal(whole, alone) and torch.equal(s_whole, s_alone)
