"""Rows a workgroup of the residual add and norm, and whether it asks for every load ahead: the lines, and the same bits on both
sides of each."""
import pytest
import torch

from test_kernels import DEV, ops, rnd


def test_lines_lie_where_both_sides_were_timed():
    from spite_amd.csrc.hipops import lib
    at = lambda n, d, P=0: (lib().spite_add_rmsnorm_variant(n, d, P) % 256, lib().spite_add_rmsnorm_variant(n, d, P) >= 256)
    # wide rows: ahead up to a row a compute unit
    assert [at(n, 12288)[1] for n in (1, 256, 257, 2048)] == [True, True, False, False]
    assert at(2048, 8192) == (1, True) and at(300, 8196, 16) == (1, False)
    # two rows a workgroup
    assert {at(n, d, P)[0] for n in (257, 700, 2048) for d in (1024, 2048) for P in (16, 128, 256)} == {1}
    assert [at(n, 2560, 16)[0] for n in (330, 512, 513, 2048)] == [1, 1, 2, 2] and at(2048, 2560, 4)[0] == 1
    assert [at(330, d, 128)[0] for d in (2304, 2560, 3840)] == [1, 2, 1] and at(330, 3072, 256)[0] == 1
    assert [at(2048, d, 128)[0] for d in (4608, 5120, 6144, 8192)] == [1, 2, 2, 1]
    assert [at(n, 5120, 16)[0] for n in (330, 600, 2048)] == [1, 1, 1] and [at(n, 5120, 64)[0] for n in (256, 330, 600, 2048)] == [1, 2, 1, 2]
    assert at(600, 6144, 128)[0] == 1 and at(600, 5120, 128)[0] == 2
    assert at(2048, 5120) == (1, True)                          # nothing to share without a projection


@pytest.mark.gpu
@pytest.mark.parametrize("d,rows,P", [(8196, 257, 0), (10240, 300, 5), (12288, 258, 17), (16384, 259, 0), (2560, 515, 16), (2560, 301, 65),
                                      (5120, 331, 64), (6144, 259, 64), (4100, 515, 16)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_a_row_alone_and_among_many(d, rows, P, dtype):
    h, d1, d2, dn = (rnd(rows, d, seed=i) for i in range(4))
    w, wn, w2 = (rnd(d, seed=10 + i) + 2.0 for i in range(3))
    proj = rnd(P, d, seed=20) if P else None
    at = torch.randperm(rows, generator=torch.Generator().manual_seed(0)).to(torch.int32).to(DEV)

    def run(n, **kw):
        part = lambda t: t[-n:].clone()
        hh, out, out2 = part(h), torch.empty(n, d, dtype=dtype, device=DEV), torch.empty(n, d, dtype=dtype, device=DEV)
        out32, logits = torch.empty(n, d, device=DEV), torch.empty(n, max(P, 1), device=DEV)
        if P:
            kw.update(proj=proj, proj_out=logits)
        ops().add_rmsnorm(hh, w, 1e-5, out=out, out32=out32, d1=part(d1), d2=part(d2), normed=(part(dn), wn, 0.5, 1e-6), w2=w2, out2=out2, **kw)
        return [hh, out, out32, out2] + ([logits] if P else [])

    got = run(rows)
    for n in (1, 2, 3):
        for g, alone in zip(got, run(n)):
            assert torch.equal(g[-n:], alone), n
    for g, listed in zip(got[1:], run(rows, rows=at, write_h=False)[1:]):
        assert torch.equal(g[at.long()], listed)
    D = dn.double()
    v = h.double() + d1.double() + d2.double() + 0.5 * D / (D.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * wn.double()
    want = v / (v.pow(2).mean(1, keepdim=True) + 1e-5).sqrt()
    # fp32 sums of d terms in a tree
    assert ((got[2].double() - want * w.double()).abs() <= 2e-6 * (want * w.double()).abs().max()).all()
    if P:
        ref = (want * w.double()) @ proj.double().T
        assert ((got[4].double() - ref).abs() <= 4e-6 * d ** 0.5 * ref.abs().max()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("d,rows", [(2048, 3), (2046, 3), (12288, 300)])
def test_the_second_output_alone_needs_no_first_weight(d, rows):
    h, w, w2 = rnd(rows, d), rnd(d, seed=1) + 2.0, rnd(d, seed=2) + 2.0
    got, both, out = (torch.empty(rows, d, dtype=torch.bfloat16, device=DEV) for _ in range(3))
    ops().add_rmsnorm(h, None, 1e-5, w2=w2, out2=got)
    ops().add_rmsnorm(h, w, 1e-5, out=out, w2=w2, out2=both)
    assert torch.equal(got, both)


@pytest.mark.gpu
@pytest.mark.parametrize("d,P", [(516, 17), (2048, 17), (2048, 130), (5120, 64), (5120, 130), (8192, 16), (9216, 5)])
@pytest.mark.parametrize("rows", [1, 255, 256, 331])
def test_logits_are_the_routers(d, P, rows):
    """Two rows of the projection a wave, two rows a workgroup, four tokens a workgroup of the router (from 256 on), and one."""
    h, w, proj = rnd(rows, d), rnd(d, seed=1) + 2.0, rnd(P, d, seed=2)
    out32, logits, again = torch.empty(rows, d, device=DEV), torch.empty(rows, P, device=DEV), torch.empty(rows, P, device=DEV)
    ops().add_rmsnorm(h, w, 1e-5, out32=out32, proj=proj, proj_out=logits)
    expert, weight = torch.empty(rows, dtype=torch.int32, device=DEV), torch.empty(rows, device=DEV)
    ops().router_top1(out32, proj, expert, weight, again)
    assert torch.equal(logits, again)
    exact, size = out32.double() @ proj.double().T, out32.double().abs() @ proj.double().abs().T
    # a lane adds d/256 fours of four roundings each, then six steps of the butterfly
    assert ((logits.double() - exact).abs() <= (d / 256 + 11) * 2.0 ** -24 * size).all()
