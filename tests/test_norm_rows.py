"""The residual add and norm at the edges of its groups of loads: widths on both sides of every count a thread, rows one and two a
workgroup, with every increment and output, against float64; and a row's bits alone and among many."""
import pytest
import torch

from test_kernels import DEV, ops, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [4, 2044, 2048, 2052, 4100, 6144, 6148, 8196, 12288])
@pytest.mark.parametrize("rows,P", [(1, 3), (3, 16), (257, 9), (515, 17)])
def test_rows_with_logits(d, rows, P):
    h, d1, d2, dn = (rnd(rows, d, seed=i) for i in range(4))
    w, wn, w2 = (rnd(d, seed=10 + i) + 2.0 for i in range(3))
    proj = rnd(P, d, seed=20)

    def run(n):
        part = lambda t: t[-n:].clone()
        hh, out, out2 = part(h), torch.empty(n, d, dtype=torch.bfloat16, device=DEV), torch.empty(n, d, dtype=torch.bfloat16, device=DEV)
        out32, logits = torch.empty(n, d, device=DEV), torch.empty(n, P, device=DEV)
        ops().add_rmsnorm(hh, w, 1e-5, out=out, out32=out32, d1=part(d1), d2=part(d2), normed=(part(dn), wn, 0.5, 1e-6), proj=proj,
                          proj_out=logits, w2=w2, out2=out2)
        return hh, out32, out, out2, logits

    got = run(rows)
    D = dn.double()
    v = h.double() + d1.double() + d2.double() + 0.5 * D / (D.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * wn.double()
    unit = v / (v.pow(2).mean(1, keepdim=True) + 1e-5).sqrt()
    want = (v, unit * w.double(), unit * w.double(), unit * w2.double(), unit * w.double() @ proj.double().T)
    # fp32 sums of d terms in a tree, and half a unit of bfloat16
    for g, ref, tol in zip(got, want, (1e-6, 2e-6, 2.0 ** -8, 2.0 ** -8, 4e-6 * d ** 0.5)):
        assert ((g.double() - ref).abs() <= tol * ref.abs().max()).all()
    for n in {1, 2, min(rows, 300)} - {rows}:
        if n <= rows:
            for g, part in zip(got, run(n)):
                assert torch.equal(g[-n:], part), n


@pytest.mark.parametrize("d,rows", [(2048, 5), (5120, 300), (16384, 2), (16388, 2)])
def test_rows_by_a_list_and_without_outputs(d, rows):
    h, d1, w = rnd(rows, d), rnd(rows, d, seed=1), rnd(d, seed=2)
    at = torch.randperm(rows, generator=torch.Generator().manual_seed(0)).to(torch.int32).to(DEV)
    out, plain, hh = torch.empty(rows, d, device=DEV), torch.empty(rows, d, device=DEV), h.clone()
    ops().add_rmsnorm(hh, w, 1e-5, out=out, d1=d1, rows=at, write_h=False)
    ops().add_rmsnorm(hh, None, 1e-5, out=plain, d1=d1, plain_out=True, write_h=False)
    assert torch.equal(hh, h) and torch.equal(plain, h + d1)
    v = (h + d1).double()
    want = (v / (v.pow(2).mean(1, keepdim=True) + 1e-5).sqrt() * w.double())[at.long()]
    assert ((out.double() - want).abs() <= 2e-6 * want.abs().max()).all()
    ops().add_rmsnorm(hh, None, 1e-5, d1=d1)
    assert torch.equal(hh, h + d1)


@pytest.mark.parametrize("d", [2048, 5120, 5121])
def test_a_second_norm_beside_a_plain_row(d):
    h, d1, w2 = rnd(3, d), rnd(3, d, seed=1), rnd(d, seed=2)
    plain, out2 = torch.empty(3, d, device=DEV), torch.empty(3, d, device=DEV)
    ops().add_rmsnorm(h, None, 1e-5, out=plain, d1=d1, plain_out=True, w2=w2, out2=out2, write_h=False)
    assert torch.equal(plain, h + d1)
    v = (h + d1).double()
    want = v / (v.pow(2).mean(1, keepdim=True) + 1e-5).sqrt() * w2.double()
    assert ((out2.double() - want).abs() <= 2e-6 * want.abs().max()).all()      # fp32 sums of d terms in a tree
