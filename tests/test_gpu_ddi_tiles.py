"""DDI pair integrals at the edges of their 64-pair tiles, for every path of the coefficient rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,L,n,offset", [(1, 5, 1, 0), (1, 5, 64, 1), (7, 5, 63, 0), (7, 5, 65, 0), (7, 50, 4097, 2),
                                           (8, 5, 128, 0), (16, 8, 200, 3), (16, 26, 65, 0), (3, 5, 700000, 0)])
def test_ddi_tiles(cuda, nc, L, n, offset):
    """Against float64: every sum has nc^2 terms of three roundings each, so the error is below
    (nc^2 + 3) 2^-24 times the sum of the terms' magnitudes; the last shape takes several tiles a block,
    offset: floats by which the arrays miss 16-byte alignment."""
    from ngspsr import additive
    print(f"[case] ddi tiles nc={nc} L={L} n={n} offset={offset}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(n + nc)

    def rows():
        flat = torch.empty(n * 3 * nc + offset, device=cuda)
        v = flat[offset:].view(n, 3 * nc)
        v.copy_(torch.randn(n, 3 * nc, generator=g))
        return v

    s, t = rows().requires_grad_(), rows().requires_grad_()
    rel = torch.randint(L, (n, 3), generator=g).to(cuda)
    ff, dd = (torch.randn(nc, nc, L, generator=g).to(cuda) for _ in range(2))
    gp, gq = (torch.randn(n, 3, generator=g).to(cuda) for _ in range(2))
    p, q = additive.ddi_forward(s, t, rel, ff, dd)
    gs, gt = torch.autograd.grad((p, q), (s, t), (gp, gq))
    s3, t3 = (v.detach().double().view(n, nc, 3) for v in (s, t))
    eps = (nc * nc + 3) * 2.0 ** -24
    for a in range(3):
        fa, da = (m.double()[:, :, rel[:, a]].permute(2, 0, 1) for m in (ff, dd))
        st = s3[:, :, None, a] * t3[:, None, :, a]
        for got, m in ((p, fa), (q, da)):
            err = (got[:, a].double() - (st * m).sum((1, 2))).abs()
            assert bool((err <= eps * (st * m).abs().sum((1, 2))).all())
        c = gp[:, a, None, None].double() * fa + gq[:, a, None, None].double() * da
        ca = gp[:, a, None, None].double().abs() * fa.abs() + gq[:, a, None, None].double().abs() * da.abs()
        for got, u, dim in ((gs, t3[:, None, :, a], 2), (gt, s3[:, :, None, a], 1)):
            err = (got.view(n, nc, 3)[:, :, a].double() - (c * u).sum(dim)).abs()
            assert bool((err <= eps * (ca * u.abs()).sum(dim)).all())
