"""DDI pair integrals where a block takes several tiles (more tiles than one or four rounds of resident blocks)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,L,n", [(10, 50, 512 * 64), (10, 50, 512 * 64 + 1), (7, 50, 1280 * 64 + 65), (16, 14, 70001),
                                    (1, 5, 10240 * 64 + 1)])
def test_pairs_are_independent(cuda, nc, L, n):
    """Every pair gets the bits that it gets in a call of its own chunk of 64 blocks of tiles."""
    from ngspsr import additive
    print(f"[case] ddi rounds nc={nc} L={L} n={n}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(n + nc)
    s, t = (torch.randn(n, 3 * nc, generator=g).to(cuda).requires_grad_() for _ in range(2))
    rel = torch.randint(L, (n, 3), generator=g).to(cuda)
    ff, dd = (torch.randn(nc, nc, L, generator=g).to(cuda) for _ in range(2))
    gp, gq = (torch.randn(n, 3, generator=g).to(cuda) for _ in range(2))

    def both(a, b):
        sa, ta = s[a:b].detach().requires_grad_(), t[a:b].detach().requires_grad_()
        p, q = additive.ddi_forward(sa, ta, rel[a:b], ff, dd)
        return (p, q) + torch.autograd.grad((p, q), (sa, ta), (gp[a:b], gq[a:b]))

    whole = both(0, n)
    for a in range(0, n, 4096):
        for w, c in zip(whole, both(a, min(a + 4096, n))):
            assert torch.equal(w[a:a + 4096], c)
