"""Field evaluation at the edges of its 12-byte coefficient loads, and in a permuted order, against float64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,stride", [(1, 1), (2, 1), (3, 2), (4, 1), (31, 4), (2000, 1)])
def test_field_on_few_voxels(cuda, n, stride):
    """n random voxels of a small box (single voxels, columns that end the coefficient array): values and
    gradients against the sum over all voxels in float64. 27 terms of five roundings each: 32 x 2^-23 of
    the terms' magnitudes. The permuted evaluation gives the same bits."""
    from ngspsr._lib import call, ptr, stream
    from ngspsr.grid import SparseGrid
    print(f"[case] field on {n} voxels, stride {stride}", flush=True)
    rng = np.random.default_rng(n + stride)
    side = max(2, int(np.ceil((1.7 * n) ** (1 / 3))))
    lin = rng.choice(side ** 3, size=n, replace=False)
    c = (np.stack([lin // side ** 2, lin // side % side, lin % side], 1) * stride).astype(np.int32)
    g = SparseGrid([0, 0, 0], (c.max(0) // stride).tolist(), stride, cuda)
    g.mark_coords(torch.from_numpy(c).to(cuda))
    g.finalize()
    f = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(cuda)
    m = 3001
    q = torch.from_numpy((rng.random((m, 3)) * (side + 4) * stride - 2 * stride).astype(np.float32)).to(cuda)
    v, g3 = torch.zeros(m, device=cuda), torch.zeros((m, 3), device=cuda)
    call("ngs_eval_field", g.struct(), ptr(f), ptr(q), m, 1.0, 1.0, 0, ptr(v), ptr(g3), stream())
    v1, v2 = torch.full_like(v, 7.0), torch.full_like(v, 7.0)
    call("ngs_eval_field", g.struct(), ptr(f), ptr(q), m, 1.0, 1.0, 1, ptr(v1), None, stream())
    order = torch.randperm(m, device=cuda).int()
    call("ngs_eval_field_ordered", g.struct(), ptr(f), ptr(q), ptr(order), m, 1.0, 1.0, 1, ptr(v2), stream())
    assert torch.equal(v1, v2) and torch.equal(v1, v + 7.0)
    u = (q.double()[:, None, :] - g.coords.double()[None] - stride / 2) / stride
    a = u.abs()
    b = torch.where(a < 0.5, 1.5 - 2 * a * a, torch.where(a < 1.5, (a - 1.5) ** 2, torch.zeros_like(a)))
    db = torch.where(a < 0.5, -4 * u, torch.where(a < 1.5, 2 * (a - 1.5) * torch.sign(u), torch.zeros_like(a))) / stride
    for got, t in ((v, b.prod(2)), (g3[:, 0], db[..., 0] * b[..., 1] * b[..., 2]),
                   (g3[:, 1], b[..., 0] * db[..., 1] * b[..., 2]), (g3[:, 2], b[..., 0] * b[..., 1] * db[..., 2])):
        # the positions' own rounding moves u by 2^-23 of the box per axis: the field's slope is at most 9
        tol = 32 * 2.0 ** -23 * (t * f.double()).abs().sum(1) + 40 * 2.0 ** -23 * (side + 4) * float(f.abs().sum())
        assert bool(((got.double() - (t * f.double()).sum(1)).abs() <= tol).all())
