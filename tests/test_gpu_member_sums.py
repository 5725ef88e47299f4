"""Additions into a grid's members (LDS sums per block or direct atomics), at the sizes where the path changes,
and the per-level point counts."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _grid(cuda, n, stride, seed):
    from ngspsr.grid import SparseGrid
    rng = np.random.default_rng(seed)
    side = max(2, int(np.ceil((1.5 * n) ** (1 / 3))))
    lin = rng.choice(side ** 3, size=n, replace=False)
    c = (np.stack([lin // side ** 2, lin // side % side, lin % side], 1) * stride).astype(np.int32)
    g = SparseGrid([0, 0, 0], (c.max(0) // stride).tolist(), stride, cuda)
    g.mark_coords(torch.from_numpy(c).to(cuda))
    g.finalize()
    return g, side * stride


@pytest.mark.parametrize("members,points", [(1, 1), (3, 700), (110, 10000), (6144, 400000), (6145, 400000), (2033, 3000)])
def test_basis_splat_is_the_transposed_field(cuda, members, points):
    """<w, field(f)> = <f, splat(w)>: the field in float64 from the same basis formula; 27 products of
    five float32 roundings per point, so 32 x 2^-23 of the terms' magnitudes on either side, and the
    positions' rounding as in the field's own test."""
    from ngspsr._lib import call, ptr, stream
    print(f"[case] basis splat members={members} points={points}", flush=True)
    g, box = _grid(cuda, members, 2, members)
    gen = torch.Generator(device="cpu").manual_seed(points)
    q = ((torch.rand(points, 3, generator=gen) * 1.2 - 0.1) * box).to(cuda)
    w = torch.randn(points, generator=gen).to(cuda)
    w[::7] = 0.0
    out = torch.full((members,), 0.25, dtype=torch.float64, device=cuda)
    call("ngs_basis_splat", g.struct(), ptr(w), ptr(q), points, 1.0, -0.5, ptr(out), stream())
    want = torch.full_like(out, 0.25)
    mag = torch.zeros_like(out)
    lut = torch.full((box // 2 + 6,) * 3, members, dtype=torch.int64, device=cuda)
    c = g.coords.long() // 2 + 2
    lut[c[:, 0], c[:, 1], c[:, 2]] = torch.arange(members, device=cuda)
    cell = torch.floor(q.double() / 2).long()
    for o in [(x, y, z) for x in (-1, 0, 1) for y in (-1, 0, 1) for z in (-1, 0, 1)]:
        v = cell + torch.tensor(o, device=cuda)
        a = ((q.double() - v * 2 - 1) / 2).abs()
        b = torch.where(a < 0.5, 1.5 - 2 * a * a, torch.where(a < 1.5, (a - 1.5) ** 2, torch.zeros_like(a))).prod(1)
        vi = (v + 2).clamp(0, lut.shape[0] - 1)
        j = torch.where(((v + 2) == vi).all(1), lut[vi[:, 0], vi[:, 1], vi[:, 2]], members)
        on = j < members
        want.index_add_(0, j[on], (-0.5 * w.double() * b)[on])
        mag.index_add_(0, j[on], (w.double().abs() * (b + 1e-3))[on])
    assert bool(((out - want).abs() <= 64 * 2.0 ** -23 * box * mag + 1e-12).all())


@pytest.mark.parametrize("n", [40, 400, 3000])
def test_cross_stiffness_transpose_is_the_adjoint(cuda, n):
    """K^T g over three pairs of levels (strides 1-2, 1-4, 2-4) against the matrix whose columns the forward
    kernel gives for unit vectors (its float32 entries themselves): a product with g and a sum in FP64 per
    entry, 4 x 2^-23 of the magnitudes for the entry's own roundings in another order."""
    import ngspsr
    from ngspsr._lib import call, ptr, stream
    from ngspsr.bases import ensure_device_tables
    print(f"[case] cross stiffness transpose n={n}", flush=True)
    ensure_device_tables(cuda)
    gen = torch.Generator(device="cpu").manual_seed(n)
    xyz = torch.rand(n, 3, generator=gen)
    xyz[:, 2] *= 0.1
    tree = ngspsr.HashTree(xyz.to(cuda), voxel_size=1 / 32, depth=3)
    tree.build_encoder_hierarchy_adaptive(uniform_density=True, min_density=1.0)
    tree.reflect_decoder_coords()
    for d, dd in ((0, 1), (0, 2), (1, 2)):
        M, Mc = tree.get_coords_size(None, d), tree.get_coords_size(None, dd)
        gv = torch.randn(M, generator=gen).to(cuda)
        gv[::5] = 0.0
        o = torch.full((Mc,), 2.0, dtype=torch.float64, device=cuda)
        call("ngs_cross_stiffness_transpose", tree.level(d), tree.level(dd), ptr(gv), -1.0, ptr(o), stream())
        x = torch.zeros(Mc, device=cuda)
        for j in range(Mc):
            x[j] = 1.0
            r = torch.zeros(M, dtype=torch.float64, device=cuda)  # minus column j
            call("ngs_rhs_cross_stiffness", tree.level(d), tree.level(dd), ptr(x), ptr(r), stream())
            x[j] = 0.0
            t = r * gv.double()
            assert abs(float(t.sum()) - float(o[j] - 2.0)) <= 4 * 2.0 ** -23 * float(t.abs().sum()) + 1e-12, (d, dd, j)


@pytest.mark.parametrize("n,depth", [(1, 1), (255, 4), (257, 5), (300001, 4)])
def test_level_counts(cuda, n, depth):
    """Counts equal torch.bincount's, imposed levels past the depth lengthen them, negative ones are
    refused."""
    import ngspsr
    print(f"[case] level counts n={n} depth={depth}", flush=True)
    gen = torch.Generator(device="cpu").manual_seed(n)
    tree = ngspsr.HashTree(torch.rand(max(n, 1), 3, generator=gen).to(cuda), voxel_size=1 / 32, depth=depth)
    lv = torch.randint(depth, (n,), generator=gen, dtype=torch.int32).to(cuda)
    assert tree._count_levels(lv).tolist() == torch.bincount(lv.long(), minlength=depth).tolist()
    lv[0] = depth + 2
    assert tree._count_levels(lv).tolist() == torch.bincount(lv.long(), minlength=depth).tolist()
    lv[0] = -1
    with pytest.raises(RuntimeError):
        tree._count_levels(lv)
