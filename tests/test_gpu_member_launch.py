"""Launch shapes of the additions into a grid's members: a thread per bitmap column or per point (or voxel), sums in
LDS or directly, at the sizes where they change. The whole against its parts: the same FP32 terms added in
another order in FP64, so 1e-12 of the added magnitudes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

WIDE = 24576


def _grid(cuda, n, stride, seed):
    from ngspsr._lib import Level
    from ngspsr.grid import SparseGrid
    rng = np.random.default_rng(seed)
    side = max(2, int(np.ceil((1.5 * n) ** (1 / 3))))
    lin = rng.choice(side ** 3, size=n, replace=False)
    c = (np.stack([lin // side ** 2, lin // side % side, lin % side], 1) * stride).astype(np.int32)
    g = SparseGrid([0, 0, 0], (c.max(0) // stride).tolist(), stride, cuda)
    g.mark_coords(torch.from_numpy(c).to(cuda))
    g.finalize()
    lv = Level()
    lv.grid, lv.coords, lv.M, lv.stride = g.struct(), g.coords.data_ptr(), g.count, stride
    return g, lv, side * stride


@pytest.mark.parametrize("members", [1, 300, 6144, 6145])
@pytest.mark.parametrize("n", [255, WIDE, WIDE + 1, 70001])
def test_splat_equals_the_sum_of_its_parts(cuda, members, n):
    from ngspsr._lib import call, ptr, stream
    print(f"[case] member launch members={members} n={n}", flush=True)
    g, lv, box = _grid(cuda, members, 2, members)
    gen = torch.Generator(device="cpu").manual_seed(n)
    q = ((torch.rand(n, 3, generator=gen) * 1.2 - 0.1) * box).to(cuda)
    w = torch.randn(n, generator=gen).to(cuda)
    w[::9] = 0.0
    outs = [torch.full((members,), 0.25, dtype=torch.float64, device=cuda) for _ in range(3)]
    mag = torch.zeros(members, dtype=torch.float64, device=cuda)
    call("ngs_basis_splat", g.struct(), ptr(w), ptr(q), n, 1.0, -0.5, ptr(outs[0]), stream())
    call("ngs_basis_splat_level", lv, ptr(w), ptr(q), n, 1.0, -0.5, ptr(outs[1]), stream())
    for a in range(0, n, 1000):
        m = min(1000, n - a)
        call("ngs_basis_splat_level", lv, ptr(w[a:]), ptr(q[a:]), m, 1.0, -0.5, ptr(outs[2]), stream())
        call("ngs_basis_splat_level", lv, ptr(w[a:a + m].abs()), ptr(q[a:]), m, 1.0, 0.5, ptr(mag), stream())
    assert float(mag.max()) > 0
    for o in outs[:2]:
        assert bool(((o - outs[2]).abs() <= 1e-12 * (mag + 1.0)).all())


@pytest.mark.parametrize("members", [300, 6145])
@pytest.mark.parametrize("n", [WIDE, WIDE + 1, 60000])
def test_transposed_stiffness_equals_the_sum_of_its_parts(cuda, members, n):
    from ngspsr._lib import Level, call, ptr, stream
    from ngspsr.bases import ensure_device_tables
    ensure_device_tables(cuda)
    print(f"[case] transposed stiffness members={members} n={n}", flush=True)
    g, coarse, box = _grid(cuda, members, 4, members)
    gen = torch.Generator(device="cpu").manual_seed(n)
    c = torch.randint(0, box, (n, 3), generator=gen, dtype=torch.int32).to(cuda)
    gv = torch.randn(n, generator=gen).to(cuda)
    gv[::9] = 0.0

    def rows(a, m):
        lv = Level()
        lv.coords, lv.M, lv.stride = c[a:].data_ptr(), m, 1
        return lv

    whole = torch.zeros(members, dtype=torch.float64, device=cuda)
    parts, mag = torch.zeros_like(whole), torch.zeros_like(whole)
    call("ngs_cross_stiffness_transpose", rows(0, n), coarse, ptr(gv), -1.0, ptr(whole), stream())
    for a in range(0, n, 1000):
        m = min(1000, n - a)
        part = torch.zeros_like(whole)
        call("ngs_cross_stiffness_transpose", rows(a, m), coarse, ptr(gv[a:]), -1.0, ptr(part), stream())
        parts += part
        mag += part.abs()
    # terms of both signs: a part of 1000 rows holds up to 100 times its own sum
    assert float(mag.max()) > 0
    assert bool(((whole - parts).abs() <= 1e-10 * mag.max()).all())
