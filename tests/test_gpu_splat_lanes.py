"""The gather splat with 1, 4, 16 and 64 lanes per node, at the node and point counts where the number changes,
against the atomic scatter: the same FP32 terms added in FP64 in another order, at most a few thousand per
node, so 1e-12 of the sums of their magnitudes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _box(nodes, dev):
    """A grid of exactly `nodes` nodes: full x-planes of a cube, the last one in part."""
    from ngspsr.grid import SparseGrid
    side = 1
    while side ** 3 < nodes:
        side += 1
    lin = torch.arange(nodes, device=dev)
    c = torch.stack([lin // (side * side), lin // side % side, lin % side], 1).to(torch.int32)
    g = SparseGrid([0, 0, 0], [side - 1] * 3, 1, dev)
    g.mark_coords(c)
    g.finalize()
    assert g.count == nodes
    return g, side


@pytest.mark.parametrize("nodes,points", [
    (12000, 30000), (12001, 30000),  # 64, 16
    (100000, 50000), (100001, 50000), (100001, 400003), (100001, 400004),  # 16, 4, 4, 16
    (400000, 200000), (400001, 300000), (400001, 300001),  # 4, 1, 4
    (1500000, 1125000), (1500001, 1500001), (700000, 20000)])  # 4, 1, 1
@pytest.mark.parametrize("ncomp", [0, 3])
def test_lanes_equal_the_scatter(cuda, nodes, points, ncomp):
    from ngspsr._lib import call, lib, ptr, stream
    print(f"[case] splat lanes nodes={nodes} points={points} ncomp={ncomp}", flush=True)
    g, side = _box(nodes, cuda)
    gen = torch.Generator().manual_seed(nodes + points)
    xyz = (torch.rand((points, 3), generator=gen) * (side + 2) - 1).to(cuda)  # some outside the box
    xyz[: points // 50] = xyz[0]  # one long bin
    data = torch.randn((points, max(ncomp, 1)), generator=gen).to(cuda)
    scale = (torch.rand(points, generator=gen) + 0.5).to(cuda)
    levels = torch.randint(0, 3, (points,), generator=gen, dtype=torch.int32).to(cuda)
    shape = (nodes, ncomp) if ncomp else (nodes,)

    def splat(name, d, *ws):
        out = torch.zeros(shape, dtype=torch.float64, device=cuda)
        head = (g.struct(),) if name == "ngs_splat" else (g.struct(), ptr(g.coords), nodes)
        call(name, *head, ptr(xyz), points, 1.0, ptr(d) if ncomp else None, ncomp, ptr(scale), ptr(levels), 1, 1.0,
             ptr(out), *ws, stream())
        return out

    want, mag = splat("ngs_splat", data), splat("ngs_splat", data.abs())
    wsb = lib().ngs_splat_gather_workspace_bytes(points, nodes)
    ws = torch.empty(wsb, dtype=torch.uint8, device=cuda)
    got = splat("ngs_splat_gather", data, ptr(ws), wsb)
    assert float(mag.max()) > 0
    assert bool(((got - want).abs() <= 1e-12 * mag).all())
