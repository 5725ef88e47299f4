"""Cubes with triangles gathered without the other centres' slots (MI355X): equal, row by row, to the
cubes of all centres with complete corners and changing signs, on fewer centres than a block, on
blocks with all and with few of theirs, and cut off at the end; the mesh with and without the report."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# leaves per axis of the filled box, share of them kept
@pytest.mark.parametrize("dims,keep", [((1, 1, 1), 1.0), ((2, 3, 5), 1.0), ((17, 23, 31), 1.0), ((40, 9, 130), 0.5),
                                       ((60, 60, 60), 0.03)])
def test_active_cubes(cuda, dims, keep):
    from ngspsr._lib import Grid, call, lib, ptr, stream
    from ngspsr.hashtree import SparseGrid
    print(f"[case] active cubes dims={dims} keep={keep}", flush=True)
    rng = np.random.default_rng(sum(dims))
    c = np.stack(np.meshgrid(*[np.arange(d) for d in dims], indexing="ij"), -1).reshape(-1, 3) - 3
    c = c[rng.random(c.shape[0]) < keep].astype(np.int32)
    n = c.shape[0]
    leaves = torch.from_numpy(c).to(cuda)
    lg = SparseGrid([-3] * 3, [d - 3 for d in dims], 1, cuda)
    lg.mark_coords(leaves)
    cg = SparseGrid([-8] * 3, [2 * d for d in dims], 1, cuda)
    call("ngs_mark_dual_leaf_words", cg.struct(), lg.struct(), stream())
    DC = cg.finalize()
    lg.finalize(emit=False, count=False)
    ranks = torch.empty(n, dtype=torch.int32, device=cuda)
    call("ngs_grid_rank_rows", lg.struct(), ptr(leaves), n, ptr(ranks), stream())
    li = torch.empty(n, dtype=torch.int32, device=cuda)
    li[ranks.long()] = torch.arange(n, dtype=torch.int32, device=cuda)
    values = torch.from_numpy(rng.standard_normal(8 * n).astype(np.float32)).to(cuda)
    garr, iarr, barr = (Grid * 1)(lg.struct()), (ctypes.c_void_p * 1)(li.data_ptr()), (ctypes.c_int32 * 1)(0)
    i32 = lambda *s: torch.full(s, -7, dtype=torch.int32, device=cuda)  # noqa: E731
    acc, cnt, cubes, flags, offs = i32(DC, 8), i32(DC), i32(DC, 8), i32(DC), i32(DC + 1)
    ws = torch.empty(lib().ngs_scan_workspace_bytes(DC), dtype=torch.uint8, device=cuda)
    call("ngs_dual_gather_cubes", ptr(cg.coords), DC, 1, garr, iarr, barr, ptr(values), ptr(acc), ptr(cnt), stream())
    call("ngs_dual_compact", ptr(acc), ptr(cnt), 1, DC, ptr(cubes), ptr(flags), ptr(offs), ptr(ws), stream())
    nb = lib().ngs_dual_active_blocks(DC)
    rows, bc, boff, got = i32(DC, 8), i32(nb), i32(nb + 1), i32(DC, 8)
    ws = torch.empty(lib().ngs_scan_workspace_bytes(nb), dtype=torch.uint8, device=cuda)
    call("ngs_dual_gather_active", ptr(cg.coords), DC, 1, garr, iarr, barr, ptr(values), ptr(rows), ptr(bc), stream())
    call("ngs_dual_compact_active", ptr(rows), ptr(bc), DC, ptr(boff), ptr(got), ptr(ws), stream())
    K = int(offs[DC].item())
    assert int(boff[nb].item()) == K and K > 0
    np.testing.assert_array_equal(got[:K].cpu().numpy(), cubes[:K].cpu().numpy())
    assert bool((got[K:] == -7).all())


@pytest.mark.parametrize("n,depth,trim", [(300, 2, False), (6000, 3, True), (6000, 4, False)])
def test_mesh_with_and_without_report(cuda, n, depth, trim):
    import ngspsr
    from ngspsr import synthetic
    print(f"[case] mesh report n={n} depth={depth} trim={trim}", flush=True)
    xyz, nrm = synthetic.sphere(n, seed=n + depth)
    lv = torch.from_numpy(np.random.default_rng(n).integers(0, depth, n).astype(np.int32)).to(cuda)
    res = ngspsr.reconstruct(torch.from_numpy(xyz).to(cuda), torch.from_numpy(nrm).to(cuda), 1 / 32, depth=depth,
                             min_density=4.0, xyz_depth=lv, return_result=True)
    v, f, _ = res.reconstructor.extract_multiscale_mesh(n_upsample=2, trim=trim, return_info=True)
    v2, f2 = res.reconstructor.extract_multiscale_mesh(n_upsample=2, trim=trim, build_o3d_mesh=False)
    assert f.shape[0] > 50
    np.testing.assert_array_equal(f2.cpu().numpy(), f.cpu().numpy())
    np.testing.assert_array_equal(v2.cpu().numpy(), v.cpu().numpy())
