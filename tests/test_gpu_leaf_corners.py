"""Field values at leaf corners (MI355X): the window read per leaf equals evaluating the written corner
positions bit for bit, with leaves at and past the border of the field's box, levels with one member and
with none, and level strides below, at and above the leaf's."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("members", [0, 1, 2, 3, 400])
@pytest.mark.parametrize("s_leaf", [1, 2])
def test_leaf_corners_at_borders(cuda, members, s_leaf):
    from ngspsr._lib import Grid, call, lib, ptr, stream
    from ngspsr.hashtree import SparseGrid
    print(f"[case] leaf corners members={members} s_leaf={s_leaf}", flush=True)
    rng = np.random.default_rng(members + s_leaf)
    vs = np.float32(1 / 16)
    scale = float(np.float32(vs / np.float32(2)))
    inv_vs = float(np.float32(1) / vs)
    leaves = torch.from_numpy((rng.integers(-9, 14, (700, 3)) * s_leaf).astype(np.int32)).to(cuda)
    n = leaves.shape[0]
    pos = torch.empty((8 * n, 3), dtype=torch.float32, device=cuda)
    call("ngs_leaf_corner_positions", ptr(leaves), n, s_leaf, 2, scale, ptr(pos), stream())
    grids, fields = [], []
    want = torch.zeros(8 * n, dtype=torch.float32, device=cuda)
    for s in (1, 2, 4):
        g = SparseGrid([-5] * 3, [6, 7, 40], s, cuda)
        if members:
            g.mark_coords(torch.from_numpy((rng.integers(-5, 7, (members, 3)) * s).astype(np.int32)).to(cuda))
        count = g.finalize()
        assert (count > 0) == (members > 0)
        f = torch.from_numpy(rng.standard_normal(max(count, 1)).astype(np.float32)).to(cuda)
        one = torch.empty(8 * n, dtype=torch.float32, device=cuda)
        got = torch.empty_like(one)
        if count:
            call("ngs_eval_field", g.struct(), ptr(f), ptr(pos), n * 8, inv_vs, 1.0, 0, ptr(one), None, stream())
        else:
            one.zero_()
        call("ngs_eval_leaf_corners", g.struct(), ptr(f), ptr(leaves), n, s_leaf, 2, scale, inv_vs, 0, ptr(got), stream())
        np.testing.assert_array_equal(got.cpu().numpy(), one.cpu().numpy())
        want += one
        grids.append(g)
        fields.append(f)
    got = torch.empty_like(want)
    garr = (Grid * 3)(*[g.struct() for g in grids])
    farr = (ctypes.c_void_p * 3)(*[f.data_ptr() for f in fields])
    call("ngs_eval_leaf_corners_levels", 3, garr, farr, ptr(leaves), n, s_leaf, 2, scale, inv_vs, 0, ptr(got), stream())
    np.testing.assert_array_equal(got.cpu().numpy(), want.cpu().numpy())
