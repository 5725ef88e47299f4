"""Products, residuals and filter steps of packed systems that stream their matrix past the caches (values above
650k rows, run words too above 2.7M) against the cached loads of the slot form and of smaller systems."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _system(cuda, n):
    """Level system of n voxels in full x-planes of a cube, and random points in their cells."""
    import ngspsr
    from ngspsr.reconstructor import PointBinning
    side = 1
    while side ** 3 < n:
        side += 1
    lin = torch.arange(n)
    c = torch.stack([lin // side ** 2, lin // side % side, lin % side], 1).to(torch.int32)
    g = torch.Generator().manual_seed(n)
    at = c[torch.randint(n, (n // 4,), generator=g)].float()
    xyz = ((at + torch.rand(at.shape, generator=g)) / 256).to(cuda)
    tree = ngspsr.HashTree(xyz, voxel_size=1 / 256, depth=1)
    tree.update_coords(tree.DECODER, 0, c)
    rec = ngspsr.Reconstructor(tree)
    rhs = torch.randn(n, generator=g, dtype=torch.float64).to(cuda)
    return rec.assemble_level(0, PointBinning(tree, xyz, 0, 4.0), None, 1.0, 0.1, rhs.clone(), form="runs"), rhs


@pytest.mark.parametrize("n", [650000, 650001, 700001, 2700000, 2700001, 2800003])
def test_streamed_products_match_the_slot_form(cuda, n):
    """y = A x bit for bit the slot form's; the FP64 residual against the slot form's kernel (125 terms and b in
    FP64, in any order: 130 x 2^-53 of their magnitudes); one filtered step from the words by plain torch in FP64 (27
    FP32 products: 3e-6 of the vector's norm, as for the smaller systems)."""
    from ngspsr import solver
    print(f"[case] streamed packed system n={n}", flush=True)
    system, rhs = _system(cuda, n)
    assert system.M == n and system.is_packed
    g = torch.Generator(device="cpu").manual_seed(n)
    x = torch.randn(n, generator=g).to(cuda)
    assert torch.equal(system.matvec(x), system.matvec_slots(x))
    slots = solver.RunSystem(system.runs, system.rvals, system.inv_diag, packed=False)
    x64 = x.double() + 1e-9
    r, rr, bb = system.residual_f64(rhs, x64)
    rs, _, _ = slots.residual_f64(rhs, x64)
    size = solver.RunSystem(system.runs, system.rvals.abs(), system.inv_diag, packed=False)
    assert bool(((r - rs).abs() <= 130 * 2.0 ** -53 * size.residual_f64(rhs.abs(), -x64.abs())[0]).all())
    del slots, size
    f = system.filter()
    b = rhs.float()
    got, info = solver.pcg(system, b, tol=0.0, maxiter=1, chunk=2, raise_on_cap=False, filt=f)
    assert info.iters == 1
    c = system.level_grid.coords.long()
    side = int(c.max()) + 3
    lut = torch.full((side, side, side), n, dtype=torch.int64, device=cuda)
    lut[c[:, 0] + 1, c[:, 1] + 1, c[:, 2] + 1] = torch.arange(n, device=cuda)
    w = [1.0] + [float(v) for v in f.struct.weights]
    sd = system.inv_diag.double() ** 0.5
    s = torch.cat([sd * b.double(), torch.zeros(1, dtype=torch.float64, device=cuda)])
    z = torch.zeros(n, dtype=torch.float64, device=cuda)
    for o in np.ndindex(3, 3, 3):
        k = sum(int(v != 1) for v in o)
        z += w[k] * s[lut[c[:, 0] + o[0], c[:, 1] + o[1], c[:, 2] + o[2]]]
    rz = float(s[:n] @ z)
    z *= sd
    az = rhs - system.residual_f64(rhs, z)[0]
    want = rz / float(z @ az) * z
    assert float((got.double() - want).norm()) <= 3e-6 * float(want.norm())
