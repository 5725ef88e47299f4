"""Packed-form products of small systems (a slice over five waves) at the edges of their slices, blocks and
of the size rule, against the slot form and the pool's products."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _system(cuda, n):
    """Level system of n voxels filling about half of a box, with points in their cells."""
    import ngspsr
    from ngspsr.reconstructor import PointBinning
    rng = np.random.default_rng(n)
    side = max(2, int(np.ceil((2.0 * n) ** (1 / 3))))
    lin = np.sort(rng.choice(side ** 3, size=n, replace=False))
    c = np.stack([lin // side ** 2, lin // side % side, lin % side], 1).astype(np.int32)
    xyz = torch.from_numpy(((c + rng.random((n, 3))) / 64).astype(np.float32)).to(cuda)
    tree = ngspsr.HashTree(xyz, voxel_size=1 / 64, depth=1)
    tree.update_coords(tree.DECODER, 0, torch.from_numpy(c))
    rec = ngspsr.Reconstructor(tree)
    rhs = torch.from_numpy(rng.standard_normal(n)).to(cuda)
    return rec.assemble_level(0, PointBinning(tree, xyz, 0, 4.0), None, 1.0, 0.1, rhs.clone()), rhs


@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 129, 2049, 9429, 65536, 65537])
def test_products_and_solves_match(cuda, n):
    """y = A x equals the slot form's bit for bit, and a solve equals the pool's (which runs the other
    product kernel, and sums the FP64 partials in another order) with the same number of iterations."""
    from ngspsr import serving, solver
    print(f"[case] wide packed product n={n}", flush=True)
    system, rhs = _system(cuda, n)
    assert system.M == n and system.is_packed
    g = torch.Generator(device="cpu").manual_seed(n)
    for _ in range(2):
        x = torch.randn(n, generator=g).to(cuda)
        assert torch.equal(system.matvec(x), system.matvec_slots(x))
    pool = serving.BatchedPCG(cuda, chunk=4)
    try:
        for filt in (None, system.filter()):
            x, info = solver.pcg(system, rhs.float(), tol=1e-6, chunk=6, filt=filt)
            torch.cuda.synchronize()
            xp, ip = pool.solve(system, rhs.float(), tol=1e-6, filt=filt)
            assert info.iters == ip.iters
            assert torch.equal(x, xp)
            _, rr, bb = system.residual_f64(rhs.float().double(), x.double())
            assert (rr / bb) ** 0.5 <= 1.5e-6
    finally:
        pool.close()
