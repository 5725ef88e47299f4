"""Which preconditioner the refined and adjoint solves take: by the screening strength, per-point weights counting
with their mean."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _levels(cuda, alphas):
    import ngspsr
    from ngspsr import synthetic
    from ngspsr.reconstructor import PointBinning
    xyz, _ = synthetic.ellipsoids(12000, k=5, sigma=0.003, seed=23)
    x = torch.from_numpy(xyz).to(cuda)
    tree = ngspsr.HashTree(x, voxel_size=1 / 64, depth=3)
    tree.build_encoder_hierarchy_adaptive(min_density=1.0)
    tree.reflect_decoder_coords()
    rec = ngspsr.Reconstructor(tree)
    for d in range(3):
        rhs = torch.randn(tree.get_coords_size(None, d), generator=torch.Generator().manual_seed(d),
                          dtype=torch.float64).to(cuda)
        bins = PointBinning.levels(tree, x, [d], alphas[0])[d], PointBinning(tree, x, d, alphas[1])
        yield [rec.assemble_level(d, b, None, 0.25 ** d, 0.1, rhs.clone()) for b in bins], rhs


@pytest.mark.parametrize("mean", [0.0, 1e-4, 0.02, 1.0, 4.0, 30.0, 400.0])
def test_weights_choose_as_their_mean(cuda, mean):
    """Weights spread evenly around a mean take the filter that this mean takes as a scalar, or none."""
    from ngspsr import solver
    print(f"[case] filter choice mean={mean}", flush=True)
    ramp = torch.linspace(0.5, 1.5, 12000, device=cuda)
    chosen = []
    for (a, b), _ in _levels(cuda, (mean * ramp, mean)):
        assert abs(a.screening_strength() - b.screening_strength()) <= 1e-6 * b.screening_strength()
        fa, fb = solver.system_filter(a), solver.system_filter(b)
        assert (fa is None) == (fb is None) == (b.screening_strength() < solver.FILTER_STRENGTH)
        assert fa is None or list(fa.struct.weights) == list(fb.struct.weights)
        chosen.append(fa)
    if mean <= 1e-4:
        assert all(f is None for f in chosen)
    if mean >= 4.0:
        assert all(f is not None for f in chosen)


@pytest.mark.parametrize("value", [0.0, 1e-5, -1e-5, float("nan")])
def test_weak_weights_are_solved_with_jacobi(cuda, value):
    """Weights near zero, negative or NaN on the mean: no filter, and a refined solve takes Jacobi's iterations."""
    from ngspsr import solver
    print(f"[case] weak weights {value}", flush=True)
    for (a, b), rhs in _levels(cuda, (torch.full((12000,), value, device=cuda), 0.0)):
        assert solver.system_filter(a) is None and solver.system_filter(b) is None
        if value == value:
            _, info = solver.refine(a, rhs, tol=1e-6)
            _, jac = solver.pcg(a, rhs.float(), tol=(0.3 if value > 0 else 0.5) * 1e-6, chunk=16)
            assert info.outer == 1 and info.iters == jac.iters and info.true_rel_resid <= 1e-6
