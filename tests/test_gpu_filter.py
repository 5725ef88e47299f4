"""Filtered preconditioner of the refined solves: its words against a brute-force neighbour search, its
application through one PCG step, and filtered solves alone and in the pool."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _grid(coords, stride, dev):
    from ngspsr.grid import SparseGrid
    c = np.asarray(coords, np.int32)
    g = SparseGrid((c.min(0) // stride).tolist(), (c.max(0) // stride).tolist(), stride, dev)
    g.mark_coords(torch.from_numpy(c).to(dev))
    g.finalize()
    return g


def _voxels(n, stride, seed):
    """n distinct voxels in a box tight around them (so neighbours also fall outside the box)."""
    rng = np.random.default_rng(seed)
    side = max(1, int(np.ceil((2.2 * n) ** (1 / 3))))
    lin = rng.choice(side ** 3, size=n, replace=False)
    return np.stack([lin // side ** 2, lin // side % side, lin % side], 1) * stride - 3 * stride


@pytest.mark.parametrize("n,stride", [(1, 1), (2, 4), (63, 1), (64, 2), (65, 1), (257, 8), (4097, 1)])
def test_filter_words_match_brute_force(cuda, n, stride):
    from ngspsr._lib import Level, call, ptr, stream
    print(f"[case] filter words n={n} stride={stride}", flush=True)
    g = _grid(_voxels(n, stride, n), stride, cuda)
    assert g.count == n
    P = (n + 63) // 64 * 64
    words = torch.full((9, P), -1, dtype=torch.int32, device=cuda)
    lv = Level()
    lv.grid, lv.coords, lv.M, lv.stride = g.struct(), g.coords.data_ptr(), n, stride
    call("ngs_level_filter_words", lv, ptr(words), stream())
    w = words.cpu().numpy().view(np.uint32)[:, :n]
    c = g.coords.cpu().numpy()
    row = {tuple(v): i for i, v in enumerate(c)}
    for k in range(9):
        for i in range(n):
            nb = [row.get((c[i, 0] + (k // 3 - 1) * stride, c[i, 1] + (k % 3 - 1) * stride, c[i, 2] + dz * stride))
                  for dz in (-1, 0, 1)]
            mask = sum(1 << j for j, v in enumerate(nb) if v is not None)
            first = next((v for v in nb if v is not None), 0)
            assert (int(w[k, i]) >> 29, int(w[k, i]) & ((1 << 29) - 1)) == (mask, first), (k, i)


def _systems(cuda, alpha=4.0, per_point=False):
    import ngspsr
    from ngspsr import synthetic
    from ngspsr.reconstructor import PointBinning
    xyz, nrm = synthetic.ellipsoids(12000, k=5, sigma=0.003, seed=23)
    x = torch.from_numpy(xyz).to(cuda)
    tree = ngspsr.HashTree(x, voxel_size=1 / 64, depth=3)
    tree.build_encoder_hierarchy_adaptive(min_density=1.0)
    tree.reflect_decoder_coords()
    rec = ngspsr.Reconstructor(tree)
    a = alpha * (0.5 + torch.rand(x.shape[0], device=cuda)) if per_point else alpha
    g = torch.Generator(device="cpu").manual_seed(5)
    out = []
    for d in range(3):
        M = tree.get_coords_size(None, d)
        rhs = torch.randn(M, generator=g, dtype=torch.float64).to(cuda)
        out.append((rec.assemble_level(d, PointBinning(tree, x, d, a), None, 0.25 ** d, 0.1, rhs), rhs))
    return out


def test_one_step_applies_the_filter(cuda):
    """After one iteration x = (r.z / z.Az) z with z = D^-1/2 P D^-1/2 b: checked in float64 against P built
    from the voxel coordinates. Each z sums 27 FP32 products, so a relative error of 2^-24 times a small
    multiple of 27 (3e-6 against the vector's norm)."""
    print("[case] one filtered step", flush=True)
    from ngspsr import solver
    for system, rhs in _systems(cuda):
        f = system.filter()
        b = rhs.float()
        x, info = solver.pcg(system, b, tol=0.0, maxiter=1, chunk=2, raise_on_cap=False, filt=f)
        assert info.iters == 1
        c = system.level_grid.coords.cpu().numpy().astype(np.int64) // system.level_stride
        row = {tuple(v): i for i, v in enumerate(c)}
        w = [1.0] + [float(v) for v in f.struct.weights]
        sd = system.inv_diag.double().cpu().numpy() ** 0.5
        s = sd * b.double().cpu().numpy()
        z = np.zeros_like(s)
        for dx in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dz in (-1, 0, 1):
                    j = np.array([row.get((v[0] + dx, v[1] + dy, v[2] + dz), -1) for v in c])
                    z += w[abs(dx) + abs(dy) + abs(dz)] * np.where(j >= 0, s[j], 0.0)
        rz = float(s @ z)
        z *= sd
        az = system.to_scipy() @ z
        want = rz / float(z @ az) * z
        got = x.double().cpu().numpy()
        assert np.linalg.norm(got - want) <= 3e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("alpha,per_point", [(0.05, False), (1.0, False), (4.0, False), (200.0, False), (4.0, True)])
def test_filtered_solves_alone_and_in_the_pool(cuda, alpha, per_point):
    """A filtered solve reaches the tolerance it is asked for (FP64 residual, 1.5 times for the FP32
    recurrence's drift), in fewer iterations than Jacobi where screening dominates, and the pool, mixing
    filtered and Jacobi systems, gives each its single solve bit for bit."""
    import threading
    from ngspsr import serving, solver
    print(f"[case] filtered solves alpha={alpha} per_point={per_point}", flush=True)
    jobs = []
    for system, rhs in _systems(cuda, alpha, per_point):
        f = system.filter()
        assert f is not None
        b = rhs.float()
        x, info = solver.pcg(system, b, tol=1e-6, chunk=solver.FILTER_CHUNK, filt=f)
        r, rr, bb = system.residual_f64(b.double(), x.double())
        assert (rr / bb) ** 0.5 <= 1.5e-6, (alpha, (rr / bb) ** 0.5)
        _, jac = solver.pcg(system, b, tol=1e-6)
        if alpha >= 4.0:
            assert info.iters < jac.iters, (info.iters, jac.iters)
        x64, ri = solver.refine(system, rhs, tol=1e-9)
        assert ri.true_rel_resid <= 1e-9
        jobs += [(system, b, f), (system, b, None)]
    pool = serving.BatchedPCG(cuda, chunk=4)
    outs = [None] * len(jobs)
    torch.cuda.synchronize()
    try:
        def work(i):
            outs[i] = pool.solve(jobs[i][0], jobs[i][1], tol=1e-6, filt=jobs[i][2])
        th = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
        [t.start() for t in th]
        [t.join() for t in th]
    finally:
        pool.close()
    for (system, b, f), (xp, ip) in zip(jobs, outs):
        x, info = solver.pcg(system, b, tol=1e-6, filt=f)
        torch.cuda.synchronize()
        assert info.iters == ip.iters and torch.equal(x, xp)


def test_filter_needs_screening_and_positive_weights(cuda):
    """No filter without screening points or for a system of unknown level; weights whose symbol is not
    positive are refused on the host."""
    from ngspsr import solver
    from ngspsr._lib import NgsError
    print("[case] filter refusals", flush=True)
    system, rhs = _systems(cuda)[0]
    bare = solver.RunSystem(system.runs, system.rvals.clone(), system.inv_diag)
    assert bare.filter() is None
    system.screening = 0.0
    assert system.filter() is None
    system.screening = 1.0
    f = system.filter()
    f.struct.weights[0] = -0.5
    with pytest.raises(NgsError, match="positive definite"):
        solver.pcg(system, rhs.float(), filt=f)
