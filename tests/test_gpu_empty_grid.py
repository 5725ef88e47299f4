"""Calls on a grid without words (a zero-initialised struct, no buffers): nothing is read from it, the field is 0
everywhere and additions into it have no effect."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 300])
def test_field_and_its_transpose_on_a_grid_without_words(cuda, n):
    from ngspsr._lib import Grid, Level, call, ptr, stream
    from ngspsr.bases import ensure_device_tables
    ensure_device_tables(cuda)
    print(f"[case] empty grid n={n}", flush=True)
    q = torch.rand(n, 3, device=cuda)
    order = torch.randperm(n, dtype=torch.int32, device=cuda)
    for accumulate in (0, 1):
        want = torch.full((n,), 0.75 if accumulate else 0.0, device=cuda)
        out = torch.full((n,), 0.75, device=cuda)
        call("ngs_eval_field", Grid(), None, ptr(q), n, 1.0, 2.0, accumulate, ptr(out), None, stream())
        assert torch.equal(out, want)
        out = torch.full((n,), 0.75, device=cuda)
        grad = torch.full((n, 3), 0.75, device=cuda)
        call("ngs_eval_field", Grid(), None, ptr(q), n, 1.0, 2.0, accumulate, ptr(out), ptr(grad), stream())
        assert torch.equal(out, want) and torch.equal(grad, want[:, None].expand(n, 3))
        out = torch.full((n,), 0.75, device=cuda)
        call("ngs_eval_field_ordered", Grid(), None, ptr(q), ptr(order), n, 1.0, 2.0, accumulate, ptr(out), stream())
        assert torch.equal(out, want)
    cell = torch.zeros((n, 3), dtype=torch.int32, device=cuda)
    basis = torch.rand(n, 9, device=cuda)
    out = torch.full((n,), 0.75, device=cuda)
    call("ngs_eval_field_binned", Grid(), ptr(q), ptr(cell), ptr(basis), ptr(order), n, 1.0, ptr(out), stream())
    assert bool((out == 0.75).all())
    # no member receives anything: a null output is not written
    call("ngs_basis_splat", Grid(), ptr(out), ptr(q), n, 1.0, 1.0, None, stream())
    fine, coarse = Level(), Level()
    coords = torch.zeros((n, 3), dtype=torch.int32, device=cuda)
    fine.coords, fine.M, fine.stride, coarse.stride = coords.data_ptr(), n, 1, 2
    call("ngs_cross_stiffness_transpose", fine, coarse, ptr(out), 1.0, None, stream())
    torch.cuda.synchronize()
