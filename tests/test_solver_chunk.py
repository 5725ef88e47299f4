"""Iterations per launch sequence that a solver string asks for (host logic, no GPU): a named chunk reaches the
PCG as given, a string without one takes the method's own."""
import pytest
import torch


class _System:
    M, device = 3, "cpu"

    def residual_f64(self, b64, x64):
        r = b64 if x64 is None else b64 - x64  # the unit matrix
        return r, float(r @ r), float(b64 @ b64)


@pytest.mark.parametrize("filtered", [False, True])
@pytest.mark.parametrize("spec,chunk", [("pcg", 16), ("pcg@chunk=32", 32), ("pcg@tol=1e-4@chunk=6", 6), ("mixed", 16),
                                        ("mixed@chunk=32", 32), ("refine", None), ("refine@chunk=32", 32),
                                        ("refine@chunk=4@tol=1e-9", 4), ("refine@tol=1e-6@chunk=16", 16)])
def test_chunk_of_a_solver_string(monkeypatch, spec, chunk, filtered):
    from ngspsr import solver
    seen = []

    def pcg(system, b, tol=1e-5, maxiter=-1, chunk=32, x_out=None, raise_on_cap=True, filt=None):
        seen.append((chunk, filt))
        return b.float(), solver.SolveInfo(1, 0.0)

    filt = object() if filtered else None
    monkeypatch.setattr(solver, "pcg", pcg)
    monkeypatch.setattr(solver, "system_filter", lambda system: filt)
    solver.solve(_System(), torch.tensor([1.0, 2.0, 3.0], dtype=torch.float64), spec)
    if chunk is None:
        chunk = 8 if filtered else 16
    assert seen and all(c == chunk for c, _ in seen)
    assert all(f is (filt if spec.startswith("refine") else None) for _, f in seen)
    assert solver.parse_solver(spec)[1].get("chunk") == (chunk if "chunk" in spec else solver.DEFAULTS[spec]["chunk"])
