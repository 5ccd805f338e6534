"""emg_solver_solve with a limit on the FP64 refinements."""
import ctypes

import pytest

from tests.test_packed_gpu import _problem

pytestmark = pytest.mark.gpu
F = 3e9


@pytest.mark.parametrize("fused", ["0", "1"])
@pytest.mark.parametrize("poly", [1, 6])
def test_a_limited_solve_gets_a_hundredfold_from_each_refinement(cuda, fused, poly, monkeypatch):
    """Restart 150 holds the steps of a hundredfold reduction here, so r refinements leave at most 1e-2^r.  A
    cycle ends by its complex64 estimate, which is off by a few hundred roundings of 6e-8 relative to the
    cycle's start, 2e-5 of it against the 1e-2 at its end: a factor 1.01 per refinement covers that."""
    import torch
    from emerge_amd import _lib
    from emerge_amd.fdsolve import GPUSolver
    monkeypatch.setenv("EMG_FUSED_STEPS", fused)
    prob = _problem("air", (16, 8, 4))
    K, b = prob.system(F), prob.rhs(prob.ports[0], F)
    s = GPUSolver(prob, precision=32, restart=150, poly_degree=poly)
    s.set_matrix(K, F)
    for limit in (1, 2, 3, 4, 5):
        x, info = torch.zeros_like(b), _lib.SolveInfo()
        _lib.check(s.L.emg_solver_solve(s.h, _lib.ptr(b), _lib.ptr(x), 1e-11, 20000, limit, ctypes.byref(info),
                                        _lib.stream_ptr()), "emg_solver_solve")
        print("limit", limit, "steps", info.iterations, "residual", info.residual, flush=True)
        assert info.refinements == limit and info.residual <= (1.01e-2) ** limit
