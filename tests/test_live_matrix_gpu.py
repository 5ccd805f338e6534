"""Matrix values that the caller changes in place between emg_solver_set_matrix and a solve."""
import pytest

from tests.test_packed_gpu import _problem

pytestmark = pytest.mark.gpu
F = 3e9


@pytest.mark.parametrize("medium", ["air", "mixed"])
def test_complex128_solves_and_probes_take_the_values_of_the_call(cuda, medium):
    """Precision 64: a solve is of K's values as they are then (preconditioned by those of set_matrix), and its
    residual theirs: recomputed with the CSR product it agrees up to the rounding of b - K x, 1e-13 of |b|.  The
    Arnoldi probe's first column is K M v for those values: its norm changes with them."""
    import ctypes
    import numpy as np
    import torch
    from emerge_amd import _lib
    from emerge_amd.fdsolve import GPUSolver
    prob = _problem(medium, (10, 5, 2))
    K, b = prob.system(F), prob.rhs(prob.ports[0], F)
    s = GPUSolver(prob, precision=64, restart=300, poly_degree=1)
    s.set_matrix(K, F)
    L = _lib.load()

    def probe():
        h = np.zeros(2 * 2, dtype=np.complex128)
        _lib.check(L.emg_solver_arnoldi_probe(s.h, 1, _lib.ptr(b), ctypes.c_void_p(h.ctypes.data), _lib.stream_ptr()), "probe")
        return h
    before = probe()
    K.copy_(prob.system(1.02 * F) * (1 + 0.1j))
    after = probe()
    x, info = s.solve(b, tol=1e-9)
    y = torch.empty_like(x)
    _lib.check(L.emg_spmv(prob.N, _lib.ptr(prob.pat.rowptr), _lib.ptr(prob.pat.cols), _lib.ptr(K), _lib.ptr(prob.mask),
                          _lib.ptr(x), _lib.ptr(y), _lib.stream_ptr()), "emg_spmv")
    rel = float(torch.linalg.vector_norm(b - y) / torch.linalg.vector_norm(b))
    print("live", medium, info.iterations, info.residual, rel, flush=True)
    assert info.converged and rel <= 1e-9 + 1e-13 and abs(rel - info.residual) <= 1e-13
    assert abs(after[0] - before[0]) > 0.05 * abs(before[0])
