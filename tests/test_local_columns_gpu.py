"""Products that gather x for 64 rows at a time into LDS (EMG_LOCAL_COLUMNS=1, used by itself on large
problems) against the CSR product, and solves with them."""
import numpy as np
import pytest

from tests.test_packed_gpu import _problem, _rand

pytestmark = pytest.mark.gpu
F = 3e9


@pytest.mark.parametrize("medium,dims", [("air", (9, 5, 3)), ("mixed", (10, 5, 2)), ("lossy", (11, 7, 5)), ("air", (16, 8, 4))])
@pytest.mark.parametrize("precision", [32, 64])
def test_product_matches_csr(cuda, medium, dims, precision, monkeypatch):
    """Row counts with and without a remainder of 64.  Bound as for the other form: at most
    4 * 64 products per row of rounded entries, |err_i| <= (2 * 64 + 8) u sum_j |K_ij| |x_j|; conductor
    DOFs of a complex128 x may hold anything."""
    import torch
    from emerge_amd import _lib
    from emerge_amd.fdsolve import GPUSolver
    monkeypatch.setenv("EMG_LOCAL_COLUMNS", "1")
    prob = _problem(medium, dims)
    K = prob.system(F)
    s = GPUSolver(prob, precision=precision, preconditioner="jacobi")
    s.set_matrix(K)
    dt = torch.complex64 if precision == 32 else torch.complex128
    m = prob.mask.cpu().numpy().astype(bool)
    x = _rand(prob, prob.N, 3, dt) * prob.mask
    xh = x.cpu().numpy().astype(np.complex128)
    if precision == 64:
        x[~torch.from_numpy(m).to(x.device)] = complex(np.inf, 1.0)
    y = torch.empty_like(x)
    L = _lib.load()
    print(f"local columns {medium} {dims} {precision}", flush=True)
    _lib.check(L.emg_solver_apply(s.h, precision, _lib.ptr(x), _lib.ptr(y), _lib.stream_ptr()), "emg_solver_apply")
    A = prob.to_scipy(K)
    assert np.diff(A.indptr).max() <= 128
    u = 2.0 ** -24 if precision == 32 else 2.0 ** -53
    err = np.abs(y.cpu().numpy() - A @ xh)[m]
    assert np.all(err <= (2 * 64 + 8) * u * (abs(A) @ np.abs(xh))[m])


@pytest.mark.parametrize("precision", [32, 64])
def test_solve_takes_the_same_steps(cuda, precision, monkeypatch):
    """Both forms sum a row's products in lanes of another number: same steps to within a look (4)."""
    from emerge_amd.fdsolve import GPUSolver
    prob = _problem("mixed", (16, 8, 4))
    K, b = prob.system(F), prob.rhs(prob.ports[0], F)
    steps = []
    monkeypatch.setenv("EMG_FUSED_STEPS", "0")
    for loc in ("0", "1"):
        monkeypatch.setenv("EMG_LOCAL_COLUMNS", loc)
        s = GPUSolver(prob, precision=precision)
        s.set_matrix(K, F)
        info = s.solve(b, tol=1e-10)[1]
        assert info.converged and info.residual <= 1e-10
        steps.append(info.iterations)
    print("steps", precision, steps, flush=True)
    assert abs(steps[0] - steps[1]) <= 4
