"""The kernels of the Krylov steps in every form a solver may choose, through solves of two steps: the iterate is
M p(K M) (y_0 b + y_1 K M p(K M) b), so every entry of a product, of the polynomial's update, of G^T, of G and of
the block inverses is in it."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from tests.test_packed_gpu import _problem, _rand

pytestmark = pytest.mark.gpu
F = 3e9
FORMS = [("lanes 4", 32), ("lanes 8", 32), ("lanes 16", 32), ("lanes 32", 32), ("local", 32), ("fused", 32),
         ("lanes 4", 64), ("lanes 8", 64), ("lanes 16", 64), ("lanes 32", 64), ("local", 64), ("csr", 64)]
CASES = [(*form, gradient, degree) for form in FORMS for gradient, degree in ((False, 1), (False, 3), (True, 1), (True, 4))
         if gradient or form[0] != "fused"]                     # fused steps need the gradient


def _operators(prob, K, gradient, dtype):
    """K with PEC rows and columns replaced by the identity's, and r -> M r, as plain scipy in dtype."""
    m = prob.mask.cpu().numpy().astype(bool)
    keep = sp.diags(m.astype(float))
    A = (keep @ prob.to_scipy(K) @ keep + sp.diags((~m).astype(float))).tocsr()
    ne = prob.N // 2
    d = A.diagonal()
    e = np.arange(ne)
    a, b, c, f = d[:ne], np.asarray(A[e, e + ne]).ravel(), np.asarray(A[e + ne, e]).ravel(), d[ne:]
    det = a * f - b * c
    J = sp.bmat([[sp.diags(f / det), sp.diags(-b / det)], [sp.diags(-c / det), sp.diags(a / det)]]).tocsr()
    G = D = None
    if gradient:
        g = prob.gradient()
        h = lambda t: t.cpu().numpy()
        G = sp.csr_matrix((h(g.vals), h(g.cols), h(g.rowptr)), shape=(prob.N, g.np2))
        s = np.asarray((G.multiply(A @ G)).sum(axis=0)).ravel()      # diag(G^T K G)
        D = np.where(s != 0, 1 / np.where(s != 0, s, 1), 0).astype(dtype)
        G = G.astype(np.zeros(1, dtype).real.dtype)
    A, J = A.astype(dtype), J.astype(dtype)
    return A, lambda r: J @ r + (0 if G is None else G @ (D * (G.T @ r)))


def _two_steps(A, M, coef, b):
    """The minimiser of ||b - K x|| over M p(K M) span{v_0, v_1}."""
    dt = b.dtype

    def precondition(x):
        q, y = x, (coef[0] * x).astype(dt)
        for i in range(len(coef) - 1):
            q = (q - coef[i] * (A @ M(q))).astype(dt)
            y = (y + coef[i + 1] * q).astype(dt)
        return M(y) if len(coef) > 1 else M(x)
    v0 = (b / np.linalg.norm(b)).astype(dt)
    w0 = A @ precondition(v0)
    v1 = w0 - np.vdot(v0, w0).astype(dt) * v0
    v1 = (v1 / np.linalg.norm(v1)).astype(dt)
    W = np.stack([w0, A @ precondition(v1)], axis=1).astype(np.complex128)
    y = np.linalg.lstsq(W, b.astype(np.complex128), rcond=None)[0]
    return precondition((y[0] * v0 + y[1] * v1).astype(dt)).astype(np.complex128)


@pytest.mark.parametrize("form,precision,gradient,degree", CASES)
@pytest.mark.parametrize("medium,dims", [("mixed", (10, 5, 2)), ("lossy", (11, 7, 5))])
def test_two_steps_match_scipy(cuda, form, precision, gradient, degree, medium, dims, monkeypatch):
    """Against the same two steps in scipy and complex128.  The same in scipy and complex64 says what rounding does to
    them: the solver's sums in another order may be 16 times as far off, scaled by the unit roundoffs'
    ratio for complex128, and no closer than 64 roundings.  An entry lost in one row would move that row by its own size."""
    import torch
    from emerge_amd import _lib
    from emerge_amd.fdsolve import GPUSolver
    lanes = form.split()[1] if form.startswith("lanes") else "16"
    monkeypatch.setenv("EMG_SPMV_BLK_LANES", lanes)
    monkeypatch.setenv("EMG_GT_LANES", {"4": "4", "32": "16"}.get(lanes, "8"))
    monkeypatch.setenv("EMG_LOCAL_COLUMNS", str(int(form == "local")))
    monkeypatch.setenv("EMG_FUSED_STEPS", str(int(form == "fused")))
    monkeypatch.setenv("EMG_PACKED_MATRIX", str(int(form != "csr")))
    prob = _problem(medium, dims)
    K = prob.system(F)
    s = GPUSolver(prob, precision=precision, restart=10, poly_degree=1,
                  preconditioner="hybrid" if gradient else "jacobi")
    s.set_matrix(K)
    b = _rand(prob, prob.N, 9, torch.complex128) * prob.mask
    coef = np.exp(0.3j * np.arange(degree)) / (0.8 + 0.4 * np.arange(degree))
    L = _lib.load()
    _lib.check(L.emg_solver_set_poly(s.h, degree, ctypes.c_void_p(coef.ctypes.data)), "emg_solver_set_poly")
    x, info = torch.zeros_like(b), _lib.SolveInfo()
    print("steps", form, precision, gradient, degree, medium, flush=True)
    _lib.check(L.emg_solver_solve(s.h, _lib.ptr(b), _lib.ptr(x), 1e-30, 2, 1, ctypes.byref(info), _lib.stream_ptr()),
               "emg_solver_solve")
    assert info.iterations == 2
    bh = b.cpu().numpy()
    want = _two_steps(*_operators(prob, K, gradient, np.complex128), coef, bh)
    rough = _two_steps(*_operators(prob, K, gradient, np.complex64), coef, bh.astype(np.complex64))
    size = np.linalg.norm(want)
    tol = 16 * np.linalg.norm(rough - want) / size + 64 * 2.0 ** -24
    if precision == 64:
        tol *= 2.0 ** -29
    err = np.linalg.norm(x.cpu().numpy() - want) / size
    print("error", err, "of", tol, flush=True)
    assert err <= tol
