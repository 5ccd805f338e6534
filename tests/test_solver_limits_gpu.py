"""Patterns at and past the limits of the products that gather x for 64 rows (1,024 distinct columns, 8,192 blocks) and of
the fused steps (512 distinct columns per row, 8,192 candidates): past them the general forms run."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from tests.test_step_kernels_gpu import _two_steps

pytestmark = pytest.mark.gpu


def _matrix(rng, columns, ne):
    """Values on the entity pattern whose entity e lists columns[e]: (rowptr, cols, vals) and the scipy matrix."""
    deg = np.array([len(c) for c in columns])
    ptr = np.concatenate([[0], np.cumsum(2 * deg)])
    rowptr = np.concatenate([ptr[:-1], ptr + ptr[-1]]).astype(np.int32)
    half = np.concatenate([np.concatenate([c, c + ne]) for c in columns])
    cols = np.concatenate([half, half]).astype(np.int32)
    vals = rng.standard_normal(cols.size) + 1j * rng.standard_normal(cols.size)
    A = sp.csr_matrix((vals, cols, rowptr), shape=(2 * ne, 2 * ne))
    A.data[A.indices == np.repeat(np.arange(2 * ne), np.diff(rowptr))] += 4 * np.sqrt(2 * deg.max())   # a diagonal to lean on
    return A


class _Solver:
    def __init__(self, cuda, A, precision, restart=10):
        import torch
        from emerge_amd import _lib
        self.L, self.lib, self.h = _lib.load(), _lib, ctypes.c_void_p()
        self.t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
        self.keep = [self.t(A.indptr.astype(np.int32)), self.t(A.indices.astype(np.int32)), self.t(A.data)]
        rp, ci, self.vals = self.keep
        _lib.check(self.L.emg_solver_create(A.shape[0], A.nnz, _lib.ptr(rp), _lib.ptr(ci), restart, precision,
                                            ctypes.byref(self.h)),
                   "emg_solver_create")

    def matrix(self):
        self.lib.check(self.L.emg_solver_set_matrix(self.h, self.lib.ptr(self.vals), None, self.lib.stream_ptr()), "set_matrix")

    def __del__(self):
        self.L.emg_solver_destroy(self.h)


@pytest.mark.parametrize("deg,pool,local", [(16, None, True), (17, None, False), (128, 1000, True), (129, 1000, False), (40, 9000, False)])
@pytest.mark.parametrize("precision", [32, 64])
def test_local_columns_at_their_limits(cuda, deg, pool, local, precision, monkeypatch):
    """deg columns per entity of 64 x 3 + 5 rows: each its own (64 x 16 = 1,024 distinct, and 17 x 64), or of `pool` (64 x 128 =
    8,192 blocks, and 64 x 129).  Sums of 2 deg products of rounded entries: |err_i| <= (2 * 2 deg + 8) u sum_j
    |K_ij| |x_j|."""
    import torch
    monkeypatch.setenv("EMG_LOCAL_COLUMNS", "1")
    ne = max(64 * deg * 2, pool or 0)
    rng = np.random.default_rng(deg)
    rows = 64 * 3 + 5
    cols = [np.sort((np.arange(deg) * 64 + e % 64) % ne if pool is None else rng.choice(pool, deg, replace=False)) for e in range(rows)]
    A = _matrix(rng, cols + [np.array([e]) for e in range(rows, ne)], ne)
    print("local", deg, pool, precision, flush=True)
    s = _Solver(cuda, A, precision)
    s.matrix()
    lanes, ms = (ctypes.c_int * 2)(), (ctypes.c_float * 8)()
    s.lib.check(s.L.emg_solver_spmv_tuning(s.h, lanes, ms), "tuning")
    assert (ms[4 if precision == 32 else 0] == 0) == local      # no search: the form of one shape
    dt = np.complex64 if precision == 32 else np.complex128
    x = (rng.standard_normal(2 * ne) + 1j * rng.standard_normal(2 * ne)).astype(dt)
    xd = s.t(x)
    y = torch.empty_like(xd)
    s.lib.check(s.L.emg_solver_apply(s.h, precision, s.lib.ptr(xd), s.lib.ptr(y), s.lib.stream_ptr()), "emg_solver_apply")
    u = 2.0 ** -24 if precision == 32 else 2.0 ** -53
    xh = x.astype(np.complex128)
    assert np.all(np.abs(y.cpu().numpy() - A @ xh) <= (4 * deg + 8) * u * (abs(A) @ np.abs(xh)))


@pytest.mark.parametrize("ne,np2,deg", [(400, 300, 60), (512, 512, 300), (900, 300, 60), (400, 2000, 100), (1500, 300, 1100)])
def test_fused_steps_at_their_limits(cuda, ne, np2, deg, monkeypatch):
    """Gradients of 4 nodes per row on random patterns: every row within the limits, at 512 distinct columns, with more in H, with
    more in K G, and with more than 8,192 candidates.  Two steps as in test_step_kernels_gpu.py."""
    import torch
    monkeypatch.setenv("EMG_FUSED_STEPS", "1")
    rng = np.random.default_rng(ne + deg)
    cols = [np.unique(np.append(rng.choice(ne, deg, replace=False), e)) for e in range(ne)]
    A = _matrix(rng, cols, ne)
    nodes = np.sort((4 * np.arange(2 * ne)[:, None] + np.arange(4)) % np2, axis=1).ravel()
    G = sp.csr_matrix((rng.standard_normal(8 * ne), nodes, np.arange(0, 8 * ne + 1, 4)), shape=(2 * ne, np2))
    T = G.T.tocsr()
    T.sort_indices()
    s = _Solver(cuda, A, 32)
    g = [s.t(a) for a in (G.indptr.astype(np.int32), G.indices.astype(np.int32), G.data, T.indptr.astype(np.int32),
                          T.indices.astype(np.int32), T.data)]
    print("fused", ne, np2, deg, flush=True)
    s.lib.check(s.L.emg_solver_set_gradient(s.h, np2, *(s.lib.ptr(a) for a in g), s.lib.stream_ptr()), "set_gradient")
    s.matrix()
    coef = np.exp(0.3j * np.arange(3)) / (0.8 + 0.4 * np.arange(3)) / 4
    s.lib.check(s.L.emg_solver_set_poly(s.h, 3, ctypes.c_void_p(coef.ctypes.data)), "emg_solver_set_poly")
    b = rng.standard_normal(2 * ne) + 1j * rng.standard_normal(2 * ne)
    bd = s.t(b)
    x, info = torch.zeros_like(bd), s.lib.SolveInfo()
    s.lib.check(s.L.emg_solver_solve(s.h, s.lib.ptr(bd), s.lib.ptr(x), 1e-30, 2, 1, ctypes.byref(info), s.lib.stream_ptr()), "solve")
    assert info.iterations == 2

    def operators(dtype):
        e = np.arange(ne)
        a, p, q, f = (np.asarray(A[i, j]).ravel() for i, j in ((e, e), (e, e + ne), (e + ne, e), (e + ne, e + ne)))
        det = a * f - p * q
        J = sp.bmat([[sp.diags(f / det), sp.diags(-p / det)], [sp.diags(-q / det), sp.diags(a / det)]]).tocsr().astype(dtype)
        D = (1 / np.asarray(G.multiply(A @ G).sum(axis=0)).ravel()).astype(dtype)
        Gr = G.astype(np.zeros(1, dtype).real.dtype)
        return A.astype(dtype), lambda r: J @ r + Gr @ (D * (Gr.T @ r))
    want = _two_steps(*operators(np.complex128), coef, b)
    rough = _two_steps(*operators(np.complex64), coef, b.astype(np.complex64))
    size = np.linalg.norm(want)
    err, tol = np.linalg.norm(x.cpu().numpy() - want) / size, 16 * np.linalg.norm(rough - want) / size + 64 * 2.0 ** -24
    print("error", err, "of", tol, flush=True)
    assert err <= tol


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("shared", [0, 1, 3])
@pytest.mark.parametrize("ne", [500, 70001])
@pytest.mark.parametrize("restart", [10, 150])
def test_a_krylov_space_that_ends_early(cuda, ne, shared, precision, restart):
    """K M is the identity but for the 2 `shared` columns that every row lists, so the Krylov space holds at most 2 shared + 2
    vectors: the next one cancels to rounding.  A space is looked at every 4 (2) steps, and complex64 may begin it
    anew up to 4 times on the way to 1e-13: both precisions reach it in these steps."""
    import torch
    rng = np.random.default_rng(ne + shared)
    A = _matrix(rng, [np.unique(np.append(np.arange(shared), e)) for e in range(ne)], ne)
    s = _Solver(cuda, A, precision, restart)
    s.matrix()
    b = rng.standard_normal(2 * ne) + 1j * rng.standard_normal(2 * ne)
    bd = s.t(b)
    x, info = torch.zeros_like(bd), s.lib.SolveInfo()
    print("early", ne, shared, precision, restart, flush=True)
    s.lib.check(s.L.emg_solver_solve(s.h, s.lib.ptr(bd), s.lib.ptr(x), 1e-13, 200, 0, ctypes.byref(info), s.lib.stream_ptr()), "solve")
    print("steps", info.iterations, "residual", info.residual, flush=True)
    assert info.converged and info.iterations <= (2 * shared + 2 + 4) * (4 if precision == 32 else 1)
    assert np.linalg.norm(b - A @ x.cpu().numpy()) <= 2e-13 * np.linalg.norm(b)
