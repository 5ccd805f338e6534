"""The solver's packed layout (emg_krylov.hip): the planes of K with rows flagged real or complex, the
packed gradient, the multi-dot and multi-AXPY at the edges of their tiles, and the refinement cycles
that share one basis."""
import numpy as np
import pytest

from emerge_amd import meshgen
from emerge_amd.bc import Material

pytestmark = pytest.mark.gpu


def _problem(medium, dims):
    from emerge_amd import workloads
    phys = workloads.posts(*dims, freqs=[3e9])
    if medium == "lossy":
        phys.set_material(1, Material(er=2.2, tand=0.02))
    elif medium == "mixed":                      # lossy and lossless tets, real and complex rows side by side
        phys.mesh.tet_tags = np.where(phys.mesh.centers[0] < 0.02, 1, 2)
        phys.set_material(2, Material(er=4.4, tand=0.02))
    return phys.problem()


def _rand(prob, n, seed, dtype):
    import torch
    g = torch.Generator(device=prob.dev)
    g.manual_seed(seed)
    return torch.view_as_complex(torch.randn((n, 2), generator=g, dtype=torch.float64, device=prob.dev)).to(dtype).contiguous()


@pytest.mark.parametrize("medium,dims", [("air", (9, 5, 3)), ("mixed", (10, 5, 2)), ("lossy", (11, 7, 5)), ("air", (16, 8, 4))])
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("lanes", [4, 8, 16, 32])
def test_packed_product_matches_csr(cuda, medium, dims, precision, lanes, monkeypatch):
    """y = K x from the packed planes against the CSR product in complex128, entry by entry: a row sums
    at most 4 * 64 products (deg <= 64 here, asserted) of rounded entries in precision u, so
    |err_i| <= (2 * 64 + 8) u sum_j |K_ij| |x_j| covers the roundings of entries, products and sums."""
    import torch
    from emerge_amd import _lib
    from emerge_amd.fdsolve import GPUSolver
    monkeypatch.setenv("EMG_SPMV_BLK_LANES", str(lanes))
    prob = _problem(medium, dims)
    K = prob.system(3e9)
    s = GPUSolver(prob, precision=precision, preconditioner="jacobi")
    s.set_matrix(K)
    dt = torch.complex64 if precision == 32 else torch.complex128
    x = _rand(prob, prob.N, 3, dt) * prob.mask
    y = torch.empty_like(x)
    L = _lib.load()
    _lib.check(L.emg_solver_apply(s.h, precision, _lib.ptr(x), _lib.ptr(y), _lib.stream_ptr()), "emg_solver_apply")
    A = prob.to_scipy(K)
    assert np.diff(A.indptr).max() <= 128
    m = prob.mask.cpu().numpy().astype(bool)
    xh = x.cpu().numpy().astype(np.complex128)
    want = A @ xh
    size = abs(A) @ np.abs(xh)
    got = y.cpu().numpy()
    u = 2.0 ** -24 if precision == 32 else 2.0 ** -53
    assert np.all(np.abs(got - want)[m] <= (2 * 64 + 8) * u * size[m])
    assert np.all(got[~m] == 0)


def test_packed_product_leaves_conductor_values_out(cuda):
    """complex128: values of x on PEC DOFs, whatever they are, reach no other row."""
    import torch
    from emerge_amd import _lib
    from emerge_amd.fdsolve import GPUSolver
    prob = _problem("air", (9, 5, 3))
    s = GPUSolver(prob, precision=64, preconditioner="jacobi")
    s.set_matrix(prob.system(3e9))
    x = _rand(prob, prob.N, 5, torch.complex128) * prob.mask
    bad = torch.where(prob.mask.bool(), x, torch.full_like(x, complex(float("inf"), float("nan"))))
    y0, y1 = torch.empty_like(x), torch.empty_like(x)
    L = _lib.load()
    for v, y in ((x, y0), (bad, y1)):
        _lib.check(L.emg_solver_apply(s.h, 64, _lib.ptr(v), _lib.ptr(y), _lib.stream_ptr()), "emg_solver_apply")
    keep = prob.mask.bool()
    assert torch.equal(y0[keep], y1[keep])


@pytest.mark.parametrize("n", [1, 2, 255, 513, 8191, 65535, 65536, 70001])
@pytest.mark.parametrize("nv", [1, 7, 8, 9, 33])
def test_multi_dot_and_axpy(cuda, n, nv):
    """emg_mdotc and emg_maxpy against torch in complex128: errors of sums of n (nv) products, bounded by
    their lengths times the unit roundoff times the sums of magnitudes."""
    import torch
    from emerge_amd import _lib
    L = _lib.load()
    g = torch.Generator(device=cuda)
    g.manual_seed(n + nv)
    r = lambda *s: torch.view_as_complex(torch.randn((*s, 2), generator=g, dtype=torch.float64, device=cuda)).contiguous()
    V, w = r(nv, n), r(n)
    h = torch.empty(nv, dtype=torch.complex128, device=cuda)
    work = torch.empty(((nv + 7) // 8) * 1024 * 16 + 1024, dtype=torch.float64, device=cuda)
    nrm = torch.empty(4, dtype=torch.float64, device=cuda)
    u = 2.0 ** -53
    _lib.check(L.emg_mdotc(n, nv, _lib.ptr(V), _lib.ptr(w), _lib.ptr(h), _lib.ptr(work), _lib.stream_ptr()), "emg_mdotc")
    want = V.conj().resolve_conj() @ w
    assert torch.all((h - want).abs() <= 8 * (n + 8) * u * (V.abs() @ w.abs()))
    out = w.clone()
    _lib.check(L.emg_maxpy(n, nv, _lib.ptr(V), _lib.ptr(h), _lib.ptr(out), _lib.ptr(nrm), _lib.ptr(work),
                           _lib.stream_ptr()), "emg_maxpy")
    ref = w - h @ V
    assert torch.all((out - ref).abs() <= 8 * (nv + 8) * u * (w.abs() + h.abs() @ V.abs()))
    n2 = float(torch.linalg.vector_norm(out))
    assert abs(float(nrm[0]) - n2) <= 4 * (n + 8) * u * n2


@pytest.mark.parametrize("restart", [8, 20, 60, 150])
@pytest.mark.parametrize("poly", [1, 6])
def test_shared_cycles_reach_the_residual(cuda, restart, poly):
    """Complex64 cycles in FP64 refinement with bases that never fill, fill once, and fill often: the
    residual they report is the true one (recomputed by the CSR product, up to the rounding of b - K x:
    1e-13 of |b| here); where the basis (two restart lengths) holds the whole unrestarted complex128
    solve, tol is reached in at most a quarter and 16 more steps than that takes."""
    import torch
    from emerge_amd import _lib
    from emerge_amd.fdsolve import GPUSolver
    prob = _problem("mixed", (16, 8, 4))
    f = 3e9
    K = prob.system(f)
    b = prob.rhs(prob.ports[0], f)
    full = GPUSolver(prob, precision=64, restart=400, poly_degree=poly)
    full.set_matrix(K, f)
    _, ref = full.solve(b, tol=1e-11, maxiter=4000)
    assert ref.converged
    s = GPUSolver(prob, precision=32, restart=restart, poly_degree=poly)
    s.set_matrix(K, f)
    x, info = s.solve(b, tol=1e-10, maxiter=60000)
    y = torch.empty_like(x)
    _lib.check(_lib.load().emg_spmv(prob.N, _lib.ptr(prob.pat.rowptr), _lib.ptr(prob.pat.cols), _lib.ptr(K),
                                    _lib.ptr(prob.mask), _lib.ptr(x), _lib.ptr(y), _lib.stream_ptr()), "emg_spmv")
    rel = float(torch.linalg.vector_norm(b - y) / torch.linalg.vector_norm(b))
    print("restart", restart, "poly", poly, "steps", info.iterations, "of", ref.iterations, "cycles", info.refinements,
          "residual", info.residual, rel, flush=True)
    assert abs(rel - info.residual) <= 1e-13
    if 2 * restart >= ref.iterations:
        assert info.converged and rel <= 1e-10
        assert info.iterations <= 1.25 * ref.iterations + 16


def test_gradient_rows_in_any_order(cuda):
    """The packed G and G^T of rows that are not ascending, or whose two modes list their nodes in
    different orders, act as the ascending ones: the solves take the same steps to within the rounding
    of reordered sums (two steps of slack) and agree to the tolerance's multiple of the residual."""
    import torch
    from emerge_amd import _lib
    from emerge_amd.fdsolve import GPUSolver
    prob = _problem("air", (10, 5, 2))
    f = 3e9
    K = prob.system(f)
    b = prob.rhs(prob.ports[0], f)
    G = prob.gradient()
    rng = np.random.default_rng(0)

    def shuffled(ptr, idx, val):
        ptr, idx, val = ptr.cpu().numpy(), idx.cpu().numpy().copy(), val.cpu().numpy().copy()
        for i in range(len(ptr) - 1):
            p = ptr[i] + rng.permutation(ptr[i + 1] - ptr[i])
            idx[ptr[i]:ptr[i + 1]], val[ptr[i]:ptr[i + 1]] = idx[p], val[p]
        return torch.from_numpy(idx).to(prob.dev), torch.from_numpy(val).to(prob.dev)

    gc, gv = shuffled(G.rowptr, G.cols, G.vals)
    tc, tv = shuffled(G.t_rowptr, G.t_cols, G.t_vals)
    steps = []
    for cols, vals, tcols, tvals in ((G.cols, G.vals, G.t_cols, G.t_vals), (gc, gv, tc, tv)):
        for precision in (32, 64):
            s = GPUSolver(prob, precision=precision)
            _lib.check(s.L.emg_solver_set_gradient(s.h, G.np2, _lib.ptr(G.rowptr), _lib.ptr(cols), _lib.ptr(vals),
                                                   _lib.ptr(G.t_rowptr), _lib.ptr(tcols), _lib.ptr(tvals),
                                                   _lib.stream_ptr()), "emg_solver_set_gradient")
            s.set_matrix(K, f)
            x, info = s.solve(b, tol=1e-9)
            assert info.converged
            steps.append((precision, info.iterations))
    print("steps", steps, flush=True)
    for p in (32, 64):
        a, c = [n for q, n in steps if q == p]
        assert abs(a - c) <= max(4, 0.1 * a)
