"""The fused steps of small complex64 solves (products with K, K G, G^T K and G^T K G in one launch) against
the separate launches they replace (EMG_FUSED_STEPS=0)."""
import numpy as np
import pytest

from tests.test_packed_gpu import _problem

pytestmark = pytest.mark.gpu
F = 3e9


def _solver(prob, monkeypatch, fused, precision=32, poly=6, **kw):
    from emerge_amd.fdsolve import GPUSolver
    monkeypatch.setenv("EMG_FUSED_STEPS", str(fused))
    return GPUSolver(prob, precision=precision, poly_degree=poly, **kw)


@pytest.mark.parametrize("medium,dims", [("air", (9, 5, 3)), ("mixed", (10, 5, 2)), ("lossy", (11, 7, 5))])
@pytest.mark.parametrize("poly", [1, 2, 6])
@pytest.mark.parametrize("steps", [1, 3])
def test_one_cycle_matches_separate_launches(cuda, medium, dims, poly, steps, monkeypatch):
    """The iterate after one short cycle against the complex128 solver's: the fused route sums the same
    products of rounded entries in another association, so its error may be a small multiple (4) of the
    separate launches', or the rounding of a few dozen complex64 sums where theirs is less."""
    import torch
    prob = _problem(medium, dims)
    K, b = prob.system(F), prob.rhs(prob.ports[0], F)
    x = []
    for fused, precision in ((0, 64), (0, 32), (1, 32)):
        s = _solver(prob, monkeypatch, fused, precision, poly)
        s.set_matrix(K, F)
        x.append(s.solve(b, tol=1e-14, maxiter=steps * max(1, s.poly_active), max_refine=1)[0])
    n = float(torch.linalg.vector_norm(x[0]))
    e0, e1 = (float(torch.linalg.vector_norm(v - x[0])) / n for v in x[1:])
    print("one cycle", medium, "poly", poly, "steps", steps, "separate", e0, "fused", e1, flush=True)
    assert e1 <= 4 * e0 + 64 * 2.0 ** -24


@pytest.mark.parametrize("medium,dims", [("air", (16, 8, 4)), ("mixed", (16, 8, 4)), ("lossy", (20, 10, 4))])
@pytest.mark.parametrize("restart", [16, 60])
def test_solves_take_the_same_steps(cuda, medium, dims, restart, monkeypatch):
    """Whole solves, a second matrix and a second gradient (its entries in another order) on one solver:
    both routes reach tol, in steps that differ by what rounding moves a cycle's end (two looks of 4 steps,
    or a tenth).  (At restart 12 the separate launches stall or take thousands of steps, by a third more or
    fewer from run to run, so there is nothing to compare with.)"""
    import torch
    from emerge_amd import _lib
    prob = _problem(medium, dims)
    G = prob.gradient()
    rng = np.random.default_rng(1)

    def shuffled(ptr, idx, val):
        ptr, idx, val = ptr.cpu().numpy(), idx.cpu().numpy().copy(), val.cpu().numpy().copy()
        for i in range(len(ptr) - 1):
            p = ptr[i] + rng.permutation(ptr[i + 1] - ptr[i])
            idx[ptr[i]:ptr[i + 1]], val[ptr[i]:ptr[i + 1]] = idx[p], val[p]
        return torch.from_numpy(idx).to(prob.dev), torch.from_numpy(val).to(prob.dev)

    g, t = shuffled(G.rowptr, G.cols, G.vals), shuffled(G.t_rowptr, G.t_cols, G.t_vals)
    steps = []
    for fused in (0, 1):
        s = _solver(prob, monkeypatch, fused, restart=restart)
        for f, again in ((F, False), (1.1 * F, False), (F, True)):
            if again:
                _lib.check(s.L.emg_solver_set_gradient(s.h, G.np2, _lib.ptr(G.rowptr), _lib.ptr(g[0]), _lib.ptr(g[1]),
                                                       _lib.ptr(G.t_rowptr), _lib.ptr(t[0]), _lib.ptr(t[1]),
                                                       _lib.stream_ptr()), "emg_solver_set_gradient")
            s.set_matrix(prob.system(f), f)
            info = s.solve(prob.rhs(prob.ports[0], f), tol=1e-10, maxiter=60000)[1]
            assert info.converged and info.residual <= 1e-10
            steps.append(info.iterations)
    print("steps", medium, restart, steps, flush=True)
    for a, c in zip(steps[:3], steps[3:]):
        assert abs(a - c) <= max(8, 0.1 * a)
