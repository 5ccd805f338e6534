"""The rounding of the complex64 products that give a row few lanes."""
import numpy as np
import pytest

from tests.test_packed_gpu import _problem, _rand

pytestmark = pytest.mark.gpu


def _fma(a, b, c):
    """float32 a * b + c, rounded once (the product of two float32 is exact in float64)."""
    return (a.astype(np.float64) * b + c).astype(np.float32)


def _sixteen_lanes(A, x):
    """A x in complex64 as 16 lanes per row form it: each sums every sixteenth 2 x 2 block's products, then the lanes
    add up in pairs, all in FP32 with fused multiply-adds."""
    n, width = A.shape[0], 64
    deg = np.diff(A.indptr) // 2
    assert deg.max() <= width
    k = np.arange(width)
    at = A.indptr[:-1, None] + np.minimum(k, deg[:, None] - 1)
    live = (k < deg[:, None])
    def pair(off):
        v = np.where(live, A.data[at + off * deg[:, None]], 0).astype(np.complex64)
        return v, np.where(live, x[A.indices[at + off * deg[:, None]]], 0).astype(np.complex64)
    def mul(a, b):
        return _fma(a.real, b.real, -(a.imag * b.imag)), _fma(a.real, b.imag, a.imag * b.real)
    (v0, x0), (v1, x1) = pair(0), pair(1)
    (r0, i0), (r1, i1) = mul(v0, x0), mul(v1, x1)
    out = []
    for block in (r0 + r1, i0 + i1):
        lanes = np.zeros((n, 16), np.float32)
        for t in range(0, width, 16):
            lanes = lanes + block[:, t:t + 16]
        while lanes.shape[1] > 1:
            lanes = lanes[:, ::2] + lanes[:, 1::2]
        assert lanes.dtype == np.float32
        out.append(lanes[:, 0])
    return out[0] + 1j * out[1].astype(np.float64)


@pytest.mark.parametrize("medium", ["air", "lossy"])
@pytest.mark.parametrize("local", ["0", "1"])
def test_few_lanes_round_no_more_than_sixteen(cuda, medium, local, monkeypatch):
    """Products of 4 and 8 lanes per row are no further from the 64-bit product, in the mean square over 20,000 rows,
    than the sums of 16 shorter chains."""
    import torch
    from emerge_amd import _lib
    from emerge_amd.fdsolve import GPUSolver
    monkeypatch.setenv("EMG_LOCAL_COLUMNS", local)
    prob = _problem(medium, (16, 8, 4))
    K = prob.system(3e9)
    s = GPUSolver(prob, precision=32, preconditioner="jacobi")
    s.set_matrix(K)
    x = _rand(prob, prob.N, 3, torch.complex64) * prob.mask
    y = torch.empty_like(x)
    print("rounding", medium, local, flush=True)
    _lib.check(_lib.load().emg_solver_apply(s.h, 32, _lib.ptr(x), _lib.ptr(y), _lib.stream_ptr()), "emg_solver_apply")
    A, xh, m = prob.to_scipy(K), x.cpu().numpy(), prob.mask.cpu().numpy().astype(bool)
    exact = (A @ xh.astype(np.complex128))[m]
    err, ref = (np.linalg.norm(v[m] - exact) / np.linalg.norm(exact) for v in (y.cpu().numpy(), _sixteen_lanes(A, xh)))
    print("error", err, "sixteen lanes", ref, flush=True)
    assert err <= ref
