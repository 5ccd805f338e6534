"""emg_sweep_residual and emg_basis_combine against NumPy at the edges of their work split: row lengths
0 and above the 32 columns held at a time, fewer entities than a block, grids that the XCD order does
and does not divide, row counts with a remainder, and the largest block of coefficients."""
import numpy as np
import pytest

from emerge_amd import _lib

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


def _dev(cuda, a, dtype):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a).astype(dtype)).to(cuda)


def _cplx(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


@pytest.mark.parametrize("nvec", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("ne", [1, 7, 64, 333, 8200])
def test_residual_of_ragged_rows(cuda, nvec, ne):
    """Rows of 0 to 100 column entities, 1 column outside the pattern that must be left out.  A residual
    entry is a sum of 2 deg products (a complex product and a scale: 6 roundings on each), the port term
    and the source: within (2 deg + 16) * 2 unit roundoffs of the sum of magnitudes.  The norms are sums
    of 2 ne squares of the entries returned."""
    import torch
    rng = np.random.default_rng(100 * nvec + ne)
    n = 2 * ne
    deg = rng.integers(0, 12, ne)
    deg[rng.integers(0, ne, max(1, ne // 50))] = 100
    if ne > 8:
        deg[:6] = (0, 31, 32, 33, 64, 65)
    rows = [rng.integers(0, ne, d) for d in deg]
    bad = int(np.argmax(deg))
    if deg[bad]:
        rows[bad][0] = ne
    cols = np.concatenate([np.concatenate([r, r + ne]) for r in rows] * 2).astype(np.int64)
    rowptr = np.concatenate([[0], np.cumsum(np.concatenate([2 * deg, 2 * deg]))])
    nnz = int(rowptr[-1])
    E, B = _cplx(rng, nnz), _cplx(rng, nnz)
    mask = (rng.uniform(size=n) > 0.2).astype(np.uint8)
    X = _cplx(rng, n, nvec)
    Q, qidx, c, s = _cplx(rng, 3, n), rng.integers(0, 3, nvec), _cplx(rng, nvec), rng.uniform(1, 2, nvec)
    prow = np.where(rng.uniform(size=n) < 0.3, rng.integers(0, 5, n), -1)
    Zp = _cplx(rng, 5, nvec)

    row = np.repeat(np.arange(n), np.diff(rowptr))
    ent = np.concatenate([np.concatenate([r, r]) for r in rows] * 2)
    ok = ent < ne
    ref, mag = np.zeros((n, nvec), complex), np.zeros((n, nvec))
    xg = X[np.where(ok, cols, 0) % n]
    for j in range(nvec):
        np.add.at(ref[:, j], row[ok], ((E - s[j] * B) * xg[:, j])[ok])
        np.add.at(mag[:, j], row[ok], ((abs(E) + s[j] * abs(B)) * abs(xg[:, j]))[ok])
    z = np.where(prow[:, None] >= 0, Zp[np.maximum(prow, 0)], 0)
    b = (c[:, None] * Q[qidx]).T
    ref = mask[:, None] * (b - ref - z)
    mag += abs(z) + abs(b)

    p = _lib.ptr
    d = dict(rowptr=_dev(cuda, rowptr, np.int32), cols=_dev(cuda, cols, np.int32), E=_dev(cuda, E, np.complex128),
             B=_dev(cuda, B, np.complex128), mask=_dev(cuda, mask, np.uint8), s=_dev(cuda, s, np.float64),
             X=_dev(cuda, X, np.complex128), Q=_dev(cuda, Q, np.complex128), q=_dev(cuda, qidx, np.int32),
             c=_dev(cuda, c, np.complex128), prow=_dev(cuda, prow, np.int32), Z=_dev(cuda, Zp, np.complex128))
    R = torch.full((n, nvec), complex(np.nan, np.nan), dtype=torch.complex128, device=cuda)
    norms = torch.full((2 * nvec,), np.nan, dtype=torch.float64, device=cuda)
    work = torch.full((4096 * nvec * 2,), np.nan, dtype=torch.float64, device=cuda)
    print(f"residual nvec={nvec} entities={ne}", flush=True)
    _lib.check(_lib.load().emg_sweep_residual(
        n, p(d["rowptr"]), p(d["cols"]), p(d["E"]), p(d["B"]), p(d["mask"]), nvec, p(d["s"]), p(d["X"]), p(d["Q"]),
        p(d["q"]), p(d["c"]), p(d["prow"]), p(d["Z"]), p(R), p(norms), p(work), _lib.stream_ptr()), "emg_sweep_residual")
    got, nr = R.cpu().numpy(), norms.cpu().numpy()
    lim = (2 * np.concatenate([deg, deg])[:, None] + 16) * 2 * U * mag
    assert np.all(abs(got - ref) <= lim)
    for j in range(nvec):
        for v, w in ((got[:, j], nr[2 * j]), (b[:, j] * mask, nr[2 * j + 1])):
            t = float(np.sum(abs(v) ** 2))
            assert abs(w - t) <= (n + 16) * 2 * U * t


@pytest.mark.parametrize("nvec", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("n", [2, 126, 1000])
@pytest.mark.parametrize("m", [1, 14, 2048])
def test_combine_rows(cuda, nvec, n, m):
    """X = V Y at row counts with a remainder, for one vector, an ordinary basis and the 2,048
    coefficients a call may hold: sums of m complex products, within (m + 4) * 2 unit roundoffs of the
    sum of magnitudes."""
    import torch
    m = min(m, 2048 // nvec)
    rng = np.random.default_rng(n + m + nvec)
    V, Y = _cplx(rng, m, n), _cplx(rng, nvec, m)
    X = torch.full((n, nvec), complex(np.nan, np.nan), dtype=torch.complex128, device=cuda)
    Vd, Yd = _dev(cuda, V, np.complex128), _dev(cuda, Y, np.complex128)
    print(f"combine nvec={nvec} n={n} m={m}", flush=True)
    _lib.check(_lib.load().emg_basis_combine(n, m, _lib.ptr(Vd), nvec, _lib.ptr(Yd), _lib.ptr(X), _lib.stream_ptr()),
               "emg_basis_combine")
    lim = (m + 4) * 2 * U * (abs(V).T @ abs(Y).T)
    assert np.all(abs(X.cpu().numpy() - V.T @ Y.T) <= lim)
