"""Tensor-material assembly from per-tet records (k_tet_tensor, k_assemble_tensor_staged) against the
lane-per-entry kernel it replaces (EMG_FORCE_TWO_PHASE), itself pinned against the oracle in
test_assembly_gpu.py."""
import numpy as np
import pytest

from emerge_amd import _lib, meshgen
from emerge_amd.assembly import EXACT_FACE_MASS, FORCE_TWO_PHASE, GPUPattern

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 1, 1), (5, 4, 3), (9, 7, 6)])
@pytest.mark.parametrize("flags", [0, EXACT_FACE_MASS])
@pytest.mark.parametrize("kind", ["full", "diagonal"])
def test_staged_equals_direct(cuda, dims, flags, kind):
    """Non-symmetric complex tensors (the edge-face blocks are mirrored by transposition) and diagonal
    ones, from one chunk of entries to many with a remainder.  Both kernels sum the same terms, at most
    9 per curl and 4 per mass entry and tet, at most 64 tets, in another order: the difference is below
    64 * 13 * 4 unit roundoffs of the largest element entry, which the largest assembled entry of
    either mode pair bounds to within the cancellation of a Kuhn mesh (a factor 16)."""
    import torch
    mesh = meshgen.structured_box(*dims, size=(1.0, 0.8, 0.6), jitter=0.1, seed=5)
    pat = GPUPattern(mesh)
    rng = np.random.default_rng(sum(dims))
    m = rng.standard_normal((2, mesh.n_tets, 3, 3)) + 1j * rng.standard_normal((2, mesh.n_tets, 3, 3))
    if kind == "diagonal":
        m *= np.eye(3)
    mm, ms = (torch.from_numpy(np.ascontiguousarray(a)).to(cuda) for a in m)
    L = _lib.load()
    out = []
    for f in (flags, flags | FORCE_TWO_PHASE):
        E = torch.full((pat.nnz,), complex(np.nan, np.nan), dtype=torch.complex128, device=cuda)
        B = torch.full_like(E, complex(np.nan, np.nan))
        _lib.check(L.emg_assemble_tensor(pat.handle, _lib.ptr(pat.nodes), _lib.ptr(pat.tets), _lib.ptr(mm), _lib.ptr(ms),
                                         f, _lib.ptr(E), _lib.ptr(B), _lib.stream_ptr()), "emg_assemble_tensor")
        out.append((E, B))
    for a, b in zip(*out):
        assert torch.all(torch.isfinite(torch.view_as_real(a)))
        assert float((a - b).abs().max()) <= 64 * 13 * 4 * 16 * 2.0 ** -53 * float(b.abs().max())


@pytest.mark.parametrize("tets", [64, 65, 96, 97, 120])
@pytest.mark.parametrize("flags", [0, EXACT_FACE_MASS])
def test_staged_equals_direct_where_chunks_hold_many_tets(cuda, tets, flags):
    """The layouts of 64, 96 and 128 records, at their edges: a fan of tets round one edge, whose row makes a chunk
    of all of them.  Bound as in test_staged_equals_direct, with up to 120 tets per entry."""
    import torch
    from tests.test_assembly_chunks_gpu import _fan
    mesh = _fan(tets)
    pat = GPUPattern(mesh)
    rng = np.random.default_rng(tets)
    m = rng.standard_normal((2, mesh.n_tets, 3, 3)) + 1j * rng.standard_normal((2, mesh.n_tets, 3, 3))
    mm, ms = (torch.from_numpy(np.ascontiguousarray(a)).to(cuda) for a in m)
    L = _lib.load()
    print(f"tensor fan {tets} flags={flags}", flush=True)
    out = []
    for f in (flags, flags | FORCE_TWO_PHASE):
        E = torch.full((pat.nnz,), complex(np.nan, np.nan), dtype=torch.complex128, device=cuda)
        B = torch.full_like(E, complex(np.nan, np.nan))
        _lib.check(L.emg_assemble_tensor(pat.handle, _lib.ptr(pat.nodes), _lib.ptr(pat.tets), _lib.ptr(mm), _lib.ptr(ms),
                                         f, _lib.ptr(E), _lib.ptr(B), _lib.stream_ptr()), "emg_assemble_tensor")
        out.append((E, B))
    for a, b in zip(*out):
        assert float((a - b).abs().max()) <= 120 * 13 * 4 * 16 * 2.0 ** -53 * float(b.abs().max())
