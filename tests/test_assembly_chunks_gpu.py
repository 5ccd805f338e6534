"""The fused assembly's chunks of 512 entries at their edges, against the two-phase kernels: a row longer
than a chunk (a fan of tets round one edge), chunks that begin and end inside rows, a last chunk with a
remainder, several chunks per run, and value arrays at every 16-byte place within a 128-byte line."""
import numpy as np
import pytest

from emerge_amd import _lib, meshgen
from emerge_amd.assembly import EXACT_FACE_MASS, FORCE_TWO_PHASE, GPUPattern
from emerge_amd.mesh import Mesh3D

pytestmark = pytest.mark.gpu


def _fan(n):
    """n tets round the edge (0, 1): its row holds 1 + 3 n edges and 3 n faces."""
    a = 2 * np.pi * np.arange(n) / n
    nodes = np.concatenate([[[0, 0], [0, 0], [-1, 1]], np.stack([np.cos(a), np.sin(a), 0.1 * np.cos(3 * a)])], axis=1)
    ring = 2 + np.arange(n)
    return Mesh3D(nodes, np.stack([np.zeros(n, int), np.ones(n, int), ring, np.roll(ring, -1)]))


MESHES = {"fan 120": lambda: _fan(120), "fan 30": lambda: _fan(30),
          "1 hex": lambda: meshgen.structured_box(1, 1, 1, jitter=0.0, seed=0),
          "5x4x3": lambda: meshgen.structured_box(5, 4, 3, jitter=0.1, seed=3),
          "13x11x10": lambda: meshgen.structured_box(13, 11, 10, jitter=0.1, seed=4)}


@pytest.mark.parametrize("name", list(MESHES))
@pytest.mark.parametrize("flags", [0, EXACT_FACE_MASS])
def test_chunks_equal_two_phase(cuda, name, flags):
    """Both paths sum the same terms, at most 9 per curl and 4 per mass entry and tet and at most 128
    tets, in another order: within 128 * 13 * 4 unit roundoffs of the largest element entry, which the
    largest assembled entry bounds to within the cancellation between tets (a factor 16)."""
    import torch
    mesh = MESHES[name]()
    pat = GPUPattern(mesh)
    rng = np.random.default_rng(mesh.n_tets)
    eps, nu = (torch.from_numpy(rng.uniform(1, 4, mesh.n_tets) * (1 - 0.1j * rng.uniform(0, 1, mesh.n_tets))).to(cuda)
               for _ in range(2))
    L = _lib.load()

    def run(f, offset):
        vals = [torch.full((pat.nnz + 16,), complex(7.0, -7.0), dtype=torch.complex128, device=cuda) for _ in range(2)]
        E, B = (v[o:o + pat.nnz] for v, o in zip(vals, (offset, (3 * offset) % 8)))
        _lib.check(L.emg_assemble_iso(pat.handle, _lib.ptr(pat.nodes), _lib.ptr(pat.tets), _lib.ptr(eps), _lib.ptr(nu),
                                      f, _lib.ptr(E), _lib.ptr(B), _lib.stream_ptr()), "emg_assemble_iso")
        for v, o in zip(vals, (offset, (3 * offset) % 8)):   # nothing beside the values is written
            assert torch.all(v[:o] == complex(7.0, -7.0)) and torch.all(v[o + pat.nnz:] == complex(7.0, -7.0))
        return E, B

    print(f"chunks {name} flags={flags} nnz={pat.nnz}", flush=True)
    ref = run(flags | FORCE_TWO_PHASE, 0)
    first = run(flags, 0)
    for a, r in zip(first, ref):
        assert float((a - r).abs().max()) <= 128 * 13 * 4 * 16 * 2.0 ** -53 * float(r.abs().max())
    for offset in range(1, 8):
        for a, b in zip(run(flags, offset), first):
            assert torch.equal(a, b)


@pytest.mark.parametrize("batch", [3, 300, 1100])
def test_batches_share_the_workgroups(cuda, batch):
    """The workgroups per mesh fall as a batch grows, to the least there are: every chunk of every mesh is
    still written, with the single assembly's values bit for bit."""
    import torch
    mesh = meshgen.structured_box(3, 3, 2, jitter=0.1, seed=7)
    pat = GPUPattern(mesh)
    rng = np.random.default_rng(batch)
    eps, nu = (torch.from_numpy(rng.uniform(1, 4, (batch, mesh.n_tets)) + 0j).to(cuda) for _ in range(2))
    nodes = torch.from_numpy(np.ascontiguousarray(np.broadcast_to(mesh.nodes.T, (batch,) + mesh.nodes.T.shape))).to(cuda)
    print(f"batch of {batch}", flush=True)
    E, B = pat.assemble_iso_batched(nodes, eps, nu)
    Es, Bs = torch.empty_like(E[0]), torch.empty_like(B[0])
    for i in (0, 1, batch // 2, batch - 1):
        pat.assemble_iso_device(eps[i].contiguous(), nu[i].contiguous(), 0, Es, Bs)
        assert torch.equal(E[i], Es) and torch.equal(B[i], Bs)


@pytest.mark.parametrize("tets", [7, 8, 12])
def test_entities_in_several_slots_of_a_tet(cuda, tets):
    """All edges of every tet one entity and all faces another, as where a single cell lies between periodic faces:
    the entry of the edges has 36 incidences per tet, 252, 288 and 432, and each is in it.  Against the blocks
    of the same tets with entities of their own, summed; at most 36 * 12 * 13 * 4 terms of them per entry."""
    import ctypes
    import torch
    rng = np.random.default_rng(tets)
    nodes = torch.from_numpy(rng.uniform(0, 1, (4 * tets, 3)) + 2 * np.arange(tets).repeat(4)[:, None]).to(cuda)
    verts = torch.arange(4 * tets, dtype=torch.int32, device=cuda).reshape(tets, 4)
    eps, nu = (torch.from_numpy(rng.uniform(1, 4, tets) * (1 - 0.1j)).to(cuda) for _ in range(2))
    mm, ms = (torch.eye(3, device=cuda) * v[:, None, None] for v in (eps, nu))
    L = _lib.load()

    def dense(ent, n_ent, call):
        h, sizes = ctypes.c_void_p(), [ctypes.c_int64() for _ in range(4)]
        _lib.check(L.emg_pattern_build(_lib.ptr(ent), tets, n_ent, _lib.stream_ptr(), ctypes.byref(h)), "emg_pattern_build")
        _lib.check(L.emg_pattern_info(h, *(ctypes.byref(v) for v in sizes)), "emg_pattern_info")
        n, nnz = sizes[0].value, sizes[1].value
        rp, ci = (torch.empty(k, dtype=torch.int32, device=cuda) for k in (n + 1, nnz))
        _lib.check(L.emg_pattern_csr(h, _lib.ptr(rp), _lib.ptr(ci), _lib.stream_ptr()), "emg_pattern_csr")
        E, B = (torch.empty(nnz, dtype=torch.complex128, device=cuda) for _ in range(2))
        args = (eps, nu) if call is L.emg_assemble_iso else (mm.contiguous(), ms.contiguous())
        _lib.check(call(h, _lib.ptr(nodes), _lib.ptr(verts), _lib.ptr(args[0]), _lib.ptr(args[1]), 0, _lib.ptr(E), _lib.ptr(B),
                        _lib.stream_ptr()), "assemble")
        out = [torch.sparse_csr_tensor(rp.long(), ci.long(), v, (n, n)).to_dense().cpu().numpy() for v in (E, B)]
        L.emg_pattern_destroy(h)
        return out

    own = torch.cat([torch.arange(6 * tets).reshape(tets, 6), 6 * tets + torch.arange(4 * tets).reshape(tets, 4)], dim=1).to(cuda, torch.int32)
    shared = torch.tensor([[0] * 6 + [1] * 4] * tets, dtype=torch.int32, device=cuda)
    fold = np.zeros((2 * 10 * tets, 4))
    for m in range(2):
        fold[m * 10 * tets: m * 10 * tets + 6 * tets, 2 * m] = 1
        fold[m * 10 * tets + 6 * tets: (m + 1) * 10 * tets, 2 * m + 1] = 1
    for call in (L.emg_assemble_iso, L.emg_assemble_tensor):
        print("several slots", tets, call.__name__, flush=True)
        for got, blocks in zip(dense(shared, 2, call), dense(own.contiguous(), 10 * tets, call)):
            tol = 36 * 12 * 13 * 4 * 2.0 ** -53 * (fold.T @ np.abs(blocks) @ fold).max()
            assert np.abs(got - fold.T @ blocks @ fold).max() <= tol
