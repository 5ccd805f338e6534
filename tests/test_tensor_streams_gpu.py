"""Tensor assemblies of one pattern on several streams and in a captured graph."""
import numpy as np
import pytest

from emerge_amd import _lib, meshgen
from emerge_amd.assembly import GPUPattern

pytestmark = pytest.mark.gpu


def _setup(cuda, variants):
    import torch
    mesh = meshgen.structured_box(13, 11, 10, size=(1.0, 0.8, 0.6), jitter=0.1, seed=5)
    rng = np.random.default_rng(3)
    m = rng.standard_normal((variants, 2, mesh.n_tets, 3, 3)) + 1j * rng.standard_normal((variants, 2, mesh.n_tets, 3, 3))
    return GPUPattern(mesh), torch.from_numpy(m).to(cuda)


def _assemble(pat, m, E, B):
    _lib.check(_lib.load().emg_assemble_tensor(pat.handle, _lib.ptr(pat.nodes), _lib.ptr(pat.tets), _lib.ptr(m[0]),
                                               _lib.ptr(m[1]), 0, _lib.ptr(E), _lib.ptr(B), _lib.stream_ptr()),
               "emg_assemble_tensor")


def test_two_streams_keep_their_media_apart(cuda):
    """Calls on two streams, without a wait between them, give each medium's values bit for bit."""
    import torch
    pat, m = _setup(cuda, 6)
    new = lambda: torch.empty((6, pat.nnz), dtype=torch.complex128, device=cuda)
    E, B, E0, B0 = new(), new(), new(), new()
    for v in range(6):
        _assemble(pat, m[v], E0[v], B0[v])
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    print("two streams", flush=True)
    for v in range(6):
        with torch.cuda.stream(streams[v % 2]):
            _assemble(pat, m[v], E[v], B[v])
    torch.cuda.synchronize()
    assert torch.equal(E, E0) and torch.equal(B, B0)


def test_captured_call_replays_beside_eager_ones(cuda):
    """A graph holds no record of the pattern's: replays between eager calls with another medium give the
    captured medium's values, to the bound of test_tensor_assembly_gpu.py (the same sums in another order)."""
    import torch
    pat, m = _setup(cuda, 2)
    new = lambda: torch.empty(pat.nnz, dtype=torch.complex128, device=cuda)
    E0, B0, E, B, Ex, Bx = (new() for _ in range(6))
    _assemble(pat, m[0], E0, B0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    print("capture", flush=True)
    with torch.cuda.graph(graph):
        _assemble(pat, m[0], E, B)
    side = torch.cuda.Stream()
    for _ in range(3):
        E.zero_()
        B.zero_()
        torch.cuda.synchronize()
        graph.replay()
        with torch.cuda.stream(side):
            _assemble(pat, m[1], Ex, Bx)
        torch.cuda.synchronize()
        for a, b in ((E, E0), (B, B0)):
            assert float((a - b).abs().max()) <= 64 * 13 * 4 * 16 * 2.0 ** -53 * float(b.abs().max())
