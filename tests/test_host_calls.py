"""What the library's host code allocates, launches and waits for, recorded on the CPU (tests/hip_recorder.c)."""
import pytest

from tests.host_calls import run

PATTERN = """
def pattern(nt):
    h = P()
    te = np.zeros((nt, 10), np.int32)
    assert L.emg_pattern_build(at(te), nt, 20, P(7), ctypes.byref(h)) == 0
    rec.rec_clear()
    return h
a = np.zeros(64)
def tensor(h, stream):
    rc = L.emg_assemble_tensor(h, at(a), at(a), at(a), at(a), 0, at(a), at(a), P(stream))
    out([rc] + log())
"""


def _kernels(lines):
    return [x.split()[1] for x in lines if x.startswith("launch")]


def test_tensor_assemblies_on_two_streams_follow_each_other(tmp_path):
    """The records of a pattern are one buffer: a call on another stream begins behind the last reader of the
    call before."""
    first, second, third = run(PATTERN + "h = pattern(4)\ntensor(h, 8)\ntensor(h, 9)\ntensor(h, 8)\n", tmp_path)
    two = ["k_tet_tensor", "k_assemble_tensor_staged"]
    for lines in (first, second, third):
        assert lines[0] == 0 and _kernels(lines[1:]) == two
    event = first[-1].split()[2]
    assert first[-1] == f"record event {event} stream 8"
    for lines, stream in ((second, 9), (third, 8)):
        assert lines[1] == f"stream {stream} waits for event {event}"
        assert lines[-1] == f"record event {event} stream {stream}"


ISO = "assert L.emg_assemble_iso(h, at(a), at(a), at(a), at(a), 0, at(a), at(a), P(8)) == 0\nrec.rec_clear()\n"


@pytest.mark.parametrize("nt", [4, 60000])
def test_the_first_assembly_takes_over_the_build_s_buffer(tmp_path, nt):
    """The sort buffer that a build leaves serves as the records of whichever assembly comes first, at every size
    of mesh: that one allocates nothing, the other allocates its own, and a pattern that sees one kind of
    media holds one buffer."""
    tensor_first, tensor_after_iso, again = run(PATTERN + f"h = pattern({nt})\ntensor(h, 8)\n"
                                                f"h = pattern({nt})\n{ISO}tensor(h, 8)\ntensor(h, 8)\n", tmp_path)
    assert not any("malloc" in x for x in tensor_first[1:] + again[1:])
    assert [x for x in tensor_after_iso[1:] if "malloc" in x] == [f"malloc {nt * 896} -> 0"]


@pytest.mark.parametrize("nt", [4, 60000])
def test_tensor_assembly_under_capture_uses_no_memory_of_the_pattern(tmp_path, nt):
    """A captured call replays on any stream, so it neither allocates nor uses the pattern's records."""
    (lines,) = run(PATTERN + f"h = pattern({nt})\nrec.rec_capturing(1)\ntensor(h, 8)\n", tmp_path)
    assert lines[0] == 0 and len(lines) == 2 and _kernels(lines[1:]) == ["k_assemble"]


def test_tensor_assembly_without_memory_for_the_records(tmp_path):
    """A mesh whose records do not fit is assembled as before there were any; with memory, from them."""
    none, some = run(PATTERN + "h = pattern(60000)\n" + ISO + "rec.rec_budget(rec.rec_used())\ntensor(h, 8)\n"
                     "rec.rec_budget(2 ** 62)\ntensor(h, 8)\n", tmp_path)
    assert none[0] == 0 and _kernels(none[1:]) == ["k_assemble"]
    assert some[0] == 0 and _kernels(some[1:]) == ["k_tet_tensor", "k_assemble_tensor_staged"]


SOLVER = """
def solver(precision, n=20, restart=10):
    s = P()
    rp = np.zeros(n + 1, np.int32)
    rp[1:] = np.arange(1, n + 1) * 2                     # entity e's rows list entity e: 2 x 2 blocks
    c = np.stack([np.arange(n) % (n // 2), np.arange(n) % (n // 2) + n // 2], axis=1).astype(np.int32).ravel()
    rc = L.emg_solver_create(n, 2 * n, at(rp), at(c), restart, precision, ctypes.byref(s))
    return rc, s
v, x = np.zeros(4000), np.zeros(4000)
info = _lib.SolveInfo()
"""


@pytest.mark.parametrize("precision", [32, 64])
def test_a_solve_leaves_nothing_in_flight(tmp_path, precision):
    """emg_solver_solve synchronises its stream: no launch or copy follows its last wait, so that the caller's
    next call may come on another stream."""
    (lines,) = run(SOLVER + f"""
rc, s = solver({precision})
assert rc == 0 and L.emg_solver_set_matrix(s, at(v), None, P(9)) == 0
rec.rec_clear()
out([L.emg_solver_solve(s, at(v), at(x), 1e-8, 100, 0, ctypes.byref(info), P(9))] + log())
""", tmp_path)
    assert lines[0] == 0 and lines[-1] == "wait stream 9"
