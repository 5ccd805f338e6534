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


@pytest.mark.parametrize("precision,local", [(32, "0"), (32, "1"), (64, "0"), (64, "1")])
def test_a_solver_is_made_wherever_its_least_buffers_fit(tmp_path, precision, local):
    """What serves speed (a second restart length of the complex64 basis, the packed copy of a complex128 K, the
    tables of the products that gather locally) is taken where the card has room, whichever buffer the memory
    ends at; what is needed without it is found by halving."""
    tries, least, most = run(SOLVER + """
def fits(budget):
    rec.rec_budget(budget)
    rc, s = solver(PRECISION, n=2000, restart=50)
    used = rec.rec_used()
    if rc == 0:
        L.emg_solver_destroy(s)
    assert rec.rec_used() == 0
    return rc == 0, used
most = fits(2 ** 62)[1]
lo, hi = 0, most
while hi - lo > 1:
    mid = (lo + hi) // 2
    lo, hi = (lo, mid) if fits(mid)[0] else (mid, hi)
out([fits(b)[0] for b in np.linspace(hi, most, 400).astype(int).tolist()])
out([hi])
out([most])
""".replace("PRECISION", str(precision)), tmp_path, env={"EMG_LOCAL_COLUMNS": local})
    assert all(tries)
    # a restart length of vectors; 16 bytes per entry of the 2,000 rows of two
    assert most[0] - least[0] >= (50 * 2000 * 8 if precision == 32 else 2000 * 2 * 16)


@pytest.mark.parametrize("precision", [32, 64])
def test_a_gradient_that_does_not_fit_gets_room(tmp_path, precision):
    """emg_solver_set_gradient on a full card: the longer half of a complex64 basis, or the packed copy of a
    complex128 K, makes room."""
    (rc,) = run(SOLVER + """
n, np2 = 2000, 300
rc, s = solver(PRECISION, n=n, restart=50)
gp, tp = np.zeros(n + 1, np.int32), np.zeros(np2 + 1, np.int32)
gp[n] = tp[np2] = 900
c = np.zeros(900, np.int32)
g = np.zeros(900)
rec.rec_budget(rec.rec_used())
out([rc, L.emg_solver_set_gradient(s, np2, at(gp), at(c), at(g), at(tp), at(c), at(g), P(9)),
     L.emg_solver_set_matrix(s, at(v.repeat(20)), None, P(9)),
     L.emg_solver_solve(s, at(v), at(x), 1e-8, 100, 0, ctypes.byref(info), P(9))])
""".replace("PRECISION", str(precision)), tmp_path, env={"EMG_FUSED_STEPS": "0"})
    assert rc == [0, 0, 0, 0]


@pytest.mark.parametrize("precision,local,lanes,searches", [(64, "0", None, 5), (64, "1", [4, 4], 0), (32, "1", [None, 4], 5)])
def test_products_of_one_shape_are_not_tuned(tmp_path, precision, local, lanes, searches):
    """A search captures and times a graph per candidate and one of what precedes them: five for the products of four
    shapes, none for those that gather x for 64 rows (precision 32 still searches for its CSR product)."""
    lines, got = run(SOLVER + f"""
rc, s = solver({precision}, n=2000)
assert rc == 0
rec.rec_clear()
out([L.emg_solver_set_matrix(s, at(v.repeat(20)), None, P(9))] + log())
n, ms = (ctypes.c_int * 2)(), (ctypes.c_float * 8)()
assert L.emg_solver_spmv_tuning(s, n, ms) == 0
out(list(n))
""", tmp_path, env={"EMG_LOCAL_COLUMNS": local})
    assert lines[0] == 0 and sum(x.startswith("capture") for x in lines[1:]) == searches
    assert lanes is None or all(want in (None, have) for want, have in zip(lanes, got))


def test_host_memory_that_runs_out_is_an_error_not_an_exception(tmp_path):
    """A table that emg_solver_set_gradient makes on the host and cannot have ends the call with an error."""
    (rcs,) = run(SOLVER + """
n, np2 = 2000, 300000
rc, s = solver(32, n=n, restart=50)
gp, tp = np.zeros(n + 1, np.int32), np.zeros(np2 + 1, np.int32)
gp[n] = tp[np2] = 900
c, g = np.zeros(900, np.int32), np.zeros(900)
rcs = [rc]
for block in (100000, 2 ** 62):
    rec.rec_host_block(block)
    rcs.append(L.emg_solver_set_gradient(s, np2, at(gp), at(c), at(g), at(tp), at(c), at(g), P(9)))
out(rcs)
""", tmp_path, env={"EMG_FUSED_STEPS": "0"})
    assert rcs == [0, -2, 0]
