"""The host side of the solver without a GPU: a stand-in HIP runtime
(tests/fake_hip.c), preloaded into a process of its own, whose kernels do
nothing, shows what the driver launches, polls and waits for."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

PRELUDE = """
import ctypes as C, numpy as np
from mfix_amd import _lib, leq
L = _lib.load()
leq.init(0)
def arrays(n3):
    return [leq.DeviceArray(k * n3) for k in (1, 7, 1)]
"""


@pytest.fixture(scope="session")
def fake(tmp_path_factory, native_lib):
    so = tmp_path_factory.mktemp("fake") / "fake_hip.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-pthread", "-o", str(so), str(ROOT / "tests" / "fake_hip.c")],
                   check=True)

    def run(mode, code, log):
        env = dict(os.environ, LD_PRELOAD=str(so), FAKE_HIP=mode, FAKE_HIP_LOG=str(log))
        p = subprocess.run([sys.executable, "-c", PRELUDE + code], cwd=ROOT, env=env, capture_output=True, text=True,
                           timeout=120)
        assert p.returncode == 0, p.stderr
        return p.stdout.strip(), log.read_text().splitlines() if log.exists() else []
    return run


@pytest.mark.parametrize("pc", ["DIAG", "LINE"])
def test_a_poll_leaves_the_words_of_the_one_before_alone(fake, tmp_path, pc):
    """The next poll is under way while the host reads one: its words are others."""
    _, log = fake("count", f"""
leq.grid_init(60, 60, 60)
dx, da, db = arrays(62 ** 3)
leq.bicgs_dev(dx, da, db, pc="{pc}", tol=1e-10, itmax=40)
""", tmp_path / "log")
    polls = [(int(p, 16), int(n), int(k)) for _, p, n, k in (s.split() for s in log if s.startswith("poll"))]
    assert len(polls) >= 4 and [k for _, _, k in polls] == list(range(polls[0][2], polls[0][2] + len(polls)))
    for (p, n, _), (q, m, _) in zip(polls, polls[1:]):
        assert p + 4 * (2 + n) <= q or q + 4 * (2 + m) <= p


def test_an_error_returns_when_nothing_runs_any_more(fake, tmp_path):
    """No poll is answered: the call ends with an error, and with a wait for what
    it had under way, also without the events that other entries wait for."""
    out, log = fake("silent", """
leq.grid_init(20, 20, 20)
dx, da, db = arrays(22 ** 3)
st, o = _lib.Stats(), _lib.Opts()
f = L.mfix_leq_bicgs_dev_noalloc
f.argtypes = [C.c_char_p, C.c_double, C.c_char_p, C.c_int] + [C.c_void_p] * 6
print(f(b"RSRS", 1e-10, b"DIAG", 40, dx.ptr, da.ptr, db.ptr, C.addressof(o), C.addressof(st), None))
""", tmp_path / "log")
    assert int(out) < 0
    last = max(k for k, s in enumerate(log) if s.startswith(("launch", "poll")))
    assert "wait" in log[last:]


@pytest.mark.skipif(len(os.sched_getaffinity(0)) < 2, reason="one processor: the caller's thread copies")
def test_a_failed_launch_of_a_copying_thread_is_an_error(fake, tmp_path):
    out, log = fake("threads", """
leq.grid_init(60, 60, 60)
n = 62 ** 3
ier = C.c_int(7)
x, a, b = np.zeros(n), np.zeros(7 * n), np.zeros(n)
print(L.mfix_leq_bicgs(b"u", 1, 1, *(v.ctypes.data_as(_lib.c_double_p) for v in (x, a, b)), b"RSRS", 4, 1e-4, b"DIAG", 99,
                       C.byref(ier)))
""", tmp_path / "log")
    assert any("k_move" in s for s in log)      # the caller's own launches
    assert int(out) == -103                     # MFIX_LEQ_EHIP


def test_graphs_are_destroyed_when_they_do_not_run(fake, tmp_path):
    """The FP64 systems of a batch end before the FP32 ones: the chunk of both
    that is under way by then is let run to its end before its graph goes."""
    _, log = fake("count", """
items = []
for q in range(6):
    n = 12 + 2 * q
    dx, da, db = arrays((n + 2) ** 3)
    items.append(leq.BatchSystem(n, n, n, dx, da, db, pc="DIAG", tol=1e-10, itmax=200, mixed=q % 2 == 1))
leq.batch_solve(items)
leq.finalize()
""", tmp_path / "log")
    launched, destroyed = {}, 0
    for k, s in enumerate(log):
        what, _, graph = s.partition(" ")
        if what == "launch" and graph.startswith("0x"):
            launched[graph] = k
        elif what == "destroy" and graph in launched:
            destroyed += 1
            assert "wait" in log[launched[graph]:k], f"{graph} destroyed while it ran"
    assert destroyed >= 2
