"""The host analysis and plans of a factor when the process is short of threads
(the work is done by those that start) or of memory (an error, or the result),
run in a process with the limit."""
import os
import resource
import subprocess
import sys

import numpy as np
import pytest

from rchol_amd import factor as F
from rchol_amd.solver import chunk_apply_host, merge_apply_host

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import sys
import threading
import numpy as np
from rchol_amd.solver import chunk_apply_host, merge_apply_host

d = np.load(sys.argv[1])
Gs = (d["cp"], d["ri"], d["v"])
started = []
try:
    for _ in range(8):
        t = threading.Thread(target=lambda: ev.wait())
        ev = threading.Event()
        t.start()
        started.append((t, ev))
except RuntimeError:
    pass
for t, ev in started:
    ev.set()
    t.join()
print("threads", len(started), flush=True)
z = merge_apply_host(Gs, d["r"])
c = chunk_apply_host(Gs, d["r"])
np.savez(sys.argv[2], zm=z[0], groups=z[1], ents=z[2], zc=c[0], counts=c[1])
"""


MEMORY_CHILD = """
import resource
import sys
import numpy as np
from rchol_amd import solver as S

d = np.load(sys.argv[1])
Gs = (d["cp"], d["ri"], d["v"])
r = d["r"]
e = np.array([0, 1, 2], dtype=np.uint64)
call = {"merge": lambda G, b: S.merge_apply_host(G, b)[0],
        "chunk": lambda G, b: S.chunk_apply_host(G, b)[0],
        "analyze": lambda G, b: S.analyze(G)["fwd"]["slot_row"]}[sys.argv[3]]
call((e, e[:2], np.ones(2)), np.ones(2))  # everything is loaded
for room in sys.argv[2].split(","):
    size = next(int(l.split()[1]) << 10 for l in open("/proc/self/status") if l.startswith("VmSize"))
    resource.setrlimit(resource.RLIMIT_AS, (size + (int(room) << 20), resource.RLIM_INFINITY))
    z = None
    try:
        z = call(Gs, r)
    except (RuntimeError, MemoryError) as err:
        said = str(err)
    resource.setrlimit(resource.RLIMIT_AS, (resource.RLIM_INFINITY, resource.RLIM_INFINITY))
    print("refused " + said[:60] if z is None else
          "done %r" % float(np.dot(z, np.arange(1, z.size + 1) / z.size)), flush=True)
"""


@pytest.fixture(scope="module")
def system(tmp_path_factory):
    """A factor that the analysis and the plans spread over threads, on disk."""
    dims = (64, 64, 48)  # 196,608 rows: three ranges of at least 65,536
    A = F.varcoef_3d(*dims, 1.5, 1e-3, 4)
    perm, blocks = F.nd_grid(*dims, 4)
    Gs, _, _ = F.factor(A, perm, blocks, "mis", 2)
    r = np.random.default_rng(1).uniform(-1, 1, A.shape[0])
    path = tmp_path_factory.mktemp("limits") / "factor.npz"
    np.savez(path, cp=Gs[0], ri=Gs[1], v=Gs[2], r=r)
    return str(path), Gs, r


def child(system, out, limit):
    env = dict(os.environ, OMP_NUM_THREADS="8", OPENBLAS_NUM_THREADS="1", PYTHONPATH=ROOT)
    return subprocess.run([sys.executable, "-c", CHILD, system[0], out], env=env, cwd=ROOT,
                          preexec_fn=limit, capture_output=True, text=True, timeout=300)


@pytest.mark.parametrize("threads", [0, 3])
def test_plans_without_all_their_threads(system, tmp_path, threads):
    """Stacks of 4 GiB in an address space that holds a few of them, or none."""
    def big_stacks():
        hard = resource.getrlimit(resource.RLIMIT_STACK)[1]
        resource.setrlimit(resource.RLIMIT_STACK, (4 << 30, hard))
        room = (4 * threads + 3) << 30
        resource.setrlimit(resource.RLIMIT_AS, (room, room))

    out = str(tmp_path / "out.npz")
    p = child(system, out, big_stacks)
    print(p.stdout)
    if "threads" not in p.stdout:
        pytest.skip("the interpreter itself does not fit the limit")
    if "threads 8" in p.stdout:
        pytest.skip("every thread could be started")
    assert p.returncode == 0, (p.returncode, p.stdout, p.stderr)
    d = np.load(out)
    zm, groups, ents, _ = merge_apply_host(system[1], system[2])
    zc, counts, _, _ = chunk_apply_host(system[1], system[2])
    np.testing.assert_array_equal(d["zm"], zm)
    np.testing.assert_array_equal(d["zc"], zc)
    assert d["groups"].tolist() == groups and d["ents"].tolist() == ents
    assert d["counts"].tolist() == counts


@pytest.mark.parametrize("what", ["merge", "chunk", "analyze"])
def test_plans_without_enough_memory(system, what):
    """An allocation that fails is an error of the call, wherever it falls (one
    thread: the C library itself ends a process that has no room for a new
    thread's own data)."""
    env = dict(os.environ, OMP_NUM_THREADS="1", OPENBLAS_NUM_THREADS="1", PYTHONPATH=ROOT)
    p = subprocess.run([sys.executable, "-c", MEMORY_CHILD, system[0], "4,24,60,100,140,4000", what],
                       env=env, cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, (p.returncode, p.stdout, p.stderr)
    said = p.stdout.splitlines()
    assert len(said) == 6 and said[0].startswith("refused") and said[-1].startswith("done")
    assert all(s.startswith("refused") or s == said[-1] for s in said)
