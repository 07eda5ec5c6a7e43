"""The host analysis and plans of a factor when the process is short of threads
(the work is done by those that start), run in a process with the limit."""
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
