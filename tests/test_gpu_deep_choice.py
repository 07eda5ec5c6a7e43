"""Deep factors (GPU): which of merged levels and chunks the upload takes, on
factors of either kind and beyond the levels that are merged at all, and that
the merged cut is the one that runs."""
import numpy as np
import pytest
import scipy.sparse as sp

import rchol_amd
from rchol_amd import factor as F
from rchol_amd.solver import OPT_CHUNKED, OPT_MERGE, analyze, merge_apply_host
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def chain(n):
    w = np.random.default_rng(2).uniform(0.5, 2.0, n - 1)
    d = np.full(n, 1e-3)
    d[:-1] += w
    d[1:] += w
    A = sp.diags([-w, d, -w], [-1, 0, 1], format="csr")
    return F.factor(A, None, [n], "static", 1)[0]


def natural(*dims):
    A = F.grid_laplacian(*dims, np.ones(F.grid_edges(*dims)[0].size), 1e-2)
    return F.factor(A, None, [A.shape[0]], "static", 1)[0]


def stacked(Gs, k):
    """k copies of a factor as one block-diagonal factor."""
    cp, ri, v = (np.asarray(a) for a in Gs)
    n, m = cp.size - 1, int(cp[-1])
    cp = np.concatenate([cp[:-1].astype(np.int64) + i * m for i in range(k)] + [[k * m]])
    ri = np.concatenate([ri.astype(np.int64) + i * n for i in range(k)])
    return cp.astype(np.uint64), ri.astype(np.uint64), np.tile(v, k)


# chunked: what runs faster, measured, by 1.4 times at least
CASES = [("natural14", lambda: natural(14, 14, 14), True, 0),
         ("chain3000", lambda: chain(3000), True, 0),
         ("stack48x64x64", lambda: stacked(natural(64, 64, 1), 48), True, 1),
         ("chain30000", lambda: chain(30000), False, 1)]


@pytest.mark.parametrize("name,make,merges,chunked", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("precision", [rchol_amd.FP64, rchol_amd.FP32])
def test_the_form_that_a_deep_factor_runs_in(name, make, merges, chunked, precision):
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    Gs = make()
    n = len(Gs[0]) - 1
    an = analyze(Gs)
    lv = [an["fwd"]["nlevels"], an["bwd"]["nlevels"]]
    r = np.random.default_rng(4).uniform(-1.0, 1.0, n)
    _, groups, _, _ = merge_apply_host(Gs, r)
    assert lv[0] >= 1024
    assert all(g < l // 8 if merges else g == l for g, l in zip(groups, lv)), (groups, lv)
    print(f"case {name} prec={precision}", flush=True)
    zo = O.precond(Gs, r)
    tol = 1e-12 if precision == rchol_amd.FP64 else 1e-5  # the bars of an application
    tasks = {}
    for merge in (1, 0):
        with rchol_amd.Solver() as s:
            s.set_option(OPT_MERGE, merge)
            s.upload_G(Gs, precision)
            st = s.stats()
            assert st["chunked"] == (chunked if merge else 1)
            assert np.linalg.norm(s.precond(r) - zo) <= tol * np.linalg.norm(zo)
            s.set_option(OPT_CHUNKED, 0)  # the levels, merged or not
            assert np.linalg.norm(s.precond(r) - zo) <= tol * np.linalg.norm(zo)
            tasks[merge] = (st["fwd_tasks"], st["bwd_tasks"])
    assert (tasks[0] != tasks[1]) == merges
