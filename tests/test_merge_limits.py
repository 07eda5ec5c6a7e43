"""The limits of the merged-level plan (CPU): factors of many narrow levels whose
first plan passes one of them are merged all the same, within it."""
import numpy as np
import pytest
import scipy.sparse as sp

from rchol_amd import factor as F
from rchol_amd.solver import analyze, merge_apply_host
from oracle import oracle as O

GROWTH = 64  # merged entries of a sweep, in entries of the factor


def stored(G):
    G = sp.csc_matrix(G)
    G.sort_indices()
    return G.indptr.astype(np.uint64), G.indices.astype(np.uint64), G.data


def chain(n):
    rng = np.random.default_rng(n)
    L = sp.diags([-rng.uniform(0.1, 1.0, n - 1)], [-1], shape=(n, n))
    return stored(L + sp.diags(rng.uniform(1, 2, n)))


def natural(*dims):
    A = F.grid_laplacian(*dims, np.ones(F.grid_edges(*dims)[0].size), 1e-2)
    return F.factor(A, None, [A.shape[0]], "static", 1)[0]


def levels(Gs):
    an = analyze(Gs)
    return [an["fwd"]["nlevels"], an["bwd"]["nlevels"]]


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# below the levels of a deep factor, so that neither chunks nor its shorter
# rows are there; 256 and 8^3 pass at the first attempt
@pytest.mark.parametrize("name,Gs", [(f"chain{n}", chain(n)) for n in (256, 258, 300, 900, 1023)]
                         + [("x".join(map(str, d)), natural(*d))
                            for d in ((8, 8, 8), (10, 10, 10), (32, 32, 1), (2, 1, 400))])
def test_small_factors_of_many_narrow_levels_are_merged(name, Gs):
    n, nnz = len(Gs[0]) - 1, int(Gs[0][-1])
    r = np.random.default_rng(7).uniform(-1, 1, n)
    z, groups, ents, est = merge_apply_host(Gs, r)
    lv = levels(Gs)
    assert lv[0] > 100
    # a tenth of the levels at most: a merged row may hold at least 64 entries
    assert all(g <= l // 10 for g, l in zip(groups, lv)), (groups, lv)
    assert all(0 < e <= GROWTH * nnz for e in ents)
    assert rel(z, O.precond(Gs, r)) <= 1e-12
