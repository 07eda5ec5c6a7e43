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


def with_chain(rows, cols, vals, n):
    """Given rows 0 .. n - 1, and after them a chain of 600 rows of its own."""
    m = 600
    rng = np.random.default_rng(3)
    rows = np.concatenate([rows, np.arange(n + 1, n + m)])
    cols = np.concatenate([cols, np.arange(n, n + m - 1)])
    vals = np.concatenate([vals, -rng.uniform(0.1, 1.0, m - 1)])
    L = sp.csc_matrix((vals, (rows, cols)), shape=(n + m, n + m))
    return stored(L + sp.diags(np.concatenate([np.ones(n), rng.uniform(1, 2, m)])))


def large_ratios():
    """A chain of 20 rows whose merged coefficients pass 1e30."""
    return with_chain(np.arange(1, 20), np.arange(19), np.full(19, -1e4), 20)


def long_row():
    """A row that reads 9000 others, read by one of 51 rows of its level (the
    last: not one of those whose merged length is looked at)."""
    k = 9000
    side = np.arange(50)
    rows = np.concatenate([k + 50 + side, k + 100 + side, np.full(k, k + 150), [k + 151]])
    cols = np.concatenate([k + side, k + 50 + side, np.arange(k), [k + 150]])
    return with_chain(rows, cols, np.full(rows.size, -1e-3), k + 152)


@pytest.mark.parametrize("second", [large_ratios, long_row])
def test_a_row_that_cannot_be_merged_leaves_its_group_alone(second):
    """Not the whole sweep: the other chain is merged."""
    Gs = second()
    n = len(Gs[0]) - 1
    r = np.random.default_rng(8).uniform(0.1, 1, n)
    z, groups, ents, est = merge_apply_host(Gs, r)
    lv = levels(Gs)
    assert groups[0] < lv[0] // 2 and ents[0] > 0, (groups, lv, ents)
    # rounding of sums of one sign in either order, relative to each value
    zo = O.precond(Gs, r)
    assert np.max(np.abs(z - zo) / np.abs(zo)) <= 1e-11


def chain_with_wide_levels(n, wide, w):
    """A chain of n rows in which every level of `wide` also holds w rows that
    read the chain's row before."""
    rows, cols = [np.arange(1, n)], [np.arange(n - 1)]
    k = n
    for l in wide:
        rows.append(np.arange(k, k + w))
        cols.append(np.full(w, l - 1))
        k += w
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    rng = np.random.default_rng(5)
    L = sp.csc_matrix((-rng.uniform(0.1, 1.0, rows.size), (rows, cols)), shape=(k, k))
    return stored(L + sp.diags(rng.uniform(1, 2, k)))


def test_a_wide_level_inside_a_group_is_looked_at():
    """A level of w rows is merged only while the entries this adds cost less
    than 0.2 us at 5 ps each, wherever in a group's depth it lies: the wide
    levels at 100 and 150 hold 3000 rows, so none of their rows may have more
    than 14 entries (0.2 / 5e-6 / 3000, and the one it reads)."""
    n, w = 400, 3000
    Gs = chain_with_wide_levels(n, [100, 150], w)
    r = np.random.default_rng(8).uniform(-1, 1, n + 2 * w)
    z, groups, ents, est = merge_apply_host(Gs, r)
    assert rel(z, O.precond(Gs, r)) <= 1e-12
    assert groups[0] < levels(Gs)[0] // 10
    # the chain's own rows: at most one triangle of n / 2 each way
    assert ents[0] <= n * n // 2 + 2 * w * 14, (groups, ents)
