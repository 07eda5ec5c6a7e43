"""The merged-level plan of the persistent sweeps (rchol_amd_merge_apply_host:
the plan run on the CPU, with the check that a row reads only earlier groups)
against the oracle's preconditioner application and an extended-precision
substitution, over the factors it accepts and the ones it must leave alone."""
import glob
import os

import numpy as np
import pytest
import scipy.sparse as sp

from rchol_amd import factor as F
from rchol_amd.solver import analyze, merge_apply_host
from oracle import oracle as O

GOLD = os.path.join(os.path.dirname(__file__), "golden")
FIXTURES = sorted(os.path.basename(p)[:-4] for p in glob.glob(os.path.join(GOLD, "*.npz")))


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def stored(G):
    G = sp.csc_matrix(G)
    return G.indptr.astype(np.uint64), G.indices.astype(np.uint64), G.data


def levels(Gs):
    an = analyze(Gs)
    return [an["fwd"]["nlevels"], an["bwd"]["nlevels"]]


def extended(Gs, r):
    """G^-T G^-1 r in 80-bit arithmetic."""
    cp, ri, v = (np.asarray(a) for a in Gs)
    n = cp.size - 1
    y = r.astype(np.longdouble)
    d = np.zeros(n, dtype=np.longdouble)
    for j in range(n):
        e = slice(int(cp[j]), int(cp[j + 1]))
        on = ri[e] == j
        d[j] = v[e][on][0]
        y[j] /= d[j]
        np.subtract.at(y, ri[e][~on].astype(int), v[e][~on].astype(np.longdouble) * y[j])
    for j in range(n - 1, -1, -1):
        e = slice(int(cp[j]), int(cp[j + 1]))
        off = ri[e] != j
        y[j] = (y[j] - np.sum(v[e][off].astype(np.longdouble) * y[ri[e][off].astype(int)])) / d[j]
    return y


@pytest.mark.parametrize("name", FIXTURES)
def test_merged_levels_match_oracle_on_fixtures(name):
    d = np.load(os.path.join(GOLD, name + ".npz"))
    Gs = (d["g_colptr"], d["g_rowidx"], d["g_val"])
    z, groups, ents, est = merge_apply_host(Gs, d["b"])
    assert rel(z, d["z"]) <= 1e-13
    # 64-bit rounding of either order of sums: a few units in the last place
    # of each of the levels a value passes through
    assert rel(z, extended(Gs, d["b"]).astype(float)) <= 1e-14
    lv = levels(Gs)
    assert all(1 <= g <= l for g, l in zip(groups, lv))
    if lv[0] > 8:
        assert groups[0] < lv[0] and ents[0] > 0


@pytest.mark.parametrize("dims", [(7, 5, 9), (24, 1, 33), (40, 40, 1), (1, 1, 50), (20, 18, 16)])
@pytest.mark.parametrize("order", ["mis", "static"])
def test_merged_levels_match_oracle_on_boxes(dims, order):
    A = F.varcoef_3d(*dims, 1.5, 1e-3, 4)
    perm, blocks = F.nd_grid(*dims, 2)
    Gs, _, _ = F.factor(A, perm, blocks, order, 2)
    r = np.random.default_rng(1).uniform(-1, 1, A.shape[0])
    z, groups, ents, est = merge_apply_host(Gs, r)
    assert rel(z, O.precond(Gs, r)) <= 1e-12
    assert sum(groups) < sum(levels(Gs))


def test_negative_pivots_are_merged_too():
    """The rule is the sign against the row's own pivot, not a positive one."""
    rng = np.random.default_rng(0)
    n = 300
    s = np.where(rng.random(n) < 0.5, -1.0, 1.0)
    M = sp.random(n, n, 0.03, random_state=1, format="csr")
    L = sp.tril(M, -1)
    L.data[:] = -np.abs(L.data)
    # one sweep's rows: scaling row i of G by s_i keeps L_ij against d_i
    G = sp.diags(s) @ (L + sp.identity(n))
    Gs = stored(G)
    r = rng.uniform(-1, 1, n)
    z, groups, ents, est = merge_apply_host(Gs, r)
    assert groups[0] < levels(Gs)[0]
    assert rel(z, O.precond(Gs, r)) <= 1e-12


@pytest.mark.parametrize("case", ["random_sign", "nan", "one_positive", "huge_ratio"])
def test_other_factors_are_left_alone(case):
    """A factor whose elimination could cancel (or is not a number, or would
    overflow) keeps its plain levels."""
    n = 400
    rng = np.random.default_rng(3)
    L = sp.tril(sp.random(n, n, 0.02, random_state=2, format="csr"), -1).tocsr()
    L.data[:] = -np.abs(L.data)
    if case == "random_sign":
        L.data *= np.where(rng.random(L.nnz) < 0.5, -1, 1)
    elif case == "nan":
        L.data[L.nnz // 2] = np.nan
    elif case == "one_positive":
        L.data[L.nnz // 2] = 0.25
    dg = np.ones(n)
    if case == "huge_ratio":
        dg[::2] = 1e-40
        dg[1::2] = 1e40
    Gs = stored(L + sp.diags(dg))
    r = rng.uniform(-1, 1, n)
    z, groups, ents, est = merge_apply_host(Gs, r)
    assert groups == levels(Gs) and ents == [0, 0]
    if case in ("random_sign", "one_positive"):
        assert rel(z, O.precond(Gs, r)) <= 1e-10


@pytest.mark.parametrize("n", [1, 2, 3, 65, 1000])
@pytest.mark.parametrize("shape", ["diagonal", "chain", "star", "dense"])
def test_small_shapes(n, shape):
    if shape == "dense" and n > 100:
        n = 200
    rows, cols = [], []
    if shape == "chain":
        rows, cols = list(range(1, n)), list(range(n - 1))
    elif shape == "star":
        rows, cols = [n - 1] * (n - 1), list(range(n - 1))
    elif shape == "dense":
        rows, cols = map(list, np.tril_indices(n, -1))
    rng = np.random.default_rng(n)
    v = -rng.uniform(0.1, 1.0, len(rows)) / max(1, n if shape == "dense" else 1)
    G = sp.csc_matrix((v, (rows, cols)), shape=(n, n)) + sp.diags(rng.uniform(1, 2, n))
    Gs = stored(G)
    r = rng.uniform(-1, 1, n)
    z, groups, ents, est = merge_apply_host(Gs, r)
    assert rel(z, extended(Gs, r).astype(float)) <= 1e-13


def test_unsorted_columns_and_repeated_entries():
    """Entries of a stored column in any order, an entry split in two."""
    d = np.load(os.path.join(GOLD, "lap3d_8_nd4.npz"))
    cp, ri, v = d["g_colptr"].astype(np.int64), d["g_rowidx"].copy(), d["g_val"].copy()
    rng = np.random.default_rng(5)
    ncp, nri, nv = [0], [], []
    for j in range(cp.size - 1):
        e = np.arange(cp[j], cp[j + 1])
        rng.shuffle(e)
        for k in e:
            if ri[k] != j and rng.random() < 0.1:
                nri += [ri[k], ri[k]]
                nv += [0.25 * v[k], 0.75 * v[k]]
            else:
                nri.append(ri[k])
                nv.append(v[k])
        ncp.append(len(nri))
    Gs = (np.array(ncp, dtype=np.uint64), np.array(nri, dtype=np.uint64), np.array(nv))
    z, groups, ents, est = merge_apply_host(Gs, d["b"])
    assert rel(z, d["z"]) <= 1e-13
