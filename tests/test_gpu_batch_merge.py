"""Multi-column solves and applications (GPU) over the column widths on both
sides of the one up to which merged levels are taken, with idle columns, on
systems of one workgroup and of many, against the oracle column by column."""
import numpy as np
import pytest

import rchol_amd
from rchol_amd import factor as F
from rchol_amd.solver import OPT_MERGE
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def system(dims, leaves):
    A = F.varcoef_3d(*dims, 1.5, 1e-3, 11)
    perm, blocks = F.nd_grid(*dims, int(np.log2(leaves)) + 1)
    Gs, po, _ = F.factor(A, perm, blocks, "mis", 1)
    return F.permute(A, po), Gs


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("dims,leaves", [((5, 4, 3), 2), ((33, 31, 1), 4), ((20, 18, 16), 4)])
@pytest.mark.parametrize("k", [1, 3, 4, 8, 9, 32])
@pytest.mark.parametrize("precision", [rchol_amd.FP64, rchol_amd.FP32])
def test_columns_match_oracle(dims, leaves, k, precision):
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    A, Gs = system(dims, leaves)
    n = A.shape[0]
    print(f"case batch merge {dims} k={k} prec={precision}", flush=True)
    B = np.random.default_rng(k).uniform(-1.0, 1.0, (n, k))
    cols = sorted({0, k // 2, k - 1})
    zo = {c: O.precond(Gs, np.ascontiguousarray(B[:, c])) for c in cols}
    xo = {c: O.pcg(A, np.ascontiguousarray(B[:, c]), 1e-10, 500, Gs)[0] for c in cols}
    # 1e-12: the bar of every FP64 application; 1e-5: of the FP32 factor
    tol = 1e-12 if precision == rchol_amd.FP64 else 1e-5
    for merge in (1, 0):
        with rchol_amd.Solver(A) as s:
            s.set_option(OPT_MERGE, merge)
            s.upload_G(Gs, precision)
            Z = s.precond_batch(B)
            np.testing.assert_array_equal(Z, s.precond_batch(B))
            X, rr, it = s.pcg_batch(B, 1e-10, 500)
            X2, rr2, it2 = s.pcg_batch(B, 1e-10, 500)  # graph replay
            np.testing.assert_array_equal(X, X2)
            np.testing.assert_array_equal(rr, rr2)
        for c in cols:
            assert rel(Z[:, c], zo[c]) <= tol
            assert rel(X[:, c], xo[c]) <= 1e-8
        R = np.linalg.norm(A @ X - B, axis=0) / np.linalg.norm(B, axis=0)
        assert np.all(R <= 1e-9)
        np.testing.assert_allclose(rr, R, rtol=1e-4, atol=1e-14)
