"""Merged levels on values out of the ordinary (GPU): coefficients whose
products pass the largest FP32 number where the substitution's do not, and
right-hand sides that are not finite, with and without merged levels."""
import numpy as np
import pytest
import scipy.sparse as sp

import rchol_amd
from rchol_amd import factor as F
from rchol_amd.solver import OPT_MERGE

pytestmark = pytest.mark.gpu


def applied(A, Gs, r, precision, merge):
    """One application, alone and as the first of four columns."""
    with rchol_amd.Solver(A) as s:
        s.set_option(OPT_MERGE, merge)
        s.upload_G(Gs, precision)
        return s.precond(r), s.precond_batch(np.stack([r, r, 2.0 * r, -r], axis=1))[:, 0]


@pytest.mark.parametrize("precision", [rchol_amd.FP64, rchol_amd.FP32])
def test_large_coefficients_stay_finite(precision):
    """64 times x_k = 2^33, x_j = (b_j + x_k) / 2^-40 = 0, x_i = 1 + 2^56 x_j = 1.
    Merged, x_i would add and take away 2^96 x_k = 2^129.  All values are
    powers of two, so both forms are exact."""
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    m = 64
    k, j, i = np.arange(m), m + np.arange(m), 2 * m + np.arange(m)
    L = sp.csc_matrix((np.concatenate([np.full(m, -1.0), np.full(m, -2.0 ** 56)]),
                       (np.concatenate([j, i]), np.concatenate([k, j]))), shape=(3 * m, 3 * m))
    d = np.concatenate([np.ones(m), np.full(m, 2.0 ** -40), np.ones(m)])
    G = sp.csc_matrix(L + sp.diags(d))
    G.sort_indices()
    Gs = (G.indptr.astype(np.uint64), G.indices.astype(np.uint64), G.data)
    r = np.concatenate([np.full(m, 2.0 ** 33), np.full(m, -2.0 ** 33), np.ones(m)])
    # y = (2^33, 0, 1); z_i = 1, z_j = 2^56 / 2^-40, z_k = 2^33 + z_j
    z = np.concatenate([np.full(m, 2.0 ** 33 + 2.0 ** 96), np.full(m, 2.0 ** 96), np.ones(m)])
    print(f"case large coefficients prec={precision}", flush=True)
    for merge in (0, 1):
        for got in applied(sp.identity(3 * m, format="csr"), Gs, r, precision, merge):
            assert np.all(np.isfinite(got)), merge
            np.testing.assert_allclose(got, z, rtol=1e-6 if precision == rchol_amd.FP32 else 1e-15)


@pytest.mark.parametrize("precision", [rchol_amd.FP64, rchol_amd.FP32])
@pytest.mark.parametrize("bad", [[np.inf], [-np.inf], [np.nan], [np.inf, np.nan]])
def test_right_hand_sides_that_are_not_finite(precision, bad):
    """Merged levels spread an infinity or a NaN to the rows that the plain
    levels spread it to."""
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    systems = []
    for seed in (1, 2, 3):
        A = F.varcoef_3d(20, 18, 16, 1.5, 1e-3, seed)
        perm, blocks = F.nd_grid(20, 18, 16, 3)
        Gs, po, _ = F.factor(A, perm, blocks, "mis", seed)
        systems.append((F.permute(A, po), Gs))
    A, Gs, off = rchol_amd.stack_systems(systems)
    r = np.random.default_rng(6).uniform(-1.0, 1.0, A.shape[0])
    r[[int(off[1]) + 4000, 1234][:len(bad)]] = bad
    print(f"case right-hand side {bad} prec={precision}", flush=True)
    with np.errstate(all="ignore"):
        plain = applied(A, Gs, r, precision, 0)
        merged = applied(A, Gs, r, precision, 1)
    tol = 1e-12 if precision == rchol_amd.FP64 else 1e-5  # the bars of an application
    for p, m in zip(plain, merged):
        assert not np.all(np.isfinite(p))
        np.testing.assert_array_equal(np.isnan(p), np.isnan(m))
        np.testing.assert_array_equal(np.isposinf(p), np.isposinf(m))
        np.testing.assert_array_equal(np.isneginf(p), np.isneginf(m))
        f = np.isfinite(p)
        assert f.sum() >= off[1]  # a system of its own stays finite
        assert np.linalg.norm(p[f] - m[f]) <= tol * np.linalg.norm(p[f])
