"""Factors of thousands of narrow levels (GPU): the upload's own choice between
merged levels and chunks, and every form the options then select, against the
oracle."""
import numpy as np
import pytest
import scipy.sparse as sp

import rchol_amd
from rchol_amd import factor as F
from rchol_amd.solver import OPT_CHUNKED, OPT_MERGE
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def chain(n):
    w = np.random.default_rng(2).uniform(0.5, 2.0, n - 1)
    d = np.full(n, 1e-3)
    d[:-1] += w
    d[1:] += w
    return sp.diags([-w, d, -w], [-1, 0, 1], format="csr")


def box(m):
    return F.grid_laplacian(m, m, m, np.ones(F.grid_edges(m, m, m)[0].size), 1e-2)


@pytest.mark.parametrize("name", ["chain", "box"])
@pytest.mark.parametrize("precision", [rchol_amd.FP64, rchol_amd.FP32])
def test_every_form_of_a_deep_factor_matches_oracle(name, precision):
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    A = chain(30000) if name == "chain" else box(18)
    n = A.shape[0]
    Gs, _, _ = F.factor(A, None, [n], "static", 1)
    b = np.random.default_rng(4).uniform(-1.0, 1.0, n)
    print(f"case deep {name} prec={precision}", flush=True)
    zo = O.precond(Gs, b)
    xo, _, io = O.pcg(A, b, 1e-10, 500, Gs)
    # 1e-12: the bar of every FP64 application; 1e-5: of the FP32 factor
    tol = 1e-12 if precision == rchol_amd.FP64 else 1e-5

    def check(s, chunked):
        assert s.stats()["chunked"] == chunked
        z = s.precond(b)
        assert np.linalg.norm(z - zo) <= tol * np.linalg.norm(zo)
        for _ in range(2):  # the second is a graph replay
            x, rr, it = s.pcg(b, 1e-10, 500)
            assert abs(it - io) <= (1 if precision == rchol_amd.FP64 else 5)
            assert np.linalg.norm(x - xo) <= 1e-8 * np.linalg.norm(xo)

    with rchol_amd.Solver(A) as s:
        s.set_option(OPT_MERGE, 0)
        s.upload_G(Gs, precision)
        assert s.stats()["fwd_levels"] >= 1024
        check(s, 1)  # without merged levels a deep factor runs in chunks
    with rchol_amd.Solver(A) as s:
        s.upload_G(Gs, precision)
        auto = s.stats()["chunked"]
        check(s, auto)
        for mode, chunked in ((1, 1), (0, 0), (-1, auto)):
            s.set_option(OPT_CHUNKED, mode)
            check(s, chunked)
        B = np.stack([b, 2.0 * b, -b, b], axis=1)
        X, _, _ = s.pcg_batch(B, 1e-10, 500)
        assert np.linalg.norm(X[:, 1] - 2.0 * xo) <= 1e-8 * np.linalg.norm(2.0 * xo)
