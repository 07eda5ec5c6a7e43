"""Merged levels on factors of benchmark size (GPU): applications of one and of
eight columns and a solve, with and without them, against the oracle."""
import numpy as np
import pytest

import rchol_amd
from rchol_amd import factor as F
from rchol_amd.solver import OPT_MERGE
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,leaves", [((64, 64, 64), 16), ((97, 61, 83), 16)])
@pytest.mark.parametrize("precision", [rchol_amd.FP64, rchol_amd.FP32])
def test_merged_levels_of_large_factors(dims, leaves, precision):
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    A = F.varcoef_3d(*dims, 1.5, 1e-3, 11)
    perm, blocks = F.nd_grid(*dims, int(np.log2(leaves)) + 1)
    Gs, po, _ = F.factor(A, perm, blocks, "mis", 1)
    A = F.permute(A, po)
    n = A.shape[0]
    R = np.random.default_rng(5).uniform(-1.0, 1.0, (n, 8))
    print(f"case large merged {dims} prec={precision}", flush=True)
    # the bars of an application of either precision
    tol = 1e-12 if precision == rchol_amd.FP64 else 1e-5
    zo = [O.precond(Gs, R[:, c]) for c in (0, 7)]
    tasks = []
    for merge in (1, 0):
        with rchol_amd.Solver(A) as s:
            s.set_option(OPT_MERGE, merge)
            s.upload_G(Gs, precision)
            z, Z = s.precond(R[:, 0]), s.precond_batch(R)
            for got, want in ((z, zo[0]), (Z[:, 0], zo[0]), (Z[:, 7], zo[1])):
                assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
            x, rr, it = s.pcg(R[:, 0], 1e-10, 500)
            assert np.linalg.norm(A @ x - R[:, 0]) <= 1e-9 * np.linalg.norm(R[:, 0])
            tasks.append((s.stats()["fwd_tasks"], it))
    assert tasks[0][0] != tasks[1][0] and abs(tasks[0][1] - tasks[1][1]) <= 1
