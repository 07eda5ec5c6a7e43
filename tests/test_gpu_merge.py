"""Merged levels in the persistent sweeps (GPU): applications and solves of
one factor with and without them, against the oracle and each other, on
factors whose merged rows take a part of a wave, a whole wave and several
rounds."""
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
    return F.permute(A, po), Gs, np.random.default_rng(5).uniform(-1.0, 1.0, A.shape[0])


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("dims,leaves", [((9, 8, 7), 2), ((20, 18, 16), 4), ((37, 33, 1), 4),
                                         ((33, 33, 33), 8)])
@pytest.mark.parametrize("precision", [rchol_amd.FP64, rchol_amd.FP32])
def test_merged_levels_match_plain_levels_and_oracle(dims, leaves, precision):
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    A, Gs, b = system(dims, leaves)
    print(f"case merged levels {dims} prec={precision}", flush=True)
    zo = O.precond(Gs, b)
    xo, ro, io = O.pcg(A, b, 1e-10, 500, Gs)
    out = {}
    for merge in (1, 0):
        with rchol_amd.Solver(A) as s:
            s.set_option(OPT_MERGE, merge)
            s.upload_G(Gs, precision)
            z = s.precond(b)
            np.testing.assert_array_equal(z, s.precond(b))
            x, rr, it = s.pcg(b, 1e-10, 500)
            x2, rr2, it2 = s.pcg(b, 1e-10, 500)  # graph replay
            np.testing.assert_array_equal(x, x2)
            out[merge] = (s.stats()["fwd_tasks"], s.stats()["bwd_tasks"])
        # 1e-12: the bar of every FP64 application; 1e-5: of the FP32 factor
        assert rel(z, zo) <= (1e-12 if precision == rchol_amd.FP64 else 1e-5)
        assert abs(it - io) <= (1 if precision == rchol_amd.FP64 else 5)
        assert np.linalg.norm(A @ x - b) / np.linalg.norm(b) <= 1e-9
        assert rel(x, xo) <= 1e-8
    assert out[0] != out[1]  # the merged cut is another one


def test_merged_levels_through_permutation_and_static_scratch():
    """The merged sweeps on vectors in the caller's numbering, and from the
    allocation-free entry point."""
    import torch
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    dims = (20, 18, 16)
    A = F.varcoef_3d(*dims, 1.5, 1e-3, 11)
    perm, blocks = F.nd_grid(*dims, 3)
    Gs, po, _ = F.factor(A, perm, blocks, "mis", 1)
    P = po.astype(np.int64)
    b = np.random.default_rng(6).uniform(-1.0, 1.0, A.shape[0])
    zo = np.empty_like(b)
    zo[P] = O.precond(Gs, b[P])
    print("case merged perm / noalloc", flush=True)
    for precision, tol in ((rchol_amd.FP64, 1e-12), (rchol_amd.FP32, 1e-5)):
        with rchol_amd.Solver(F.permute(A, po), Gs, precision) as s:
            s.set_perm(po)
            r = torch.as_tensor(b, device="cuda")
            z = torch.empty_like(r)
            s.precond_device_noalloc(r.data_ptr(), z.data_ptr())
            assert rel(z.cpu().numpy(), zo) <= tol
            assert rel(s.precond(b), zo) <= tol
