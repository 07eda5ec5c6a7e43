"""Stacked solves (GPU) whose systems span from one workgroup to more than a
workgroup's threads of them, in layouts that the 8 XCDs do not divide: every
system's reductions against a reference of its own."""
import numpy as np
import pytest
import scipy.sparse as sp

import rchol_amd

pytestmark = pytest.mark.gpu


def jacobi_cg(A, d, b, steps):
    x, r = np.zeros_like(b), b.copy()
    z = r / d
    p, rz = z.copy(), r @ z
    for _ in range(steps):
        q = A @ p
        alpha = rz / (p @ q)
        x += alpha * p
        r -= alpha * q
        z = r / d
        rz, old = r @ z, rz
        p = z + (rz / old) * p
    return x


@pytest.mark.parametrize("sizes", [[300], [5, 400000, 3, 1500], [70, 90, 110, 64, 65, 63, 2],
                                   [1000] * 256])
def test_every_system_keeps_its_own_sums(sizes):
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    print(f"case seg blocks {sizes[:7]} of {len(sizes)}", flush=True)
    blocks, diag = [], []
    for k, n in enumerate(sizes):
        d = 2.5 + np.cos(np.arange(n) + k)
        off = np.full(n - 1, -0.5)
        blocks.append(sp.diags([off, d, off], [-1, 0, 1], format="csr"))
        diag.append(d)
    A = sp.block_diag(blocks, format="csr")
    G = sp.diags([np.sqrt(np.concatenate(diag))], [0], format="csc")
    off = np.concatenate([[0], np.cumsum(sizes)])
    b = np.sin(1.0 + np.arange(off[-1]))
    with rchol_amd.Solver(A, G) as s:
        s.set_segments(off)
        x, rr, it = s.pcg_segments(b, 1e-300, 2)
        x2, _, _ = s.pcg_segments(b, 1e-300, 2)  # graph replay
    np.testing.assert_array_equal(x, x2)
    assert np.all(it == 2)
    for k in range(len(sizes)):
        u = slice(off[k], off[k + 1])
        ref = jacobi_cg(blocks[k], diag[k], b[u], 2)
        # 2 iterations of a system of condition < 4 in FP64: a few hundred roundings
        assert np.linalg.norm(x[u] - ref) <= 1e-13 * np.linalg.norm(ref)
        res = np.linalg.norm(blocks[k] @ ref - b[u]) / np.linalg.norm(b[u])
        assert abs(rr[k] - res) <= 1e-9 * res + 1e-13
