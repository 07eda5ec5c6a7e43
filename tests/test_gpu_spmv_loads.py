"""The SpMV's two ways to load A (GPU): systems on both sides of the footprint
at which the stream form stops leaving A in the caches, and next to it, with a
diagonal factor so that the iterates have a short reference."""
import numpy as np
import pytest
import scipy.sparse as sp

import rchol_amd

pytestmark = pytest.mark.gpu

# 12 bytes per nonzero against 128 MB: the first row count that streams
LIMIT = (128 << 20) // 12


def system(n):
    """Tridiagonal, diagonally dominant, exactly 3 n - 2 nonzeros."""
    d = 2.5 + np.cos(np.arange(n))
    A = sp.diags([np.full(n - 1, -0.5), d, np.full(n - 1, -0.5)], [-1, 0, 1], format="csr")
    G = sp.diags([np.sqrt(d)], [0], format="csc")
    return A, G, d, np.sin(1.0 + np.arange(n))


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


@pytest.mark.parametrize("n", [70001, (LIMIT + 2) // 3 - 1, (LIMIT + 2) // 3 + 1])
def test_both_load_forms_give_the_iterates(n):
    if rchol_amd.device_count() < 1:
        pytest.skip("no HIP device")
    A, G, d, b = system(n)
    print(f"case spmv loads n={n} nnz={A.nnz}", flush=True)
    assert (A.nnz * 12 > 128 << 20) == (n > (LIMIT + 2) // 3)
    with rchol_amd.Solver(A, G) as s:
        x, rr, it = s.pcg(b, 1e-300, 4)
        y = s.spmv(x)
    assert it == 4
    ref = jacobi_cg(A, d, b, 4)
    # 4 iterations of a system of condition < 4 in FP64: a few hundred roundings
    assert np.linalg.norm(x - ref) <= 1e-13 * np.linalg.norm(ref)
    # 3 products and 2 sums per row, |A||x| <= 3 |A x| row norms at most
    assert np.max(np.abs(y - A @ x)) <= 8 * 2.0 ** -53 * 4.5 * np.max(np.abs(x))
