"""Sectors with singular values of exactly 0 among others, every value kept."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import __graft_entry__ as GE  # noqa: E402

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


@pytest.mark.parametrize("m,n", [(1, 1), (5, 1), (1, 200), (8, 8), (64, 40), (40, 300), (1600, 7)])
@pytest.mark.parametrize("l2r", [True, False])
def test_zero_sectors_keep_orthonormal_vectors(m, n, l2r):
    kv = GE.load_package()
    print(f"case svd zero {m}x{n} l2r {l2r}", flush=True)
    rng = np.random.default_rng([m, n])

    def cplx(*s):
        return rng.standard_normal(s) + 1j * rng.standard_normal(s)

    blocks = {(0, 0): np.zeros((m, n), complex), (1, 1): cplx(m, n), (2, 2): cplx(m, n), (3, 3): cplx(m, n)}
    blocks[2, 2][:, n // 2] = 0  # the short side's row or column: a zero pivot
    blocks[3, 3][m // 2] = 0
    left, right = kv.svd_impl(kv.Tensor.from_blocks((1, -1), blocks), 1, -1.0, 10 ** 6, l2r)
    L, R = left.to_blocks()[1], right.to_blocks()[1]
    k = min(m, n)
    for q, M in blocks.items():
        u, v = L[q], R[q]
        iso = u.conj().T @ u if l2r else v @ v.conj().T
        assert iso.shape == (k, k)
        # as test_small_sectors_svd: k rotations or reflections over a side of max(m, n)
        tol = 40 * EPS * np.sqrt(k * max(m, n))
        assert np.abs(iso - np.eye(k)).max() < tol
        assert np.linalg.norm(u @ v - M) <= tol * np.linalg.norm(M)
