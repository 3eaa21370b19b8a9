"""The matrix-core product at the edges of its strips (rows of a tile row,
16-column waves, 64-column workgroups, K chunks of 8 and 16) and of the rule
that picks them, against numpy.

Tolerance: a complex product of K terms has an error of at most about 2 K eps
times the product of the magnitudes; with CN(0, 1) entries, sqrt(K) of those
in practice.  8 K eps covers the bound.
"""

from __future__ import annotations

import numpy as np
import pytest

from mrmustard_amd import workloads as W
from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

SIZES = [
    (1, 1, 1, 1), (16, 64, 16, 1), (17, 65, 17, 3), (15, 63, 4, 2), (33, 31, 5, 1), (48, 129, 8, 1), (64, 200, 9, 2), (65, 16, 25, 1),
    (2, 70000, 3, 1), (30, 66000, 16, 1), (47, 65600, 17, 1), (70, 65537, 12, 1), (95, 65536, 7, 1), (100, 65600, 20, 1), (128, 65700, 33, 1),
    (129, 70000, 8, 1), (600, 7, 40, 1), (1024, 4096, 10, 1), (1030, 4100, 24, 1), (10, 100, 10, 700), (100, 100, 30, 90),
    (20, 33, 9, 70001),
]


@pytest.mark.parametrize("M,N,K,nb", SIZES)
def test_product(M, N, K, nb):
    from mrmustard_amd.contraction import zgemm_batched_hip

    rng = np.random.default_rng(M + 7 * N + K)
    na = 1 if nb % 2 == 0 or nb > 600 else nb  # a shared A, or one each
    A, B = W.complex_normal((na, M, K), 1.0, rng), W.complex_normal((nb, K, N), 1.0, rng)
    print(f"zgemm {M} x {N} x {K}, {nb}", flush=True)
    C = zgemm_batched_hip(A, B).cpu().numpy()
    sel = np.unique(np.r_[0 : min(nb, 50), nb // 2, max(0, nb - 50) : nb])  # the ends and the middle of a long batch
    C, B, A = C[sel], B[sel], A if na == 1 else A[sel]
    assert np.all(np.abs(C - np.matmul(A, B)) <= 8 * K * np.finfo(float).eps * np.matmul(np.abs(A), np.abs(B)))
