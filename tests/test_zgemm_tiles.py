"""The 64 x 128 tiles of the matrix-core product at ragged edges, for sizes that
the rule gives them, against numpy.  Tolerance as for the strips: 8 K eps of the
product of the magnitudes covers the bound of a complex sum of K products."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from mrmustard_amd import _lib
from mrmustard_amd import workloads as W
from tests.conftest import gpu_available

SIZES = [(1010, 4090, 10, 1), (2047, 2047, 9, 1), (961, 4033, 1, 1), (1010, 2045, 11, 2)]


@pytest.mark.parametrize("M,N,K,nb", SIZES)
def test_rule(M, N, K, nb):
    out = (ctypes.c_int64 * 4)()
    assert _lib.load().mm_zgemm_plan(M, N, nb, 0, 256, ctypes.addressof(out)) == 0
    assert out[0] == 0


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")
@pytest.mark.parametrize("M,N,K,nb", SIZES)
def test_product(M, N, K, nb):
    from mrmustard_amd.contraction import zgemm_batched_hip

    rng = np.random.default_rng(M + 7 * N + K)
    A, B = W.complex_normal((nb, M, K), 1.0, rng), W.complex_normal((nb, K, N), 1.0, rng)
    print(f"zgemm {M} x {N} x {K}, {nb}", flush=True)
    C = zgemm_batched_hip(A, B).cpu().numpy()
    assert np.all(np.abs(C - np.matmul(A, B)) <= 8 * K * np.finfo(float).eps * np.matmul(np.abs(A), np.abs(B)))
