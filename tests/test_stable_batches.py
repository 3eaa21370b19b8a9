"""Batches of the all-pivot average with more tiles than CUs, triples along one
grid axis and tile rows along the other: the oracle's bits.

Batch sizes around a multiple of the XCDs and below it, ragged tiles, and one
triple that overflows among triples that do not.
"""

import numpy as np
import pytest

from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


@pytest.mark.parametrize("shape,B", [((7, 7, 7, 7), 64), ((7, 8, 7, 6), 67), ((20, 19, 21), 145), ((16, 15, 16, 17), 9), ((10, 9, 10, 9), 129),
                                     ((6, 7, 6, 5, 6), 40), ((5, 4, 5, 4, 5, 4), 23), ((90, 70), 300), ((7, 7, 7, 7), 7)],
                         ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else s)
@pytest.mark.parametrize("overflow", [False, True])
def test_bits(shape, B, overflow):
    import oracle
    from mrmustard_amd.lattice import strategies as st

    oracle.build()
    rng = np.random.default_rng(B)
    D = len(shape)
    A = 0.4 * (rng.normal(size=(B, D, D)) + 1j * rng.normal(size=(B, D, D))) / D
    b = rng.normal(size=(B, D)) + 1j * rng.normal(size=(B, D))
    c = rng.normal(size=B) + 1j * rng.normal(size=B)
    if overflow:
        b[B // 2] *= 1e100
    print(f"stable batch {shape} x {B}", flush=True)
    G = st.vanilla_batch_hip(shape, A, b, c, stable=True).cpu().numpy()
    at = sorted({0, 1, B // 2 - 1, B // 2, B - 2, B - 1})
    ref = oracle.vanilla_batch(shape, A[at], b[at], c[at], stable=True)
    assert np.array_equal(G[at], ref, equal_nan=True)
    finite = np.isfinite(G.reshape(B, -1)).all(1)
    assert finite.sum() == B - overflow and finite[B // 2] != overflow
