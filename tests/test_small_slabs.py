"""Small slabs, one point per thread of a workgroup of as few waves as hold them.

Slab sizes around one wave, two waves and the line to the 512-thread teams, one
triple and batches: the forward has the oracle's bits, the fused VJP agrees with
the oracle's compensated sum to 1e-12 (its sums run in another order).
"""

import numpy as np
import pytest

from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

SHAPES = [(5, 63), (5, 64), (5, 65), (300, 2), (3, 128), (3, 129), (4, 384), (4, 385), (3, 511), (3, 512), (7, 8, 8), (6, 5, 13), (3, 1, 64),
          (2, 16, 24), (2, 11, 35), (5, 4, 4, 4), (4, 5, 5, 5), (3, 3, 3, 3, 2)]


@pytest.mark.parametrize("B", [1, 9])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_forward_and_fused(shape, B):
    import oracle
    from mrmustard_amd.lattice import strategies as st

    oracle.build()
    rng = np.random.default_rng(sum(shape) + B)
    D = len(shape)
    A = 0.4 * (rng.normal(size=(B, D, D)) + 1j * rng.normal(size=(B, D, D))) / D
    A = (A + A.transpose(0, 2, 1)) / 2
    b = 0.5 * (rng.normal(size=(B, D)) + 1j * rng.normal(size=(B, D)))
    c = rng.normal(size=B) + 0.4j
    ref = oracle.vanilla_batch(shape, A, b, c)
    assert np.array_equal(st.vanilla_batch_hip(shape, A, b, c).cpu().numpy(), ref)
    assert np.array_equal(st.vanilla_hip(shape, A[0], b[0], c[0]).cpu().numpy(), ref[0])
    g = rng.normal(size=(B, *shape)) + 1j * rng.normal(size=(B, *shape))
    G, dA, db, dc = (x.cpu().numpy() for x in st.vanilla_batch_fused_hip(shape, A, b, c, g))
    assert np.array_equal(G, ref)
    for k in range(B):
        for x, r in zip((dA[k], db[k], dc[k]), oracle.vanilla_vjp(ref[k], c[k], g[k])):
            assert np.abs(x - r).max() <= 1e-12 * np.abs(r).max()
