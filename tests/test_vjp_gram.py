"""The closed-form VJP as one Gram product, at the sizes where its chunks,
row groups and zero weights can go wrong, against the CPU oracle; torch's
gradient convention against the holomorphic one, bit for bit; the recompute
sweep that forms slab m + 1 from the VJP's loads against the stored lattice.

Tolerance: a sum of N products differs between two summation orders by at
most about N eps times the sum of absolute values, in practice sqrt(N) eps;
1e-12 of the largest entry leaves a factor 10 at N = 4e6.
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from mrmustard_amd import workloads as W
from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

SHAPES = [
    (1,), (2,), (257,), (4097,), (1, 1), (2, 1), (1, 5), (4099, 3), (16, 16), (33, 31), (1, 7, 1), (9, 1, 30), (8, 8, 9),
    (2, 2, 2, 2), (7, 6, 5, 13), (3, 4, 1, 5, 6), (2, 3, 4, 5, 6, 3), (3, 2, 4, 1, 3, 2, 5), (3, 3, 3, 3, 3, 3, 3, 3), (2, 1, 3, 4, 2, 5, 2, 6),
]


@pytest.mark.parametrize("shape", SHAPES)
def test_vjp_against_the_oracle(shape):
    import torch

    from mrmustard_amd.lattice import strategies as st

    rng = np.random.default_rng(sum(shape))
    G, g = W.complex_normal(shape, 1.0, rng), W.complex_normal(shape, 1.0, rng)
    c = np.complex128(0.7 - 0.2j)
    ref = oracle.vanilla_vjp(G, c, g)
    print(f"vjp shape={shape}", flush=True)
    got = st.vanilla_vjp_hip(G, c, g)
    scale = max(1.0, np.sqrt(np.prod(shape)) * max(shape))
    for x, r in zip(got, ref):
        assert np.max(np.abs(x.cpu().numpy() - r)) <= 1e-12 * max(scale, np.max(np.abs(r)))
    conj = st.vanilla_vjp_grad_hip(G, c, torch.as_tensor(g, device="cuda").conj())
    for x, y in zip(conj, got):
        assert torch.equal(x, y.conj())


@pytest.mark.parametrize("shape,B", [((5, 4, 3), 7), ((12, 11, 3, 5), 9), ((20, 21), 1500), ((3, 2, 2, 3, 2, 2, 3, 2), 5)])
def test_batched_vjp_equals_single(shape, B):
    import torch

    from mrmustard_amd.lattice import strategies as st

    rng = np.random.default_rng(B)
    G, g = W.complex_normal((B, *shape), 1.0, rng), W.complex_normal((B, *shape), 1.0, rng)
    c = W.complex_normal((B,), 1.0, rng) + 2.0
    got = st.vanilla_vjp_grad_hip(G, c, torch.as_tensor(g, device="cuda"), batched=True)
    for k in (0, B // 2, B - 1):
        ref = oracle.vanilla_vjp(G[k], c[k], g[k].conj())
        for x, r in zip(got, ref):
            assert np.max(np.abs(x[k].cpu().numpy().conj() - r)) <= 1e-12 * max(1.0, np.sqrt(np.prod(shape)) * max(shape))


@pytest.mark.parametrize("shape", [(30, 30, 30, 160), (7, 25, 26, 31, 31), (5, 12, 12, 12, 12, 41), (3, 9, 10, 11, 9, 10, 15), (3, 7, 8, 7, 8, 7, 8, 8)])
def test_recompute_window_equals_stored(shape):
    """Lattices above 64 MB: the three-slab window."""
    import torch

    from mrmustard_amd.lattice import strategies as st

    rng = np.random.default_rng(len(shape))
    A, b, c = W.gaussian_ket(len(shape), rng, r_max=0.8)
    gen = torch.Generator(device="cuda").manual_seed(3)
    g = torch.randn(shape, dtype=torch.complex128, device="cuda", generator=gen)
    G = st.vanilla_hip(shape, A, b, c)
    print(f"recompute shape={shape}", flush=True)
    ref = st.vanilla_vjp_hip(G, c, g)
    got = st.vanilla_vjp_recompute_hip(shape, A, b, c, g)
    for x, r in zip(got, ref):
        assert float((x - r).abs().max()) <= 1e-12 * float(r.abs().max())
    conj = st.vanilla_vjp_recompute_hip(shape, *st.conj_triple(A, b, c), g.conj())
    for x, y in zip(conj, got):
        assert torch.equal(x, y.conj())
