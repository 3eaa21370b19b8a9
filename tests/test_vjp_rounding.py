"""Rounding error of the closed-form VJP's sums over large lattices, whose
threads add hundreds of points each, against double-double sums.

Unit: eps times the root of the sum of |term|^2.  An addition onto a partial
sum of k terms rounds by about 0.29 eps of it at most (uniform in half an ulp),
twice per term (the complex product's two multiply-adds): chains of n terms
leave 0.084 n in the square of the error.  Chains of 16 points (1.34), 16
wave sums of 64 chains after one another (0.67), the additions of lanes, waves
and partial rows (0.6) and the products (0.3) are 1.7 units; 2.5 leaves room for
the spread of the mean over 24 or more sums.  Chains of 290 points, all of a
thread's in the second shape, leave 4.9.
"""

from __future__ import annotations

import numpy as np
import pytest

from mrmustard_amd import workloads as W
from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def _dd_sum(x):
    """Pairwise sum with the rounding errors of every addition carried along."""
    import torch

    e = torch.zeros_like(x)
    while x.numel() > 1:
        if x.numel() % 2:
            x, e = torch.cat([x, x.new_zeros(1)]), torch.cat([e, e.new_zeros(1)])
        n = x.numel() // 2
        a, b = x[:n], x[n:]
        s = a + b
        bb = s - a
        e = e[:n] + e[n:] + ((a - (s - bb)) + (b - bb))
        x = s
    return (x + e)[0]


def _terms(G, h, axes):
    """sqrt(weights) G[k - 1_axes] h[k] of dc (no axis), db (one) or an off-diagonal dA (two)."""
    import torch

    for a in axes:
        n = G.shape[a]
        w = torch.sqrt(torch.arange(1, n, dtype=torch.float64, device="cuda")).reshape([n - 1 if j == a else 1 for j in range(G.dim())])
        G, h = G.narrow(a, 0, n - 1) * w, h.narrow(a, 1, n - 1)
    return (G * h).reshape(-1)


@pytest.mark.parametrize("kind,shape", [("dm", (8,) * 8), ("ket", (11,) * 7)])
def test_rounding_of_long_sums(kind, shape):
    import torch

    from mrmustard_amd.lattice import strategies as st

    D = len(shape)
    rng = np.random.default_rng(3)
    if kind == "ket":
        A, b, c = W.gaussian_ket(D, rng, r_max=1.0)
    else:
        A, b, c = W.apply_loss(*W.ket_to_dm(*W.gaussian_ket(D // 2, rng, r_max=0.8)), rng.uniform(0.7, 1.0, D // 2))
    G = st.vanilla_hip(shape, A, b, c)
    cc = complex(c)
    sq = []
    for seed in range(3):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        h = torch.randn(shape, dtype=torch.complex128, device="cuda", generator=gen)
        print(f"vjp {shape}, cotangent {seed}", flush=True)
        dA, db, dc = st.vanilla_vjp_hip(G, c, h)
        for axes, got in [((), dc * cc), ((0, 1), 2 * dA[0, 1])] + [((j,), db[j]) for j in range(D)]:
            t = _terms(G, h, axes)
            unit = np.finfo(float).eps * t.abs().square().sum().sqrt()
            sq.append(float((got - _dd_sum(t)).abs() / unit) ** 2)
            del t
    assert np.sqrt(np.mean(sq)) <= 2.5
