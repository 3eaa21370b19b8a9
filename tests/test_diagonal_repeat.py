"""The diagonal strategy's VJP gives the same bits every time.

Every sum of the reverse sweep has a fixed order, so two calls on the same
inputs agree exactly.  At this size the blocks of the middle weights loop over
several groups of params, with their waves far apart.
"""

import pytest
import torch

from mrmustard_amd import workloads as W


@pytest.mark.gpu
@pytest.mark.parametrize("cutoffs", [(10,) * 6, (12, 9, 14, 11)])
def test_diagonal_vjp_repeats(cutoffs):
    from mrmustard_amd.lattice import compact_fock as cf

    A, b, c = W.pnr_dm(len(cutoffs), 3)
    gen = torch.Generator(device="cuda").manual_seed(5)
    g = torch.randn(cutoffs, dtype=torch.complex128, device="cuda", generator=gen)
    first = cf.diagonal_vjp_hip(A, b, c, cutoffs, g, reordered=True)
    for _ in range(15):
        again = cf.diagonal_vjp_hip(A, b, c, cutoffs, g, reordered=True)
        for x, y in zip(first, again):
            assert torch.equal(x, y)
