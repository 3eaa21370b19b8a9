"""Gradients of the one-leftover-mode strategy from the forward's kept blocks
are the bits that a backward with its own forward gives, on every call."""

import pytest
import torch

from mrmustard_amd import workloads as W
from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


@pytest.mark.parametrize("o,pnr", [(3, (0,)), (19, (14, 14)), (1, (6, 1, 5)), (40, (2, 0, 3)), (4, (3, 2, 2, 3))])
@pytest.mark.parametrize("reordered", [True, False])
def test_kept_equals_recomputed(monkeypatch, o, pnr, reordered):
    from mrmustard_amd import math
    from mrmustard_amd.lattice import compact_fock as cf

    A, b, c = (torch.as_tensor(x, dtype=torch.complex128, device="cuda") for x in W.pnr_dm(len(pnr) + 1, 5))
    gen = torch.Generator(device="cuda").manual_seed(2)
    g = torch.randn((o + 1, o + 1, *(k + 1 for k in pnr)), dtype=torch.complex128, device="cuda", generator=gen)

    def grads(times):
        xs = [x.clone().requires_grad_(True) for x in (A, b, c)]
        out = math.hermite_renormalized_1leftoverMode(*xs, o, pnr, reordered)
        return [torch.autograd.grad(out, xs, grad_outputs=g, retain_graph=True) for _ in range(times)]

    kept = grads(2)
    monkeypatch.setattr(cf, "LEFTOVER_KEEP_BYTES", 0)
    for want, *got in zip(*grads(1), *kept):
        for x in got:
            assert torch.equal(want, x)
