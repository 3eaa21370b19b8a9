"""Gradients of the one-leftover-mode strategy need b as a vector, from the
forward's kept blocks as from a backward with its own forward."""

import pytest
import torch

from mrmustard_amd import workloads as W
from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("columns", [1, 3])
def test_b_with_columns_is_refused(monkeypatch, columns, keep):
    from mrmustard_amd import math
    from mrmustard_amd.lattice import compact_fock as cf

    if not keep:
        monkeypatch.setattr(cf, "LEFTOVER_KEEP_BYTES", 0)
    A, b, c = (torch.as_tensor(x, dtype=torch.complex128, device="cuda") for x in W.pnr_dm(2, 5))
    b = b[:, None].expand(-1, columns).contiguous().requires_grad_(True)
    out = math.hermite_renormalized_1leftoverMode(A, b, c, 4, (3,))
    with pytest.raises(ValueError, match="b"):
        out.real.sum().backward()
    assert b.grad is None
