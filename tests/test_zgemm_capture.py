"""The product as a process's first call of the library, inside a graph capture:
it allocates and copies nothing, so the capture holds."""

import os
import subprocess
import sys

import pytest

from tests.conftest import ROOT, gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

PROGRAM = """
import torch
from mrmustard_amd.contraction import zgemm_hip

A, B = (torch.randn(n, dtype=torch.complex128, device="cuda") for n in ((20, 30), (30, 40)))
out = torch.empty(20, 40, dtype=torch.complex128, device="cuda")
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
    zgemm_hip(A, B, out=out)
for k in range(3):
    A.mul_(1j)
    out.zero_()
    graph.replay()
    torch.cuda.synchronize()
    want = A.cpu() @ B.cpu()
    assert float((out.cpu() - want).abs().max()) <= 8 * 30 * 2.0**-52 * float((A.cpu().abs() @ B.cpu().abs()).max())
print("captured")
"""


def test_first_call_inside_a_capture():
    r = subprocess.run([sys.executable, "-c", PROGRAM], cwd=ROOT, env=dict(os.environ, PYTHONPATH=ROOT), capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and r.stdout.strip().endswith("captured"), r.stderr[-2000:]
