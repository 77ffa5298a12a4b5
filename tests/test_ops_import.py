"""katsu_amd.ops imports on a torch without a GPU build, which lacks torch._C's CUDA functions."""
import os
import subprocess
import sys

SCRIPT = """
import torch
for name in [n for n in dir(torch._C) if n.startswith("_cuda")]:
    delattr(torch._C, name)
from katsu_amd import ops
try:
    ops.conv2d_forward(torch.zeros(1, 1, 4, 4), torch.zeros(1, 1, 3, 3), 1, 1)
except ValueError as e:
    assert "device tensors" in str(e)
else:
    raise AssertionError("host tensors were taken")
"""


def test_imports_without_gpu_build():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", SCRIPT], capture_output=True, text=True, cwd=root)
    assert r.returncode == 0, r.stderr
