"""Host side of littlebit_amd.ops (no GPU work)."""
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_imports_on_a_torch_without_gpu_support():
    code = """
import torch
del torch._C._cuda_getCurrentRawStream
import littlebit_amd, littlebit_amd.decode, littlebit_amd.lm_head
s = torch.tensor([[1, -1, 1]], dtype=torch.int8)
assert torch.equal(littlebit_amd.binary_unpacker(littlebit_amd.binary_packer(s), (1, 3)).to(torch.int8), s)
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
