"""Host side of littlebit_amd.ops (no GPU work)."""
import subprocess
import sys
from pathlib import Path
from types import SimpleNamespace

import pytest
import torch

from littlebit_amd import ops

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


@pytest.mark.parametrize("bad", [0, 1, 2])
def test_chain_link_names_the_residual_it_refuses(monkeypatch, bad):
    tensors = [torch.zeros(1, 4) for _ in range(6)]
    outs, residuals = tensors[:3], tensors[3:]

    def require(t, name):  # every other tensor passes as if it were on the GPU
        if t is residuals[bad]:
            raise RuntimeError(f"{name} must be a GPU tensor")

    monkeypatch.setattr(ops, "_require_cuda", require)
    projections = [SimpleNamespace(in_features=8, out_features=4) for _ in outs]
    with pytest.raises(RuntimeError, match=rf"residuals\[{bad}\]"):
        ops.ChainLink(projections, outs, residuals=residuals)
