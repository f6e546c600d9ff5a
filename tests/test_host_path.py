"""What the direct calls (`tokenweave_amd._hostpath`) leave to the ordinary routes, as far as it shows
without a GPU; test_gpu_host_path.py has the rest."""
import os
import subprocess
import sys

import pytest

from tokenweave_amd import _custom_ops as ops

pytestmark = pytest.mark.skipif(ops._fast is None, reason="no compiled binding")
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

NESTED = """
import torch, tokenweave_amd as tw
from tokenweave_amd import _custom_ops as ops
rows = torch.nested.nested_tensor([torch.zeros(8), torch.zeros(8)]).to(torch.bfloat16)
layer = tw.RMSNorm(8, dtype=torch.bfloat16)
assert rows.dim() == 2 and type(rows) is torch.Tensor
assert ops._fast.fused_allreduce_layernorm(layer, rows, rows, None, 2, 0, 1, 0, 0, None) is False
assert ops._fast.rms_norm_forward(layer, rows, None, None, None) is NotImplemented
try:
    tw.fused_allreduce_layernorm(layer, rows, rows, None, 2, 0, 1, 0)
except RuntimeError as e:
    print("refused:", str(e).splitlines()[0])
"""


def test_a_tensor_without_sizes_is_refused_and_does_not_end_the_process():
    """A nested tensor throws when asked for its sizes; run apart, because an exception that leaves
    through C frames aborts."""
    done = subprocess.run([sys.executable, "-c", NESTED], cwd=ROOT, capture_output=True, text=True, timeout=300,
                          env=dict(os.environ, PYTHONPATH=ROOT))
    assert done.returncode == 0 and "refused:" in done.stdout, done.stderr[-2000:]
