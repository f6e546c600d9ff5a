"""What the direct calls (`tokenweave_amd._hostpath`) leave to the ordinary routes, as far as it shows
without a GPU; test_gpu_host_path.py has the rest."""
import os
import subprocess
import sys

import pytest
import torch

import tokenweave_amd as tw
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


class AnsweredDirectly:
    """In place of the direct calls: says of every call that it was made."""

    def __getattr__(self, name):
        return lambda *args: "direct"


@pytest.fixture
def layer(monkeypatch):
    monkeypatch.setattr(ops, "_fast", AnsweredDirectly())
    return tw.RMSNorm(8, dtype=torch.bfloat16)


def fused(layer):
    x = torch.zeros(4, 8, dtype=torch.bfloat16)
    handle = tw.PartialsBuffer(1, 4, 8, device="cpu")
    return tw.fused_allreduce_layernorm(layer, x, x.clone(), handle, 4, 0, 1, 0)


@pytest.mark.parametrize("owner,name", [(tw.RMSNorm, "forward"), (tw.RMSNorm, "__call__"),
                                        (torch.nn.Module, "__call__")])
def test_a_replaced_forward_of_the_class_is_called(layer, monkeypatch, owner, name):
    x = torch.zeros(4, 8, dtype=torch.bfloat16)
    assert layer(x) == "direct" and fused(layer) is None
    calls = []
    monkeypatch.setattr(owner, name, lambda self, *args, **kwargs: calls.append(self) or "replaced")
    assert layer(x) == "replaced" and calls == [layer]
    fused(layer)
    assert calls == [layer, layer]


@pytest.mark.parametrize("of_the_class", [True, False])
def test_a_replaced_apply_inplace_is_called(layer, monkeypatch, of_the_class):
    lin = tw.RowParallelLinear(8, 8, bias=False)
    x, out = (torch.zeros(4, 8, dtype=torch.bfloat16) for _ in range(2))
    calls = []

    def replaced(*args, **kwargs):
        calls.append(kwargs["max_cus"])
        return "replaced"
    assert lin(x, out, is_tokenweave=True, gemm_cus=3) == (out, None) and calls == []
    monkeypatch.setattr(type(lin.quant_method) if of_the_class else lin.quant_method, "apply_inplace", replaced)
    assert lin(x, out, is_tokenweave=True, gemm_cus=3) == ("replaced", None) and calls == [3]


class NotUnderTracing:
    def __getattr__(self, name):
        raise AssertionError(f"the direct call {name} was made while tracing")


def test_no_direct_call_while_dynamo_traces(monkeypatch):
    """On CPU tensors every ordinary route ends in its own error."""
    monkeypatch.setattr(ops, "_fast", NotUnderTracing())
    monkeypatch.setattr(ops, "_tracing", lambda: True)
    x, out = (torch.zeros(4, 8, dtype=torch.bfloat16) for _ in range(2))
    w, scale = torch.ones(8, dtype=torch.bfloat16), torch.ones(1)
    layer, lin = tw.RMSNorm(8, dtype=torch.bfloat16), tw.RowParallelLinear(8, 8, bias=False)
    code = torch.empty(4, 8, dtype=torch.float8_e4m3fn)
    for call in (lambda: layer(x), lambda: layer(x, out), lambda: fused(layer),
                 lambda: lin(x, out, is_tokenweave=True),
                 lambda: ops.gemm_bf16_nt(out, x, lin.weight.data),
                 lambda: ops.gemm_bf16_nt_partials([out], [x], [lin.weight.data]),
                 lambda: ops.rms_norm(out, x, w, 1e-6), lambda: ops.rms_norm_inplace(out, x, w, 1e-6),
                 lambda: ops.fused_add_rms_norm(x, out, w, 1e-6),
                 lambda: ops.fused_add_rms_norm_cta(x, out, w, 0, 1e-6),
                 lambda: ops.fused_rs_ln_cta(x, out, w, 0, 0, 0, 1, 0, 1e-6),
                 lambda: ops.fused_rs_ln_ag_cta(x, out, w, 0, 0, 0, 1, 0, 1e-6),
                 lambda: ops.rms_norm_static_fp8_quant(code, x, w, scale, 1e-6),
                 lambda: ops.fused_add_rms_norm_static_fp8_quant(code, x, out, w, scale, 1e-6),
                 lambda: ops.rms_norm_dynamic_per_token_quant(x, w, 1e-6, torch.int8)):
        with pytest.raises(RuntimeError, match="on the GPU only"):
            call()
