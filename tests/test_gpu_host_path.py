"""The direct calls (`tokenweave_amd._hostpath`) give what the ordinary routes give, and leave to
them everything that is not a plain call: hooks, autograd, dispatch modes, errors."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import tokenweave_amd as tw
from tokenweave_amd import _custom_ops as ops

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(ops._fast is None, reason="no compiled binding")]
DEV = "cuda:0"
H = 1024


@pytest.fixture
def counted(monkeypatch):
    """Counts, by name, the direct calls that were carried out."""
    done = {}

    class Counting:
        def __getattr__(self, name):
            fn = getattr(real, name)

            def call(*args):
                result = fn(*args)
                if result is not False and result is not NotImplemented:
                    done[name] = done.get(name, 0) + 1
                return result
            return call
    real = ops._fast
    monkeypatch.setattr(ops, "_fast", Counting())
    return done


def tensors(T=5, dtype=torch.bfloat16, seed=3):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x, r = (torch.randn(T, H, generator=g, device=DEV).to(dtype) for _ in range(2))
    layer = tw.RMSNorm(H, dtype=dtype).to(DEV)
    layer.weight.data.copy_(1 + 0.1 * torch.randn(H, generator=g, device=DEV))
    return x, r, layer


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_layer_calls_equal_the_registered_ops(counted, dtype):
    x, r, layer = tensors(dtype=dtype)
    w, eps = layer.weight.data, layer.variance_epsilon
    plain = torch.empty_like(x)
    torch.ops.tokenweave_amd.rms_norm(plain, x, w, eps)
    assert torch.equal(layer(x), plain)
    xa, ra = x.clone(), r.clone()
    torch.ops.tokenweave_amd.fused_add_rms_norm(xa, ra, w, eps)
    xb, rb = x.clone(), r.clone()
    got = layer(xb, residual=rb)
    assert got[0] is xb and got[1] is rb and torch.equal(xb, xa) and torch.equal(rb, ra)
    xc, copy = x.clone(), torch.empty_like(x)
    assert layer(xc, out=copy) is xc and torch.equal(copy, x) and torch.equal(xc, plain)
    assert counted == {"rms_norm_call": 3}


@pytest.mark.parametrize("row_range", [None, (0, 24), (3, 4)])
def test_fused_allreduce_layernorm_equals_the_module_call(counted, row_range):
    P, T, rank = 3, 24, 1
    _, _, layer = tensors()
    g = torch.Generator(device=DEV).manual_seed(9)
    one, two = (tw.PartialsBuffer(P, T, H, rank=rank, device=DEV) for _ in range(2))
    one.storage.copy_(torch.randn(P, T, H, generator=g, device=DEV))
    two.storage.copy_(one.storage)
    r1 = torch.randn(T, H, generator=g, device=DEV).to(torch.bfloat16)
    r2 = r1.clone()
    start, end = row_range or (rank * T // P, (rank + 1) * T // P)
    tw.fused_allreduce_layernorm(layer, one.hidden_states(T), r1, one, T // P, rank, P, 7, row_range=row_range)
    assert counted == {"fused_allreduce_layernorm": 1}
    handle = layer.register_forward_hook(lambda *a: None)   # a hooked module takes the ordinary route
    tw.fused_allreduce_layernorm(layer, two.hidden_states(T), r2, two, T // P, rank, P, 7, row_range=row_range)
    handle.remove()
    assert "fused_allreduce_layernorm" not in counted or counted["fused_allreduce_layernorm"] == 1
    assert torch.equal(one.storage, two.storage) and torch.equal(r1, r2)
    assert not torch.equal(one.local[start:end], r1[start:end])


def test_projections_equal_the_ctypes_route(counted):
    M, N, K = 9, 260, 136
    g = torch.Generator(device=DEV).manual_seed(4)
    x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    for rank in (0, 1):
        lin = tw.RowParallelLinear(K * 2, N, bias=True, tp_rank=rank, tp_size=2).to(DEV)
        lin.weight.data.copy_(torch.randn(N, K, generator=g, device=DEV))
        lin.bias.data.copy_(torch.randn(N, generator=g, device=DEV))
        out, want = (torch.empty(M, N, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        got, bias = lin(x, out, is_tokenweave=True, gemm_cus=5)
        assert got is out and bias is None
        ops.bind_gemm_bf16_nt(want, x, lin.weight.data, None, lin.bias.data if rank == 0 else None)()
        assert torch.equal(out, want)
    outs = [torch.empty(M, N, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    ops.gemm_bf16_nt_partials(outs, (x, x), [lin.weight.data] * 2, None, [lin.bias.data, None])
    ops.bind_gemm_bf16_nt(want, x, lin.weight.data, None, lin.bias.data)()
    assert torch.equal(outs[0], want)
    assert counted == {"row_parallel_inplace": 2, "gemm_bf16_nt_partials": 1}


@pytest.mark.parametrize("kind", [torch.float8_e4m3fn, torch.int8])
def test_dynamic_quant_equals_the_registered_op(counted, kind):
    x, r, layer = tensors(T=7)
    r2 = r.clone()
    out, scales = ops.rms_norm_dynamic_per_token_quant(x, layer.weight.data, 1e-6, kind, None, r)
    want, want_scales = torch.empty_like(x, dtype=kind), torch.empty(7, 1, device=DEV)
    torch.ops.tokenweave_amd.rms_norm_dynamic_per_token_quant(want, x, layer.weight.data, want_scales, 1e-6, None, r2)
    assert torch.equal(out.view(torch.uint8), want.view(torch.uint8)) and torch.equal(scales, want_scales)
    assert torch.equal(r, r2) and scales.shape == (7, 1)
    assert counted == {"rms_norm_dynamic_per_token_quant": 1}


def test_hooks_autograd_and_dispatch_modes_take_the_ordinary_route(counted):
    x, r, layer = tensors()
    seen = []
    handle = layer.register_forward_hook(lambda module, args, out: seen.append(out))
    layer(x.clone(), r.clone())
    handle.remove()
    assert len(seen) == 1 and "rms_norm_call" not in counted

    class Names(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))
    with Names():
        ops.fused_add_rms_norm(x.clone(), r.clone(), layer.weight.data, 1e-6)
    assert "tokenweave_amd.fused_add_rms_norm.default" in seen and "fused_add_rms_norm" not in counted
    leaf = torch.zeros_like(x, requires_grad=True)
    with torch.no_grad():
        ops.rms_norm(leaf, x, layer.weight.data, 1e-6)
    assert counted["rms_norm"] == 1


def test_a_tensor_that_wants_its_gradient_takes_the_ordinary_route(counted):
    x, r, layer = tensors()
    w = layer.weight.data
    want, got = torch.empty_like(x), torch.empty_like(x)
    ops.rms_norm(want, x, w, 1e-6)
    assert counted.pop("rms_norm") == 1
    leaf = x.clone().requires_grad_()
    ops.rms_norm(got, leaf, w, 1e-6)
    assert counted == {} and torch.equal(got.detach(), want)
    with torch.no_grad():
        ops.rms_norm(torch.empty_like(x), leaf, w, 1e-6)
    assert counted == {"rms_norm": 1}


def test_a_lazily_negated_tensor_is_read_with_its_sign(counted):
    """`torch._neg_view` only marks a tensor as negated; the dispatcher resolves the mark before an op
    sees the storage, so such a tensor takes that route, whichever argument it is."""
    x, r, layer = tensors(dtype=torch.float32)
    w = layer.weight.data
    want = torch.empty_like(x)
    ops.rms_norm(want, torch.neg(x), w, 1e-6)
    assert counted.pop("rms_norm") == 1
    neg = torch._neg_view(x)
    assert neg.is_neg() and neg.is_contiguous() and neg.data_ptr() == x.data_ptr()
    got = torch.empty_like(x)
    ops.rms_norm(got, neg, w, 1e-6)
    assert torch.equal(got, want) and torch.equal(layer(neg), want)
    sum_, res = torch.neg(x), r.clone()
    ops.fused_add_rms_norm(sum_, res, w, 1e-6)
    written, res2 = torch._neg_view(x.clone()), r.clone()
    ops.fused_add_rms_norm(written, res2, w, 1e-6)      # an output: written back with its sign
    assert torch.equal(written, sum_) and torch.equal(res, res2)
    ops.rms_norm(got, x, torch._neg_view(w), 1e-6)
    assert torch.equal(got, want)                        # -(x w) = (-x) w
    codes, scales = ops.rms_norm_dynamic_per_token_quant(neg, w, 1e-6, torch.int8)
    want_codes, want_scales = ops.rms_norm_dynamic_per_token_quant(torch.neg(x), w, 1e-6, torch.int8)
    assert torch.equal(codes, want_codes) and torch.equal(scales, want_scales)
    assert counted == {"fused_add_rms_norm": 1, "rms_norm_dynamic_per_token_quant": 1}   # of plain tensors


def test_errors_are_those_of_the_ordinary_route():
    x, r, layer = tensors()
    with pytest.raises(RuntimeError, match="same shape"):
        layer(x, r[:2])
    with pytest.raises(RuntimeError, match="row-contiguous"):
        ops.fused_add_rms_norm(x[:, ::2], r[:, ::2], layer.weight.data, 1e-6)
    with pytest.raises(AssertionError, match="Mismatch in token count"):
        tw.fused_allreduce_layernorm(layer, x, r, tw.PartialsBuffer(2, 5, H, device=DEV), 3, 0, 2, 0)
    with pytest.raises(RuntimeError, match="inner dimensions differ"):
        ops.gemm_bf16_nt(r, x, x[:, :8].contiguous())


def test_the_handles_signal_pads_are_wanted_as_by_the_registered_op(counted):
    """One GPU has no peers to signal, but a handle that cannot name its pads is refused."""
    x, r, layer = tensors()
    buf = tw.PartialsBuffer(1, 5, H, device=DEV)
    with pytest.raises(RuntimeError, match="signal_pads"):
        ops.fused_rs_ln_ag_cta(x, r, layer.weight.data, buf.multicast_ptr, "pads", 0, 1, 0, 1e-6)
    with pytest.raises(RuntimeError, match="signal_pads"):
        ops.fused_rs_ln_cta(x, r, layer.weight.data, buf.multicast_ptr, None, 0, 1, 0, 1e-6)

    class Half:
        multicast_ptr = buf.multicast_ptr
    with pytest.raises(AttributeError, match="signal_pad_ptrs_dev"):
        tw.fused_allreduce_layernorm(layer, x, r, Half(), 5, 0, 1, 0)
    assert counted == {}
    ops.fused_rs_ln_ag_cta(x, r, layer.weight.data, buf.multicast_ptr, 0, 0, 1, 0, 1e-6)
    tw.fused_allreduce_layernorm(layer, x, r, buf, 5, 0, 1, 0)
    assert counted == {"fused_rs_ln_ag_cta": 1, "fused_allreduce_layernorm": 1}
