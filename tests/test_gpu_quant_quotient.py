"""fp8 codes of the dynamic quantisation are those of the true quotient, byte for byte.

Rows of +-1 (mean square 1, so 1 / rms rounds to 1) make the normalised values equal to
+-weight: each call states the values and the row maximum directly.  The quotients in
the oracle are torch's IEEE float32 division on the CPU."""
import pytest
import torch

from tokenweave_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn


def want_codes(n, ub):
    amax = torch.where(n.isnan(), torch.zeros_like(n), n.abs()).amax(dim=1, keepdim=True).float()
    scale = torch.clamp(torch.clamp(amax, max=ub) / 448.0, min=1.0 / (448.0 * 512.0))
    q = n.float() / scale
    q = torch.where(q.isnan(), torch.full_like(q, 448.0), q.clamp(-448.0, 448.0))
    return q.to(FP8).view(torch.uint8), scale


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["all", "odd", "floor", "bound", "inf", "nan", "zero"])
def test_codes_are_the_true_quotients(dtype, kind):
    gen = torch.Generator().manual_seed(5)
    frac = {torch.bfloat16: 128, torch.float16: 1024}[dtype]
    hidden = 8192 if kind != "odd" else 4099
    tops = torch.arange(128) if frac == 128 and kind == "all" else torch.randint(0, frac, (24,), generator=gen)
    for top in tops.tolist():
        amax = (1.0 + top / frac) * 2.0 ** (-12 if kind == "floor" else 3)
        sig = 1.0 + torch.randint(0, frac, (hidden,), generator=gen) / frac
        if frac == 128:
            sig[:128 * (hidden // 128)] = (1.0 + torch.arange(128) / 128).repeat(hidden // 128)
        w = sig * 2.0 ** torch.randint(-14 if dtype == torch.float16 else -22, 4, (hidden,), generator=gen)
        w = torch.where(w > amax, amax * torch.rand(hidden, generator=gen), w).to(dtype)
        w[0], w[1] = amax, 0.0
        ub = None
        if kind == "bound":
            ub = torch.tensor(amax / 3.0)
        elif kind == "inf":
            w[7] = float("inf")
        elif kind == "nan":
            w[5] = float("nan")
        elif kind == "zero":
            w.zero_()
        sign = torch.ones(2, hidden)
        sign[1] = -1.0
        got, scales = ops.rms_norm_dynamic_per_token_quant(
            sign.to(dtype).cuda(), w.cuda(), 0.0, FP8, None if ub is None else ub.cuda())
        want, want_scales = want_codes(sign.to(dtype) * w, float("inf") if ub is None else ub)
        assert torch.equal(scales.cpu(), want_scales), (top, kind)
        assert torch.equal(got.cpu().view(torch.uint8), want), (top, kind)
