"""The flexible vector norm kernel: fp32, hidden sizes and addresses that are not 16-byte aligned, at the
edges of its vectors, lanes and registers.

The reference is float64 arithmetic with the op's rounding points.  In 16-bit types the residual is one
rounding of an exact sum of two (bit-exact) and y may be one unit in the last place off where the fp32
value lies next to a rounding boundary; in fp32 the residual is exact and y carries the error of a
sum of H squares and a handful of operations: 2^-24 (H / 64 + 16) relative (the longest chain of additions
is H / 64 / 8 vectors deep, with room)."""
import pytest
import torch

from tokenweave_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-5
# one element .. whole vectors +- 1, one wave +- 1 vector, two vectors per lane full (2048 vectors)
# and one more, four per lane full (4096) and one more: the element-wise kernel
SIZES_16 = [1, 7, 8, 9, 511, 513, 1025, 5125, 8199, 16383, 16385, 32767, 32769]
SIZES_32 = [1, 3, 4, 5, 255, 257, 2051, 5120, 8191, 8193, 16383, 16384, 16385]


def offset_rows(T, H, dtype, g, shift):
    """[T, H] that begins `shift` elements behind an aligned address, in a buffer whose other
    elements must survive."""
    flat = torch.full((T * H + 32,), 7.0, device=DEV, dtype=dtype)
    flat[shift:shift + T * H].copy_(torch.randn(T * H, generator=g, device=DEV))
    return flat, flat[shift:shift + T * H].view(T, H)


def untouched(flat, shift, n):
    return bool((flat[:shift] == 7).all() and (flat[shift + n:] == 7).all())


@pytest.mark.parametrize("dtype,H", [(d, h) for d in (torch.bfloat16, torch.float16) for h in SIZES_16]
                         + [(torch.float32, h) for h in SIZES_32])
@pytest.mark.parametrize("T,shift", [(3, 0), (2, 1)])
def test_add_norm(dtype, H, T, shift):
    print(f"[case] flex {dtype} T={T} H={H} shift={shift}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(H * 3 + shift)
    fx, x = offset_rows(T, H, dtype, g, shift)
    fr, r = offset_rows(T, H, dtype, g, shift)
    _, w = offset_rows(1, H, dtype, g, shift)
    s = x.double() + r.double()
    want_r = s.to(dtype)
    ref = (want_r.double() / torch.sqrt(s.pow(2).mean(-1, keepdim=True) + EPS) * w.double())
    ops.fused_add_rms_norm(x, r, w.view(-1), EPS)
    torch.cuda.synchronize()
    assert torch.equal(r, want_r)
    if dtype == torch.float32:
        bound = ref.abs() * (2.0 ** -24 * (H / 64 + 16))
    else:
        bound = ref.abs() * (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) + 1e-7
    assert bool(((x.double() - ref).abs() <= bound).all())
    assert untouched(fx, shift, T * H) and untouched(fr, shift, T * H)


@pytest.mark.parametrize("H", [9, 1025, 4104])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_every_output_kind_equals_the_plain_result(dtype, H):
    """rms_norm, the in-place form, both static fp8 ops: the same normalised values, copied or
    quantised; capped grids walk the same rows."""
    T = 5
    g = torch.Generator(device=DEV).manual_seed(H)
    x, r = (torch.randn(T, H, generator=g, device=DEV).to(dtype) for _ in range(2))
    w = torch.randn(H, generator=g, device=DEV).to(dtype)
    y = torch.empty_like(x)
    ops.rms_norm(y, x, w, EPS)
    x2, copy = x.clone(), torch.empty_like(x)
    ops.rms_norm_inplace(copy, x2, w, EPS)
    assert torch.equal(x2, y) and torch.equal(copy, x)
    scale = torch.tensor([0.03], device=DEV)
    code = torch.empty(T, H, device=DEV, dtype=torch.float8_e4m3fn)

    def quantised(t):
        return (t.float() * (1.0 / scale)).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    ops.rms_norm_static_fp8_quant(code, x, w, scale, EPS)
    assert torch.equal(code.view(torch.uint8), quantised(y))
    xa, ra = x.clone(), r.clone()
    ops.fused_add_rms_norm(xa, ra, w, EPS)
    rb = r.clone()
    ops.fused_add_rms_norm_static_fp8_quant(code, x, rb, w, scale, EPS)
    assert torch.equal(code.view(torch.uint8), quantised(xa)) and torch.equal(ra, rb)


@pytest.mark.parametrize("dtype,H", [(torch.bfloat16, 127), (torch.bfloat16, 129), (torch.float16, 127),
                                     (torch.float16, 129), (torch.float32, 64), (torch.float32, 65)])
def test_rows_at_the_line_to_the_element_wise_kernel(dtype, H):
    """Up to 16 vectors of 16 bytes an element a lane, from 17 on a vector a lane."""
    for shift in (0, 1):
        test_add_norm(dtype, H, 3, shift)
    test_every_output_kind_equals_the_plain_result(dtype, H)


@pytest.mark.parametrize("dtype,H", [(d, 264 + tail) for d in (torch.bfloat16, torch.float16) for tail in range(1, 8)]
                         + [(torch.float32, 132 + tail) for tail in range(1, 4)])
def test_every_partial_last_vector(dtype, H):
    """Read with the 16 bytes that end with the row, written in at most three pieces, in place too."""
    for shift in (0, 1):
        test_add_norm(dtype, H, 4, shift)
    test_every_output_kind_equals_the_plain_result(dtype, H)


def element_order_sum(v):
    """Sums of the squares of the rows of `v` (fp32 on the CPU, values of bf16 tensors) with the element-wise kernel's order of
    additions: lane t adds the squares t, t + lanes, ... by fused multiply-adds (the squares are exact in fp32,
    the sums in fp64: one rounding each), 64 lanes as a tree in groups of 16, the rest one after the other."""
    T, H = v.shape
    lanes = (H + 63) // 64 * 64 if H < 1024 else 1024
    squares = torch.zeros(T, (H + lanes - 1) // lanes * lanes, dtype=torch.float64)
    squares[:, :H] = v.double().square()
    acc = torch.zeros(T, lanes)
    for step in squares.view(T, -1, lanes).unbind(1):
        acc = (acc.double() + step).float()
    acc = acc.view(T, -1, 4, 16)
    while acc.shape[-1] > 1:
        acc = acc[..., 0::2] + acc[..., 1::2]
    acc = acc[..., 0]
    waves = ((acc[:, :, 0] + acc[:, :, 1]) + acc[:, :, 2]) + acc[:, :, 3]
    total = waves[:, 0]
    for w in range(1, waves.shape[1]):
        total = total + waves[:, w]
    return total


def norm_factors(rows, H):
    """The kernel's 1 / rms of fp32 rows, read off element 2: 2^-60, whose square vanishes in any sum here."""
    x = torch.zeros(len(rows) * H + 1, device=DEV)[1:].view(len(rows), H)  # unaligned: never the aligned kernels
    x[:, :rows.shape[1]] = rows.to(DEV)
    x[:, 2] = 2.0 ** -60
    y = torch.empty(len(rows), H, device=DEV)
    ops.rms_norm(y, x, torch.ones(H, device=DEV), EPS)
    return (y[:, 2] * 2.0 ** 60).cpu()


@pytest.mark.parametrize("H", [65, 129, 777, 1000, 1025, 1490, 5120, 6663, 8193, 8199, 15873, 16384, 16385, 32767])
def test_sum_is_the_element_wise_kernels(H):
    """The same sum to the last bit as rows that take the element-wise kernel, and so the same norm and codes: a row
    has the factor of a row of two elements whose squares add up to the emulated sum.  (fp32 rows of more than
    16384 elements are the element-wise kernel's own; bf16 rows must have the factors of the fp32 ones.)"""
    T = 100 if H > 8192 else 300
    print(f"[case] flex order T={T} H={H}", flush=True)
    g = torch.Generator().manual_seed(H)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    x[:, 2] = 2.0 ** -60
    w = torch.randn(H, generator=g).to(torch.bfloat16)
    total = element_order_sum(x.float())
    a = total.sqrt() * (1 - 2.0 ** -20)
    b = (total - a * a).sqrt()
    assert torch.equal(a * a + b * b, total)
    inv = norm_factors(x.float(), H)
    assert torch.equal(inv, norm_factors(torch.stack([a, b], 1), H))
    if H < 129:
        return
    want = (x.float() * inv[:, None] * w.float()).to(torch.bfloat16)
    xd = torch.empty(T * H + 1, device=DEV, dtype=torch.bfloat16)[1:].view(T, H)
    xd.copy_(x)
    y, code = torch.empty_like(xd), torch.empty(T, H, device=DEV, dtype=torch.float8_e4m3fn)
    ops.rms_norm(y, xd, w.to(DEV), EPS)
    assert torch.equal(y.cpu(), want)
    scale = torch.tensor([0.03])
    ops.rms_norm_static_fp8_quant(code, xd, w.to(DEV), scale.to(DEV), EPS)
    q = (want.float() * (1.0 / scale)).clamp(-448, 448).to(torch.float8_e4m3fn)
    assert torch.equal(code.cpu().view(torch.uint8), q.view(torch.uint8))
