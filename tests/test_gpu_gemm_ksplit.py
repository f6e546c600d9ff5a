"""The K-split GEMM kernel (few rows) at the edges of its tiles and of its dispatch.

The reference is the product in float64 on the CPU.  The kernel adds fp32 products of exact
bf16 values and rounds once, so |out - ref| <= 2^-8 |ref| (rounding to bf16 is 2^-9 relative; the
other half covers the sum's own error where it moves the value across a rounding boundary) plus
K 2^-23 sum_k |a_k b_k| for the fp32 additions in any order."""
import pytest
import torch

from tokenweave_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def reference(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return a @ b.t(), a.abs() @ b.abs().t()


def assert_product(out, a, b, what):
    ref, magnitude = reference(a, b)
    bound = ref.abs() * 2.0 ** -8 + a.shape[1] * 2.0 ** -23 * magnitude
    assert bool(((out.double().cpu() - ref).abs() <= bound).all()), what


@pytest.mark.parametrize("M", [1, 31, 32, 33, 64, 65, 129, 256, 257])
@pytest.mark.parametrize("N,K", [
    (4, 8),          # one column group, less than one slab
    (260, 264),      # ragged tile in N, a last slab of one chunk, one slab for every wave and one more
    (1024, 192),     # fewer slabs than waves
    (1028, 1016),    # ragged, a last slab of seven chunks
])
def test_tile_edges(M, N, K):
    print(f"[case] ksplit M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M * 131 + N + K)
    a = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    b = torch.randn(N, K, generator=g, device=DEV).to(torch.bfloat16)
    wide = torch.full((M + 2, N + 4), 7.0, dtype=torch.bfloat16, device=DEV)
    out = wide[1:M + 1, :N]
    ops.gemm_bf16_nt(out, a, b)
    capped = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    ops.gemm_bf16_nt(capped, a, b, max_cus=3)     # the workgroups walk several tiles each
    torch.cuda.synchronize()
    assert_product(out, a, b, f"M={M} N={N} K={K}")
    assert torch.equal(out, capped), "the grid cap changed bits"
    assert bool((wide[0] == 7).all() and (wide[-1] == 7).all() and (wide[:, N:] == 7).all())


def test_several_products_in_one_launch_and_bias():
    P, M, N, K = 3, 40, 520, 328
    g = torch.Generator(device=DEV).manual_seed(11)
    a = [torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16) for _ in range(P)]
    b = [torch.randn(N, K, generator=g, device=DEV).to(torch.bfloat16) for _ in range(P)]
    bias = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)
    outs = [torch.empty((M, N), dtype=torch.bfloat16, device=DEV) for _ in range(P)]
    ops.gemm_bf16_nt_partials(outs, a, b, biases=[bias, None, None])
    for p in range(P):
        one = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
        ops.gemm_bf16_nt(one, a[p], b[p])
        torch.cuda.synchronize()
        assert_product(one, a[p], b[p], f"product {p}")
        assert torch.equal(outs[p], one + bias if p == 0 else one)


def test_inner_dimension_beyond_the_tile_descriptors():
    """K > 2^24: the rows of a tile would span more than the 32-bit offsets hold."""
    M, N, K = 3, 4, (1 << 24) + 8
    g = torch.Generator(device=DEV).manual_seed(5)
    a = torch.randn(M, K, generator=g, device=DEV, dtype=torch.bfloat16)
    b = torch.randn(N, K, generator=g, device=DEV, dtype=torch.bfloat16)
    out = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    ops.gemm_bf16_nt(out, a, b)
    torch.cuda.synchronize()
    assert_product(out, a, b, "large K")


@pytest.mark.parametrize("M", [65, 300])
@pytest.mark.parametrize("N", [32, 36])
def test_few_columns_and_more_than_64_rows(M, N):
    test_tile_edges(M, N, 328)
