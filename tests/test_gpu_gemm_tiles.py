"""The tile GEMM kernel, shape by shape: partial tiles in both directions, inner dimensions with a
partial last slab and with fewer slabs than the pipeline is deep, several tiles per workgroup, narrow
stores, bias.  The shape is forced through the measurement library where it has an entry for it
and by the grid cap otherwise: a capped call picks another shape, and every shape and cap must
give the same bits.

The reference is the product in float64 on the CPU; see test_gpu_gemm_ksplit.py for the bound."""
import pytest
import torch

from test_gpu_gemm_ksplit import assert_product
from tokenweave_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CAPS = (1, 2, 3, 5, 8, 13, 24, 40, 64, 100, 160, 200)


def operands(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    a = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    b = torch.randn(N, K, generator=g, device=DEV).to(torch.bfloat16)
    bias = torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)
    return a, b, bias


@pytest.mark.parametrize("M,N,K", [
    (129, 64, 8),        # the smallest: one slab of one chunk
    (160, 516, 64),      # one whole slab, N % 8 != 0: 8-byte stores
    (257, 384, 72),      # two slabs, the second of one chunk
    (700, 776, 200),     # four slabs, three chunks in the last: as deep as the pipeline
    (1025, 1032, 448),   # one row and eight columns past whole tiles of every shape
    (2049, 264, 1016),
])
def test_every_cap_gives_the_reference_product_and_the_same_bits(M, N, K):
    a, b, bias = operands(M, N, K, M + N + K)
    wide = torch.full((M + 2, N + 4), 7.0, dtype=torch.bfloat16, device=DEV)
    out = wide[1:M + 1, :N]
    ops.gemm_bf16_nt(out, a, b)
    torch.cuda.synchronize()
    assert_product(out, a, b, f"M={M} N={N} K={K}")
    biased = out + bias
    for cap in CAPS:
        print(f"[case] tiles M={M} N={N} K={K} cap={cap}", flush=True)
        capped = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.gemm_bf16_nt(capped, a, b, max_cus=cap, bias=bias if cap % 2 else None)
        torch.cuda.synchronize()
        assert torch.equal(capped, biased if cap % 2 else out), cap
    assert bool((wide[0] == 7).all() and (wide[-1] == 7).all() and (wide[:, N:] == 7).all())


def test_products_of_a_batch_have_the_bits_of_single_calls():
    P, M, N, K = 5, 300, 520, 328
    made = [operands(M, N, K, 40 + p) for p in range(P)]
    outs = [torch.empty((M, N), dtype=torch.bfloat16, device=DEV) for _ in range(P)]
    for cap in (None, 7):
        ops.gemm_bf16_nt_partials(outs, [m[0] for m in made], [m[1] for m in made], cap,
                                  [made[0][2]] + [None] * (P - 1))
        for p, (a, b, bias) in enumerate(made):
            one = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
            ops.gemm_bf16_nt(one, a, b, bias=bias if p == 0 else None)
            torch.cuda.synchronize()
            assert torch.equal(outs[p], one), (cap, p)
