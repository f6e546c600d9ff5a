"""The tile GEMM kernel, shape by shape: partial tiles in both directions, inner dimensions with a
partial last slab and with fewer slabs than the pipeline is deep, several tiles per workgroup, narrow
stores, bias.  Every shape is forced through the measurement library, with whole and with partial
last slabs; through the library a capped call picks another shape.  Every shape and cap must give the
same bits.

The reference is the product in float64 on the CPU; see test_gpu_gemm_ksplit.py for the bound."""
import ctypes

import pytest
import torch

from helpers import bench_lib
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


SHAPES = ((8, 8), (6, 8), (8, 6), (5, 8), (6, 6), (4, 8), (3, 8), (4, 6), (3, 6), (4, 4), (3, 4), (2, 4))


@pytest.fixture(scope="module")
def forced():
    lib = bench_lib()
    vp, i64, ci = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int
    lib.twb_gemm_bf16_nt_tile.argtypes = [vp, vp, vp, vp, i64, i64, i64, i64, ci, ci, ci, vp]

    def call(out, a, b, bias, tm, tn, cus):
        rc = lib.twb_gemm_bf16_nt_tile(out.data_ptr(), a.data_ptr(), b.data_ptr(), None if bias is None else bias.data_ptr(),
                                       a.shape[0], b.shape[0], a.shape[1], out.stride(0), tm, tn, cus,
                                       torch.cuda.current_stream().cuda_stream)
        assert rc == 0, lib.twb_last_error().decode()

    call.lib = lib
    return call


def test_the_forced_shapes_are_all_there_are(forced):
    tm, tn, found = ctypes.c_int(), ctypes.c_int(), []
    while forced.lib.twb_gemm_tile_shape(len(found), ctypes.byref(tm), ctypes.byref(tn)):
        found.append((tm.value, tn.value))
    assert tuple(found) == SHAPES


@pytest.mark.parametrize("K", [128, 448, 328, 8])     # whole slabs: 2 and 7; a partial last one: the 6th, the only
@pytest.mark.parametrize("tm,tn", SHAPES)
def test_every_shape_with_bias_and_both_stores(forced, tm, tn, K):
    M, N = 2 * 32 * tm + 17, 2 * 32 * tn + 24         # nine tiles, the last row and column of them partial
    a, b, bias = operands(M, N, K, 1000 * tm + 10 * tn + K)
    first = None
    for ld, cus, with_bias in ((N + 8, 0, False), (N + 4, 2, False), (N + 8, 4, True), (N + 4, 1, True)):
        print(f"[case] tile {32 * tm}x{32 * tn} K={K} ld={ld} cus={cus} bias={with_bias}", flush=True)
        wide = torch.full((M + 2, ld), 7.0, dtype=torch.bfloat16, device=DEV)     # ld % 8: 16- or 8-byte stores
        forced(wide[1:M + 1, :N], a, b, bias if with_bias else None, tm, tn, cus)
        torch.cuda.synchronize()
        out = wide[1:M + 1, :N]
        if first is None:
            assert_product(out, a, b, f"{tm} {tn} {K}")
            first = out.clone()
        assert torch.equal(out, first + bias if with_bias else first), (ld, cus, with_bias)
        assert bool((wide[0] == 7).all() and (wide[-1] == 7).all() and (wide[:, N:] == 7).all())
