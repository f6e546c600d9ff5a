"""The tile GEMM kernel where rows are not whole lines (K a multiple of 16, not of 64): every shape with room for
fetching whole lines of them, from the K on where it does so and below, where it fetches slabs, several tiles per
workgroup, operands that begin anywhere in a line with NaN on both sides of them, and products of a batch that begin
differently.

Zeros behind the last element of every row make the same product one of whole slabs, whose loads are others but
whose sums are the same: no bit may differ.  That product is held against float64 as in test_gpu_gemm_ksplit.py."""
import ctypes

import pytest
import torch

from test_gpu_gemm_ksplit import assert_product
from test_gpu_gemm_tiles import forced  # noqa: F401 (fixture)
from tokenweave_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LEAST_RING = ((4, 8), (3, 8))   # lines only where most rows lie on two of them
SHAPES = ((4, 8), (3, 8), (4, 6), (3, 6), (4, 4), (3, 4), (2, 4))


def placed(rows, K, offset, g):
    """[rows, K] that begins `offset` elements into a line, between NaNs."""
    flat = torch.full((rows * K + offset + 128,), float("nan"), dtype=torch.bfloat16, device=DEV)
    t = flat[offset:offset + rows * K].view(rows, K)
    return t.copy_(torch.randn(rows, K, generator=g, device=DEV))


def takes_lines(lib, tm, tn, K):
    return lib.twb_gemm_tile_rows(tm, tn, ctypes.c_int64(K)) == 2


def padded(t):
    return torch.nn.functional.pad(t, (0, -t.shape[1] % 64)).contiguous()


# From 1296 on whole lines: rows begin 2, 6 and 4 chunks of 16 bytes after one another in their lines.
@pytest.mark.parametrize("K", [16, 48, 80, 112, 208, 336, 1072, 1296, 1328, 2080, 2144])
@pytest.mark.parametrize("tm,tn", SHAPES)
def test_every_shape(forced, tm, tn, K):  # noqa: F811
    M, N = 2 * 32 * tm + 17, 2 * 32 * tn + 24         # nine tiles, the last row and column of them partial
    assert takes_lines(forced.lib, tm, tn, K) == (K > 1280 and (K % 32 == 16 or (tm, tn) not in LEAST_RING))
    g = torch.Generator(device=DEV).manual_seed(100 * tm + 10 * tn + K)
    for at_a, at_b in ((0, 0), (8, 48), (32, 56)):
        a, b = placed(M, K, at_a, g), placed(N, K, at_b, g)
        want = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
        forced(want, padded(a), padded(b), None, tm, tn, 0)
        torch.cuda.synchronize()
        assert_product(want, a, b, f"{tm} {tn} {K}")
        for cus in (0, 1, 4):
            print(f"[case] lines {32 * tm}x{32 * tn} K={K} at {at_a} {at_b} cus={cus}", flush=True)
            out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
            forced(out, a, b, None, tm, tn, cus)
            torch.cuda.synchronize()
            assert torch.equal(out, want), (at_a, at_b, cus)


@pytest.mark.parametrize("K", [1296, 2080])
@pytest.mark.parametrize("tm,tn", SHAPES)
def test_bias_and_both_stores(forced, tm, tn, K):  # noqa: F811
    """The stores of a tile, 8 or 16 bytes wide, and its bias lie between the loads that the next tile waits for."""
    M, N = 2 * 32 * tm + 17, 2 * 32 * tn + 24
    g = torch.Generator(device=DEV).manual_seed(tm + 10 * tn + K)
    a, b, bias = placed(M, K, 24, g), placed(N, K, 40, g), torch.randn(N, generator=g, device=DEV).to(torch.bfloat16)
    want = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    forced(want, padded(a), padded(b), None, tm, tn, 0)
    for ld, cus, with_bias in ((N + 8, 1, False), (N + 4, 1, False), (N + 8, 4, True), (N + 4, 4, True), (N + 4, 1, True)):
        print(f"[case] lines {32 * tm}x{32 * tn} K={K} ld={ld} cus={cus} bias={with_bias}", flush=True)
        wide = torch.full((M + 2, ld), 7.0, dtype=torch.bfloat16, device=DEV)     # ld % 8: 16- or 8-byte stores
        forced(wide[1:M + 1, :N], a, b, bias if with_bias else None, tm, tn, cus)
        torch.cuda.synchronize()
        assert torch.equal(wide[1:M + 1, :N], want + bias if with_bias else want), (ld, cus, with_bias)
        assert bool((wide[0] == 7).all() and (wide[-1] == 7).all() and (wide[:, N:] == 7).all())


@pytest.mark.parametrize("P,M,N,K,cap,tile", [(4, 150, 392, 176, None, None), (4, 150, 392, 176, 5, None),
                                              (4, 150, 520, 1296, 8, (3, 6)), (3, 330, 520, 2080, 4, (4, 6))])
def test_a_batch_whose_products_begin_differently(forced, P, M, N, K, cap, tile):  # noqa: F811
    """With a tile: workgroups walk from one product to the next, whose rows begin elsewhere in their lines."""
    if tile:
        tm, tn = ctypes.c_int(), ctypes.c_int()
        forced.lib.twb_gemm_pick_tile(ctypes.c_int64(M), ctypes.c_int64(N), P, cap, ctypes.byref(tm), ctypes.byref(tn))
        tiles = -(-M // (32 * tile[0])) * -(-N // (32 * tile[1]))
        assert (tm.value, tn.value) == tile and takes_lines(forced.lib, *tile, K) and P * tiles >= 3 * cap
    g = torch.Generator(device=DEV).manual_seed(7)
    a = [placed(M, K, 16 * p, g) for p in range(P)]
    b = [placed(N, K, 8 * p + 8, g) for p in range(P)]
    outs = [torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(P)]
    ops.gemm_bf16_nt_partials(outs, a, b, cap)
    for p in range(P):
        want = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
        ops.gemm_bf16_nt(want, padded(a[p]), padded(b[p]))
        assert torch.equal(outs[p], want), p
    assert_product(outs[P - 1], a[P - 1], b[P - 1], "last product")


@pytest.mark.parametrize("M,K", [(200, 7392), (640, 3696)])
def test_long_rows_through_the_library(M, K):
    N, g = 8192, torch.Generator(device=DEV).manual_seed(K)
    a, b = placed(M, K, 16, g), placed(N, K, 8, g)
    out, want = (torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.gemm_bf16_nt(out, a, b)
    ops.gemm_bf16_nt(want, padded(a), padded(b))
    assert torch.equal(out, want)
    assert_product(out[:, -320:], a, b[-320:], f"M={M} K={K}")
