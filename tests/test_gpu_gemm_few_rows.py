"""The K-split GEMM kernel where it leaves rows of a unfetched (up to 16 rows) and where b's loads
stream past the caches (up to 64 rows and weights of more than 96 MiB).  Neither may change a bit.

Reference and bound: see test_gpu_gemm_ksplit.py."""
import pytest
import torch

from test_gpu_gemm_ksplit import assert_product
from tokenweave_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def operands(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16),
            torch.randn(N, K, generator=g, device=DEV).to(torch.bfloat16))


def product(a, b):
    out = torch.full((a.shape[0], b.shape[0]), 3.0, dtype=torch.bfloat16, device=DEV)
    ops.gemm_bf16_nt(out, a, b)
    return out


@pytest.mark.parametrize("N,K", [(8192, 320), (1028, 832), (36, 264), (520, 64)])
def test_rows_that_are_not_fetched_reach_no_result(N, K):
    """Row m of a batch is the same in every batch of up to 32 rows, also behind a product that has
    left NaN in the local memory of the compute units."""
    a, b = operands(32, N, K, N + K)
    poison = torch.full((32, K), float("nan"), dtype=torch.bfloat16, device=DEV)
    whole = product(a, b)
    assert_product(whole, a, b, f"N={N} K={K}")
    for M in (1, 7, 8, 9, 15, 16, 17, 31):
        print(f"[case] few rows M={M} N={N} K={K}", flush=True)
        product(poison, b)
        assert torch.equal(product(a[:M].contiguous(), b), whole[:M]), M


@pytest.mark.parametrize("M", [8, 16, 17, 33, 40, 41, 48, 64, 65])
def test_large_weights(M):
    N, K = 6208, 8128                             # 100.9 MB: the streaming form up to 64 rows
    a, b = operands(M, N, K, M)
    out = product(a, b)
    assert_product(out, a, b, f"M={M}")
    small = product(a, b[:512].contiguous())      # the same rows of b in a product that does not stream
    assert torch.equal(out[:, :512], small)


def test_a_batch_whose_weights_are_large_together():
    P, M, N, K = 8, 20, 6152, 1088                # 107 MB together: streams; each one alone does not
    made = [operands(M, N, K, 60 + p) for p in range(P)]
    outs = [torch.empty((M, N), dtype=torch.bfloat16, device=DEV) for _ in range(P)]
    ops.gemm_bf16_nt_partials(outs, [m[0] for m in made], [m[1] for m in made])
    for p, (a, b) in enumerate(made):
        assert torch.equal(outs[p], product(a, b)), p
    assert_product(outs[P - 1], *made[P - 1], "last product")


@pytest.mark.parametrize("M", [65, 72, 80, 88, 96])
def test_a_batch_of_64_row_tiles_has_the_bits_of_products_that_share_rows(M):
    P, N, K = 4, 8192, 1088                       # 71 MB together: tiles of 64 rows; each one alone of 40 or 48
    made = [operands(M, N, K, 70 + p) for p in range(P)]
    outs = [torch.full((M, N), 3.0, dtype=torch.bfloat16, device=DEV) for _ in range(P)]
    ops.gemm_bf16_nt_partials(outs, [m[0] for m in made], [m[1] for m in made])
    for p, (a, b) in enumerate(made):
        assert torch.equal(outs[p], product(a, b)), p
    assert_product(outs[0][:, :512], made[0][0], made[0][1][:512], f"M={M}")


@pytest.mark.parametrize("N,K", [(8192, 320), (1028, 840), (36, 264), (6144, 64)])
def test_two_row_tiles_share_the_rows_evenly(N, K):
    """Row m is the same in every batch of 33 to 128 rows, whose tiles are of 40, 48 or 64 rows, also
    behind a product that has left NaN in the local memory of the compute units."""
    a, b = operands(128, N, K, N + K + 1)
    poison = torch.full((128, K), float("nan"), dtype=torch.bfloat16, device=DEV)
    whole = product(a, b)
    assert_product(whole, a, b, f"N={N} K={K}")
    for M in (33, 40, 41, 48, 49, 56, 57, 64, 65, 80, 81, 96, 97, 112, 113, 127):
        print(f"[case] shared rows M={M} N={N} K={K}", flush=True)
        product(poison, b)
        assert torch.equal(product(a[:M].contiguous(), b), whole[:M]), M


@pytest.mark.parametrize("K", [8, 64, 320, 328])
def test_more_tiles_than_units(K):
    """Launches that give units a second tile keep one slab less in local memory.  Same bits as launches that do
    not, also under a grid cap, where workgroups walk several tiles."""
    N = 8452                                      # 423 tiles of 20 columns for 256 units, the last one partial
    a, b = operands(32, N, K, K)
    for M in (1, 8, 9, 16, 17, 32):
        print(f"[case] more tiles than units M={M} K={K}", flush=True)
        rows = a[:M].contiguous()
        out = product(rows, b)
        assert torch.equal(out[:, :4096], product(rows, b[:4096].contiguous())), M
        assert torch.equal(out[:, 4096:], product(rows, b[4096:].contiguous())), M
        capped = torch.full_like(out, 3.0)
        ops.gemm_bf16_nt(capped, rows, b, max_cus=100)
        assert torch.equal(capped, out), M
    assert_product(out, a, b, f"K={K}")
