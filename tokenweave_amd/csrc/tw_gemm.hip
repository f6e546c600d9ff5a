// bf16 "NT" GEMM on gfx950 MFMA:  out[M, N] = a[M, K] * b[N, K]^T, fp32
// accumulate, bf16 out.  This is the row-parallel o_proj / down_proj that
// produces one rank's partial sum in the token-weave schedule; the reference
// runs it as torch.matmul(x, W.t(), out=) (vllm/model_executor/layers/
// linear.py:203-228).
//
// Both operands are K-contiguous, so the 8 consecutive k a lane feeds to an MFMA are one
// 16-byte chunk of a row of `a` or `b`.  The MFMAs are issued with `b` rows as their first
// operand, which leaves every lane with 4 consecutive n per accumulator quad.
//
// Three kernels:
//  * gemm_bf16_nt_ksplit_kernel (at most 128 rows): tiles of 8 to 64 rows and at most 32 or 64 columns
//    whose four waves share the inner dimension;
//  * gemm_bf16_nt_tile_kernel<TM, TN, ROWS> (more rows): (32 TM) x (32 TN) tiles, 64 x 128 to 256 x 256,
//    picked per problem so that the tile count wastes the fewest workgroup rounds;
//  * gemm_bf16_nt_kernel (K > 2^24, where a tile's rows outgrow 32-bit offsets): 128 x 128 x 64
//    tiles, 4 waves, register-staged loads into padded LDS, 64-bit addresses.
// The first two bring operand slabs from global memory straight into LDS (buffer_load ... lds: no
// staging registers, no LDS store instructions).  A wave instruction fills 1 KiB = 8 LDS rows of
// 128 bytes with whole lines of eight operand rows; the 16-byte chunks of a row are permuted by the
// row number so that fragment reads are conflict-free without padding.  A last partial k-slab is
// zero-filled, and the descriptors end with the operand, so that tile rows past M or N read as zeros.
// Workgroups walk the tile list with stride gridDim.x (grid cap = compute-unit budget of the weave
// schedule), and tile ids are remapped so that the workgroups of one XCD (blockIdx % 8) share operand
// panels in that XCD's L2.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>

#include "tw_common.h"

namespace tw {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int BM = 128, BN = 128, BK = 64;
constexpr int LDS_ROW = BK + 8;  // elements; 144-byte row pitch
constexpr int GEMM_THREADS = 256;
constexpr int CHUNKS_PER_ROW = BK / 8;                           // 16-byte chunks per tile row
constexpr int LOADS_PER_THREAD = BM * CHUNKS_PER_ROW / GEMM_THREADS;  // 4
constexpr int GROUP_M = 8;  // tile rows per column sweep (operand reuse in L2)

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// The optional bias of the in-place linear is added the way the reference adds it
// (vllm/model_executor/layers/linear.py:224-228: torch.matmul(..., out=output), then
// output += bias): to the product already rounded to bf16, in fp32, rounded again.
// `packed` and `bias2` hold two bf16 each, element 2i in the low half.
__device__ __forceinline__ uint32_t add_bias2(uint32_t packed, uint32_t bias2) {
  const float lo = __uint_as_float(packed << 16) + __uint_as_float(bias2 << 16);
  const float hi = __uint_as_float(packed & 0xffff0000u) + __uint_as_float(bias2 & 0xffff0000u);
  return pack2(lo, hi);
}

__global__ __launch_bounds__(GEMM_THREADS) void gemm_bf16_nt_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ a, const uint16_t* __restrict__ b,
    const uint16_t* __restrict__ bias, int M, int N, int K, int64_t ldc, int tiles_m, int tiles_n) {
  __shared__ __attribute__((aligned(16))) uint16_t lds_a[2][BM * LDS_ROW];
  __shared__ __attribute__((aligned(16))) uint16_t lds_b[2][BN * LDS_ROW];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int l32 = lane & 31, lhi = lane >> 5;
  const int num_tiles = tiles_m * tiles_n;
  const int nk = (K + BK - 1) / BK;

  for (int t = blockIdx.x; t < num_tiles; t += gridDim.x) {
    // XCD-aware remap: ids congruent mod 8 run on one XCD; give each XCD a
    // contiguous range of the grouped tile order.
    int pid = t;
    {
      const int per_xcd = num_tiles / 8;
      const int body = per_xcd * 8;
      if (t < body) pid = (t & 7) * per_xcd + (t >> 3);
    }
    const int group_size = GROUP_M * tiles_n;
    const int group = pid / group_size;
    const int first_m = group * GROUP_M;
    const int rows_in_group = min(tiles_m - first_m, GROUP_M);
    const int tm_idx = first_m + (pid % group_size) % rows_in_group;
    const int tn_idx = (pid % group_size) / rows_in_group;
    const int m0 = tm_idx * BM, n0 = tn_idx * BN;

    f32x16_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    uint4 ra[LOADS_PER_THREAD], rb[LOADS_PER_THREAD];
    auto fetch = [&](int kt) {
#pragma unroll
      for (int i = 0; i < LOADS_PER_THREAD; ++i) {
        const int c = tid + i * GEMM_THREADS;
        const int row = c / CHUNKS_PER_ROW, kc = c % CHUNKS_PER_ROW;
        const int k = kt * BK + kc * 8;
        const int am = min(m0 + row, M - 1);  // rows past M are computed, never stored
        const int bn = min(n0 + row, N - 1);
        if (k < K) {
          ra[i] = *reinterpret_cast<const uint4*>(a + (size_t)am * K + k);
          rb[i] = *reinterpret_cast<const uint4*>(b + (size_t)bn * K + k);
        } else {
          ra[i] = make_uint4(0, 0, 0, 0);
          rb[i] = make_uint4(0, 0, 0, 0);
        }
      }
    };
    auto stash = [&](int buf) {
#pragma unroll
      for (int i = 0; i < LOADS_PER_THREAD; ++i) {
        const int c = tid + i * GEMM_THREADS;
        const int row = c / CHUNKS_PER_ROW, kc = c % CHUNKS_PER_ROW;
        *reinterpret_cast<uint4*>(&lds_a[buf][row * LDS_ROW + kc * 8]) = ra[i];
        *reinterpret_cast<uint4*>(&lds_b[buf][row * LDS_ROW + kc * 8]) = rb[i];
      }
    };

    fetch(0);
    __syncthreads();  // previous tile's readers are done with both buffers
    stash(0);
    __syncthreads();

    for (int kt = 0; kt < nk; ++kt) {
      const int buf = kt & 1;
      if (kt + 1 < nk) fetch(kt + 1);
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) {
        bf16x8_t fa[2], fb[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int ar = wm * 64 + i * 32 + l32;
          const int br = wn * 64 + i * 32 + l32;
          fa[i] = __builtin_bit_cast(
              bf16x8_t, *reinterpret_cast<const uint4*>(&lds_a[buf][ar * LDS_ROW + kk * 16 + lhi * 8]));
          fb[i] = __builtin_bit_cast(
              bf16x8_t, *reinterpret_cast<const uint4*>(&lds_b[buf][br * LDS_ROW + kk * 16 + lhi * 8]));
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
      }
      if (kt + 1 < nk) stash(buf ^ 1);
      __syncthreads();
    }

    // acc[i][j][4*q + e] = out[m0 + wm*64 + i*32 + l32][n0 + wn*64 + j*32 + 8*q + 4*lhi + e]
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int m = m0 + wm * 64 + i * 32 + l32;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = n0 + wn * 64 + j * 32 + 8 * q + 4 * lhi;
          if (n < N) {
            uint2 v;
            v.x = pack2(acc[i][j][4 * q + 0], acc[i][j][4 * q + 1]);
            v.y = pack2(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
            if (bias) {  // N % 4 == 0: the four columns lie inside the row; bias is 8-byte aligned
              const uint2 bv = *reinterpret_cast<const uint2*>(bias + n);
              v.x = add_bias2(v.x, bv.x);
              v.y = add_bias2(v.y, bv.y);
            }
            *reinterpret_cast<uint2*>(out + (size_t)m * ldc + n) = v;
          }
        }
      }
    }
  }
}

// `count` independent products of one shape in one launch: out[p] = a[p] * b[p]^T.  The
// token-weave producer uses it for the P row-parallel partial sums of a token split,
// each written into its rank's staging slot; a plain GEMM is count = 1.
struct GemmBatch {
  uint16_t* out[TW_MAX_PARTIALS];
  const uint16_t* a[TW_MAX_PARTIALS];
  const uint16_t* b[TW_MAX_PARTIALS];
  const uint16_t* bias[TW_MAX_PARTIALS];  // [N] bf16 or null: added to that product only
};

// ---------------------------------------------------------------------------
// K-split kernel: few rows (a decode step, a short prefill chunk).  The product is bound by
// reading b once, so what counts is how many compute units stream it and how evenly.
//
// A workgroup owns 8 LA rows (in MT blocks of 32) x at most 32 NT columns of the output and its four waves share the
// inner dimension: wave w takes the 64-wide k-slabs w, w + 4, ... .  Each wave brings its slabs of both operands from
// global memory straight into LDS of its own, STAGES slabs deep, and reads its fragments back from there: no barrier
// in the k loop, a wave only waits for its own loads.  (Three stages up to 32 rows where no unit has a second tile,
// see ksplit_form, and up to 40 where rows are whole lines: [36, 768] x [6144, 768]^T 4.89 -> 4.68 us, [36, 2048]
// 7.10 -> 6.76, [36, 3584] x [8192, 3584]^T 11.3 -> 11.2, but [36, 3696] 12.6 -> 12.7 and [64, 3584] 12.6 -> 12.9;
// four are no better: what a unit has under way is bounded by its L1, not by LDS.)  The four partial tiles meet in
// LDS at the end and are added as ((w0+w1)+w2)+w3. Every load covers whole 128-byte lines of eight rows.  The sum of
// an output element does not depend on the tile it lies in (nor on MT, NT, the grid or the number of products).
//
// The launcher makes the tiles just wide enough for one (or a whole number of) workgroups per
// compute unit: 32 columns at N = 8192, 24 at N = 6144.  Measured on 256 units, operands
// rotated through 1.25 GB / through three sets: [32, 3584] x [8192, 3584]^T 13.6 / 11.2 us
// (59 MB: 4.4 / 5.3 TB/s) against 65 / 47 us with 64 workgroups of 128 x 128; K = 1024: 5.2 us
// against 16 us; [128, 3584]: 21 / 15 us against 69 / 50 us.
//
// What is short is also bound by the way to the first load: with rows past 16 or 8 not fetched, the partial
// last slab in an instantiation of its own, no division for one product of one row tile and every pointer
// fetched at the start, three sets: [8, 1024] 5.7 -> 4.8 us, [32, 1024] 5.8 -> 5.2, [32, 3584] 11.2 -> 10.7,
// [64, 1024] 6.6 -> 6.3, [96, 768] x [6144, 768]^T 6.0 -> 5.7.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void lds_void_t;
typedef float f32x4_t __attribute__((ext_vector_type(4)));
constexpr int KS_WAVES = 4;
constexpr int KS_THREADS = KS_WAVES * 64;
constexpr int KS_ROWB = 128;                      // bytes of a slab row: 64 elements
constexpr uint32_t KS_OUT_OF_RANGE = 0x80000000u; // a tile's rows span at most 2 GiB (KS_MAX_K)
constexpr int64_t KS_MAX_K = 1 << 24;

constexpr int ks_lds_bytes(int mt, int nt, int stages) {
  const int slabs = KS_WAVES * stages * 32 * (mt + nt) * KS_ROWB;
  const int sums = KS_WAVES * 32 * mt * (32 * nt * 4 + 16);
  return slabs > sums ? slabs : sums;
}

// One operand's share of a slab, 8 rows per wave instruction; `last`: the last slab of an inner
// dimension that is no multiple of 64 (TAIL), whose chunks past K must arrive as zeros (`even` / `odd`
// say whether this lane's chunk of an even / odd 8-row block is inside).
template <int L, int AUX, bool TAIL, int LV>
__device__ __forceinline__ void ks_issue(__amdgpu_buffer_rsrc_t d, const uint32_t (&v)[LV], uint8_t* s, uint32_t koff,
                                         bool last, bool even, bool odd) {
  if (TAIL && last) {
#pragma unroll
    for (int j = 0; j < L; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(d, (lds_void_t*)(s + j * 1024), 16,
                                               ((j & 1) ? odd : even) ? v[j] : KS_OUT_OF_RANGE, koff, 0, AUX);
  } else {
#pragma unroll
    for (int j = 0; j < L; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(d, (lds_void_t*)(s + j * 1024), 16, v[j], koff, 0, AUX);
  }
}

// LA: the tile's 8-row blocks of a: 4 MT, or only as many as its share of the rows needs (the rest of its MFMA
// blocks is then whatever LDS holds: it reaches no output row but its own, which is not stored).
// BAUX: cache policy of b's loads.
template <int MT, int NT, int STAGES, int LA, int BAUX, bool TAIL>
__global__ __launch_bounds__(KS_THREADS) void gemm_bf16_nt_ksplit_kernel(
    GemmBatch batch, int count, int M, int N, int K, int64_t ldc, int tiles_m, int tiles_n, int cols) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass only needs the stub, and cannot instantiate the device builtins
  constexpr int RA = 32 * MT, RB = 32 * NT, LB = RB / 8, ROWS = 8 * LA;
  static_assert(ROWS <= RA, "a tile's rows fit its MFMA blocks");
  constexpr int STAGE = (RA + RB) * KS_ROWB;
  static_assert(STAGES == 2 || STAGES == 3, "the k loop waits for at most two slabs beside the one in use");
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds_ks[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lhi = lane >> 5;
  const int nk = (K + BK - 1) / BK;
  const int tail_chunks = (K % BK) / 8;
  const bool even = TAIL && ((lane & 7) ^ (lane >> 4)) < tail_chunks;
  const bool odd = TAIL && ((lane & 7) ^ (lane >> 4) ^ 4) < tail_chunks;
  // Row r of a slab keeps its 16-byte chunk c at position c ^ ((r >> 1) & 7) (see the file
  // comment).  Offsets are inside the tile: its descriptors begin at its first row and end
  // behind its last one, so that rows past M, N or the tile's columns read as zeros.
  uint32_t va[LA], vb[LB], roff[4];
#pragma unroll
  for (int j = 0; j < (LA > LB ? LA : LB); ++j) {
    const int chunk = (lane & 7) ^ (((j & 1) << 2) | (lane >> 4));
    const uint32_t v = (uint32_t)((j * 8 + (lane >> 3)) * (int64_t)K + chunk * 8) * 2u;
    if (j < LA) va[j] = v;
    if (j < LB) vb[j] = v;
  }
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) roff[kk] = l32 * KS_ROWB + ((((kk << 1) | lhi) ^ ((l32 >> 1) & 7)) << 4);
  uint8_t* const mine = lds_ks + wave * (STAGES * STAGE);

  const int tiles_per_product = tiles_m * tiles_n;
  const int num_tiles = count * tiles_per_product;
  for (int t = blockIdx.x; t < num_tiles; t += gridDim.x) {
    // Every XCD a contiguous range of tiles, the row tiles of one column range next to each other:
    // they read the same rows of b through one L2.
    int pid = t;
    const int per_xcd = num_tiles / 8;
    if (t < per_xcd * 8) pid = (t & 7) * per_xcd + (t >> 3);
    // One product of one row tile, the usual call, needs no division and finds its pointers among the first
    // arguments fetched; `out` and `bias` are asked for here, not behind the k loop.
    const uint16_t *a = batch.a[0], *b = batch.b[0], *bias = batch.bias[0];
    uint16_t* out = batch.out[0];
    if (count > 1) {
      const int product = pid / tiles_per_product;
      pid -= product * tiles_per_product;
      a = batch.a[product];
      b = batch.b[product];
      bias = batch.bias[product];
      out = batch.out[product];
    }
    int m0 = 0, n0 = pid * cols;
    if (tiles_m > 1) {
      const int column = pid / tiles_m;
      m0 = (pid - column * tiles_m) * ROWS;
      n0 = column * cols;
    }
    const __amdgpu_buffer_rsrc_t da = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(a) + (size_t)m0 * K, 0, (uint32_t)min(M - m0, ROWS) * (uint32_t)K * 2u, 0x00020000);
    const __amdgpu_buffer_rsrc_t db = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(b) + (size_t)n0 * K, 0, (uint32_t)min(N - n0, cols) * (uint32_t)K * 2u, 0x00020000);

    f32x16_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    // slabs `wave`, wave + 4, ..., STAGES - 1 ahead; b first: it is the operand that comes from far
    int next = wave;
    uint32_t fill = 0, use = 0;
    auto issue = [&]() {
      const bool last = next == nk - 1;
      uint8_t* s = mine + fill;
      ks_issue<LB, BAUX, TAIL>(db, vb, s + RA * KS_ROWB, (uint32_t)next * KS_ROWB, last, even, odd);
      ks_issue<LA, 0, TAIL>(da, va, s, (uint32_t)next * KS_ROWB, last, even, odd);
      next += KS_WAVES;
      fill = fill == (STAGES - 1) * STAGE ? 0 : fill + STAGE;
    };
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i)
      if (next < nk) issue();
    for (int slab = wave; slab < nk; slab += KS_WAVES, use = use == (STAGES - 1) * STAGE ? 0 : use + STAGE) {
      if (next < nk) {  // wait for all but the slabs behind this one
        issue();
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * (LA + LB)) : "memory");
      } else if (STAGES == 3 && slab + KS_WAVES < nk) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LA + LB) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      const uint8_t* pa = mine + use;
      const uint8_t* pb = pa + RA * KS_ROWB;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        bf16x8_t fa[MT], fb[NT];
#pragma unroll
        for (int i = 0; i < MT; ++i)
          fa[i] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(pa + i * 32 * KS_ROWB + roff[kk]));
#pragma unroll
        for (int j = 0; j < NT; ++j)
          fb[j] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(pb + j * 32 * KS_ROWB + roff[kk]));
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
      }
      // the fragments are in registers: the loads issued next may overwrite this stage
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }

    // acc[i][j][4 q + e] = partial sum of out[m0 + i*32 + l32][n0 + j*32 + 8 q + 4 lhi + e].
    // The slab stages become the four waves' fp32 tiles (rows padded by 16 bytes).
    constexpr int PITCH = RB * 4 + 16;
    __syncthreads();
    uint8_t* const sums = lds_ks + wave * (RA * PITCH);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<f32x4_t*>(sums + (i * 32 + l32) * PITCH + (j * 32 + 8 * q + 4 * lhi) * 4) =
              f32x4_t{acc[i][j][4 * q + 0], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    __syncthreads();
    for (int g = tid; g < ROWS * RB / 4; g += KS_THREADS) {
      const int m = g / (RB / 4), c = (g % (RB / 4)) * 4;
      if (m0 + m < M && c < cols && n0 + c < N) {  // N and cols are multiples of 4
        const uint8_t* p = lds_ks + m * PITCH + c * 4;
        f32x4_t s = *reinterpret_cast<const f32x4_t*>(p);
#pragma unroll
        for (int w = 1; w < KS_WAVES; ++w) s += *reinterpret_cast<const f32x4_t*>(p + w * (RA * PITCH));
        uint2 v = {pack2(s.x, s.y), pack2(s.z, s.w)};
        if (bias) {
          const uint2 bv = *reinterpret_cast<const uint2*>(bias + n0 + c);
          v.x = add_bias2(v.x, bv.x);
          v.y = add_bias2(v.y, bv.y);
        }
        *reinterpret_cast<uint2*>(out + (size_t)(m0 + m) * ldc + n0 + c) = v;
      }
    }
    __syncthreads();  // the next tile's slabs overwrite the sums
  }
#endif
}

// ---------------------------------------------------------------------------
// Tile kernel: (32 TM) x (32 TN) x 64 tiles for everything with more rows.
//
// Four waves (2 x 2, one per SIMD), each (16 TM) x (16 TN) of the output in 16 x 16 accumulators
// held in accumulation registers (256 of them for the 256 x 256 tile), v_mfma_f32_16x16x32_bf16:
// its 4-register accumulators cost less register traffic than 32 x 32 ones, and a 128 x 128 wave
// tile reads a third fewer fragment bytes from LDS per flop than the 64 x 128 one of eight waves.
//
// One wave per SIMD hides nothing behind other waves, so everything is placed by hand between the
// MFMAs of the k loop and pinned there by scheduling barriers:
//  * A slab (64 of the inner dimension) is two phases of TM * TN MFMAs, one per 32 of it.  While a
//    phase runs on one set of fragments the other set is read from LDS for the next one: no MFMA
//    waits for LDS, also not across slabs or tiles.
//  * Between the phases lies the slab's one barrier.  It says that this slab's LDS is free and
//    that the next slab has arrived: a wave waits for its own loads before it, D - 1 slabs after
//    it issued them.
//  * Operand slabs go from global memory straight into LDS, D slabs ahead, one load per several
//    MFMAs: the compute unit's path to memory takes 64 bytes per cycle, half of the 256 x 256
//    tile's loop, and loads issued in a burst stall the waves behind it (all 16 loads of a wave in
//    half a phase: 786 us for 8192^3, spread over a phase 749, over the slab 714).
//  * The slab sequence runs on across tiles: a workgroup keeps its compute unit and walks the tile
//    list with stride gridDim.x, the first D slabs of the next tile are under way while the
//    accumulators of the last one are stored, and its first barrier does not wait for those stores
//    (vmcnt counts in order: they are younger than the loads it needs).  Where whole lines are fetched, the slab
//    without products between two tiles does not wait for them, the next tile's first slab does.
//  * Results leave by 16-byte stores from the registers.  The columns a lane holds are made
//    adjacent by the row order in which b's fragments are read: MFMA row r of the tile pair
//    (2 p, 2 p + 1) is column 32 p + 8 (r / 4) + 4 (tile & 1) + r % 4 of the wave's columns.  They are
//    written through (nt sc0 sc1): all compute units store 33 MB at the same moment, and what
//    stays dirty in the L2s is in the way of the next tile's loads (8192 x 8192 x 1024: 107 us, default
//    policy 112, nt 116).
// LDS: rows of 128 bytes, 16-byte chunk c of row r at position c ^ key(r), key(r) = (r >> 1) & 7 for
// a and bits 1, 3, 4 of r for b: the 16 rows that a fragment read touches at once are
// conflict-free (counter-verified).  256 x 256: three a panels and two b panels, exactly 160 KiB.
//
// The MFMAs are written as inline assembly with the accumulators tied to accumulation registers:
// left to choose, the register allocator moves accumulators between the two files and spills
// (112 against 107 us, 8192 x 8192 x 1024).
//
// Measured against the 8-wave kernel this replaces, same box: 8192^3 874 -> 714 us (1 253 -> 1 539
// TFLOP/s; matrix cores now busy 86 % of the cycles in which a unit has work, at a clock of 1.82 GHz and
// less under the board's power limit), 8192 x 8192 x 3584 406 -> 325, 8192 x 8192 x 1024 127 -> 107,
// 1024 x 8192 x 3712 59 -> 48, 512 x 8192 x 3584 49 -> 28 us.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(3))) uint8_t lds_u8_t;
typedef __attribute__((address_space(3))) const bf16x8_t lds_frag_t;
constexpr int TILE_THREADS = 256;
constexpr int64_t TILE_MAX_K = 1 << 21;    // a tile's rows span less than 2 GiB: the out-of-range marker below
constexpr int64_t TILE_MAX_LDC = 1 << 21;
[[maybe_unused]] constexpr uint32_t TILE_OUT_OF_RANGE = 0x80000000u;

// How a tile shape uses LDS and where in a slab (slots: its 2 TM TN MFMAs) its loads go out.
enum TileRows { kWholeSlabs, kPartialSlab, kLines };  // see the kernel
template <int TM, int TN, TileRows ROWS = kWholeSlabs>
struct TileShape {
  static constexpr int BM = 32 * TM, BN = 32 * TN, SLOTS = TM * TN;
  static constexpr int LA = TM, LB = TN, L = LA + LB;  // wave loads (8 rows each) per slab and operand
  static constexpr int PA = BM * 128, PB = BN * 128;   // panel bytes
  static constexpr int STAGES = 160 * 1024 / (PA + PB);
  // Two whole stages only: a third a panel, so that a's loads can go out in the phase before the
  // barrier, b's in the one behind it.
  static constexpr bool TAKES_LINES = 4 * PA + 3 * PB <= 160 * 1024;
  static constexpr bool LINES = ROWS == kLines;
  static_assert(!LINES || TAKES_LINES, "no room for the line behind the slab in use");
  static constexpr bool TIGHT = LINES ? STAGES < 4 : STAGES == 2;
  static constexpr int NEED = LINES ? 2 : 1;  // slabs behind the one in use that its barrier waits for
  // slabs ahead; three at most: with four or five the 64- to 128-row tiles take longer to start than they
  // gain ([256, 1024] x [8192, 1024]^T 8.3 -> 8.8 us, [160, 3584] x [8192, 3584]^T 18.2 -> 18.8).  Rows of
  // whole lines end in the line behind their slab: one more there.
  static constexpr int D = LINES ? (STAGES < 5 ? 3 : 4) : TIGHT ? 2 : (STAGES - 1 < 3 ? STAGES - 1 : 3);
  static constexpr int SA = D + 1, SB = TIGHT ? D : D + 1;
  static constexpr int LDS = SA * PA + SB * PB;
  static constexpr int SPREAD = 2 * SLOTS / L;
  static constexpr int A0 = TIGHT ? 1 : 0, A_STEP = TIGHT ? SLOTS / LA : SPREAD;
  static constexpr int B0 = TIGHT ? SLOTS + 1 : LA * SPREAD, B_STEP = TIGHT ? SLOTS / LB : SPREAD;
  static constexpr int READ_STEP = SLOTS / L / 2 < 1 ? 1 : SLOTS / L / 2;
  // loads that go out before the barrier
  static constexpr int before(int first, int step, int n) {
    int c = 0;
    for (int l = 0; l < n; ++l) c += first + l * step < SLOTS ? 1 : 0;
    return c;
  }
  static constexpr int EARLY = before(A0, A_STEP, LA) + before(B0, B_STEP, LB);
  // may be outstanding at a slab's barrier: slabs NEED + 1 .. D - 1 ahead and the early part of slab D
  static constexpr int IN_FLIGHT = (D - 1 - NEED) * L + EARLY;
  static constexpr int STORES = SLOTS / 2;
  static_assert(SPREAD >= 1 && D > NEED && LDS <= 160 * 1024 && IN_FLIGHT + STORES <= 63, "tile shape");
  static_assert(A0 + (LA - 1) * A_STEP < 2 * SLOTS && B0 + (LB - 1) * B_STEP < 2 * SLOTS, "every load has a slot");
  static_assert((L - 1) * READ_STEP < SLOTS, "every fragment read has a slot");
};

#ifdef __HIP_DEVICE_COMPILE__  // the host pass only needs the kernels' stubs
__device__ __forceinline__ void tile_mfma_first(f32x4_t& c, const bf16x8_t& x, const bf16x8_t& y) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(x), "v"(y));
}
__device__ __forceinline__ void tile_mfma(f32x4_t& c, const bf16x8_t& x, const bf16x8_t& y) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(x), "v"(y));
}
__device__ __forceinline__ uint32_t tile_pack2(float lo, float hi) {
  float x, y;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(lo));
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(y) : "a"(hi));
  return pack2(x, y);
}

// One phase: acc += fb x fa, and between the MFMAs the next phase's fragments (na, nb from pa, pb)
// and this half's share of the loads of the slab D ahead.
template <int TM, int TN, TileRows ROWS, bool FIRST, int HALF>
__device__ __forceinline__ void tile_phase(f32x4_t (&acc)[TM][TN], const bf16x8_t (&fa)[TM], const bf16x8_t (&fb)[TN],
                                           bf16x8_t (&na)[TM], bf16x8_t (&nb)[TN], const lds_u8_t* pa,
                                           const lds_u8_t* pb, __amdgpu_buffer_rsrc_t da,
                                           __amdgpu_buffer_rsrc_t db, const uint32_t (&va)[TM],
                                           const uint32_t (&vb)[TN], lds_u8_t* sa, lds_u8_t* sb, uint32_t koff) {
  using S = TileShape<TM, TN, ROWS>;
#pragma unroll
  for (int n = 0; n < S::SLOTS; ++n) {
    const int i = n / TN, j = n % TN, slot = n + HALF * S::SLOTS;
    if (FIRST) tile_mfma_first(acc[i][j], fb[j], fa[i]);
    else tile_mfma(acc[i][j], fb[j], fa[i]);
    __builtin_amdgcn_sched_barrier(0);
    if (n % S::READ_STEP == 0 && n / S::READ_STEP < S::L) {
      const int r = n / S::READ_STEP;
      if (r < TN) nb[r] = *(lds_frag_t*)(pb + (r >> 1) * 4096 + (r & 1) * 512);
      else na[r - TN] = *(lds_frag_t*)(pa + (r - TN) * 2048);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (slot >= S::A0 && (slot - S::A0) % S::A_STEP == 0 && (slot - S::A0) / S::A_STEP < S::LA) {
      const int l = (slot - S::A0) / S::A_STEP;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(da, (lds_void_t*)(sa + l * 1024), 16, va[l], koff, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (slot >= S::B0 && (slot - S::B0) % S::B_STEP == 0 && (slot - S::B0) / S::B_STEP < S::LB) {
      const int l = (slot - S::B0) / S::B_STEP;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(db, (lds_void_t*)(sb + l * 1024), 16, vb[l], koff, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// The loads of one half of a slab, where no MFMAs are to be had between them.
template <int TM, int TN, TileRows ROWS, int HALF>
__device__ __forceinline__ void tile_loads(__amdgpu_buffer_rsrc_t da, __amdgpu_buffer_rsrc_t db,
                                           const uint32_t (&va)[TM], const uint32_t (&vb)[TN], lds_u8_t* sa,
                                           lds_u8_t* sb, uint32_t koff) {
  using S = TileShape<TM, TN, ROWS>;
#pragma unroll
  for (int l = 0; l < S::LA; ++l)
    if ((S::A0 + l * S::A_STEP >= S::SLOTS) == (HALF == 1))
      __builtin_amdgcn_raw_ptr_buffer_load_lds(da, (lds_void_t*)(sa + l * 1024), 16, va[l], koff, 0, 0);
#pragma unroll
  for (int l = 0; l < S::LB; ++l)
    if ((S::B0 + l * S::B_STEP >= S::SLOTS) == (HALF == 1))
      __builtin_amdgcn_raw_ptr_buffer_load_lds(db, (lds_void_t*)(sb + l * 1024), 16, vb[l], koff, 0, 0);
}

constexpr int kStoreThrough = 19;  // nt sc0 sc1

// The wave's accumulators: row 16 i of `dc` at voffset + i * row_step.  WIDE: eight columns per
// store, else four (rows that are only 8-byte aligned, or N % 8 != 0).
template <int TM, int TN, bool WIDE, bool BIAS>
__device__ __forceinline__ void tile_store(const f32x4_t (&acc)[TM][TN], __amdgpu_buffer_rsrc_t dc, uint32_t row_off,
                                           uint32_t row_step, int n, int N, const uint16_t* bias) {
  uint32_t off[TN];  // of four columns each, out of range when they lie past N
  uint2 bv[BIAS ? TN : 1];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int c = n + (j >> 1) * 32 + (j & 1) * 4;
    off[j] = c < N ? row_off + (uint32_t)((j >> 1) * 64 + (j & 1) * 8) : TILE_OUT_OF_RANGE;
    if (BIAS) bv[j] = c < N ? *reinterpret_cast<const uint2*>(bias + c) : make_uint2(0, 0);
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; j += 2) {
      u32x4_t v = {tile_pack2(acc[i][j][0], acc[i][j][1]), tile_pack2(acc[i][j][2], acc[i][j][3]),
                   tile_pack2(acc[i][j + 1][0], acc[i][j + 1][1]), tile_pack2(acc[i][j + 1][2], acc[i][j + 1][3])};
      if (BIAS)
        v = u32x4_t{add_bias2(v.x, bv[j].x), add_bias2(v.y, bv[j].y), add_bias2(v.z, bv[j + 1].x),
                    add_bias2(v.w, bv[j + 1].y)};
      if (WIDE) {
        __builtin_amdgcn_raw_buffer_store_b128(v, dc, off[j] + (uint32_t)i * row_step, 0, kStoreThrough);
      } else {
        __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{v.x, v.y}, dc, off[j] + (uint32_t)i * row_step, 0, kStoreThrough);
        __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{v.z, v.w}, dc, off[j + 1] + (uint32_t)i * row_step, 0,
                                              kStoreThrough);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Where the loader stands: product, tile and slab of the next slab to request.
struct TilePlace {
  int product, m0, n0;
};

// Where in its 128-byte line a row begins, in 16-byte chunks.
__device__ __forceinline__ int line_phase(const uint16_t* row) {
  return (int)(reinterpret_cast<uintptr_t>(row) >> 4) & 7;
}

template <int TM, int TN>
__device__ __forceinline__ TilePlace tile_place(int t, int num_tiles, int tiles_m, int tiles_n) {
  using S = TileShape<TM, TN>;
  // Tile rows per sweep over the columns: the 32 tiles an XCD works on at a time then form a block
  // that needs the fewest operand bytes through that XCD's L2.
  constexpr int GROUP = S::BN >= 2 * S::BM ? 8 : 4;
  // Every XCD (workgroup ids congruent mod 8) gets a contiguous range of the tile order: with
  // eight products, one product each.
  int pid = t;
  const int per_xcd = num_tiles / 8;
  if (t < per_xcd * 8) pid = (t & 7) * per_xcd + (t >> 3);
  const int per_product = tiles_m * tiles_n;
  const int product = pid / per_product;
  pid -= product * per_product;
  const int sweep = GROUP * tiles_n, group = pid / sweep, first = group * GROUP, rows = min(tiles_m - first, GROUP);
  return {product, (first + (pid % sweep) % rows) * S::BM, ((pid % sweep) / rows) * S::BN};
}
#endif

// kPartialSlab: the last slab is a partial one.  (Apart from the others because switching the offsets costs
// the k loop a register move per load and slab: 341 against 324 us for 8192 x 8192 x 3584.  Zeroing the
// fragments instead needs no moves and is no faster, 227 against 230 us for 16384 x 8192 x 1000.)
//
// kLines: rows of such a K are not whole lines, and a slab of a row mostly lies on two of them, which a compute
// unit then requests twice ([1000, 3696] x [8192, 3696]^T: 9.9 million requests, 1.73 a slab row; its L1 has about 126
// under way whatever the kernel does).  Here a load fetches the lines themselves, one a row and slab (5.7 million
// requests, 1.01), and a fragment read finds the first part of its slab in the ring's panel of that slab and the rest
// in the next one.  That wants one panel more in the ring, and K % 16 == 0: rows two apart then begin at the
// same place of a line or half a line apart, which the swizzle takes care of.  Aligned 64 bytes have to stay with
// groups of four lanes: rotated by other amounts the loads take half of the gain back.  Same bits.
// Requests that miss the L2s gain most.  One product with 8192 columns, kPartialSlab -> kLines, weights from memory /
// three sets in turn, us: K = 3696, 200 rows 36.3 -> 27.4 / 26.2 -> 23.8, 256: 41.3 -> 30.8 / 27.5 -> 24.1, 512: 47.4
// -> 40.4 / 37.0 -> 33.5, 640: 69.4 -> 49.7 / 48.9 -> 41.4, 800: 71.5 -> 70.7 / 49.7 -> 50.6, 1000: 77.0 -> 71.1 /
// 55.0 -> 51.8; K = 7392 (both from memory), 200 rows 61 -> 50, 256: 72 -> 57, 512: 85 -> 77, 640: 122 -> 96.  On one
// set again and again the units are busy 4 % fewer cycles at 1000 rows and 3 to 7 % more at 200.
template <int TM, int TN, TileRows ROWS>
__global__ __attribute__((amdgpu_waves_per_eu(1, 1))) __launch_bounds__(TILE_THREADS) void gemm_bf16_nt_tile_kernel(
    GemmBatch batch, int count, int M, int N, int K, int64_t ldc, int tiles_m, int tiles_n, int wide_store) {
#ifdef __HIP_DEVICE_COMPILE__
  using S = TileShape<TM, TN, ROWS>;
  constexpr int LA = S::LA, LB = S::LB, PA = S::PA, PB = S::PB, D = S::D;
  constexpr uint32_t AHEAD = S::LINES ? 128 : 0;  // the loads' offsets begin a line ahead of the tile
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds_tile[];
  lds_u8_t* const lds_a = (lds_u8_t*)lds_tile;
  lds_u8_t* const lds_b = lds_a + S::SA * PA;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1, r16 = lane & 15, quad = lane >> 4;
  const int nk = (K + BK - 1) / BK, nl = nk + (S::LINES ? 1 : 0);  // slabs; loads of a tile
  const int tail_chunks = ROWS == kPartialSlab ? (K % BK) / 8 : 8;  // 16-byte chunks of the last slab that lie inside K
  const int num_tiles = count * tiles_m * tiles_n;

  // Reader: the two 32-wide halves of a slab.
  const uint32_t row_a = (wm * 16 * TM + r16) * 128, row_b = (wn * 16 * TN + (r16 >> 2) * 8 + (r16 & 3)) * 128;
  const uint32_t chunk0 = (quad ^ (r16 >> 1)) << 4, chunk1 = ((4 + quad) ^ (r16 >> 1)) << 4;
  const lds_u8_t *a0 = lds_a + row_a + chunk0, *a1 = lds_a + row_a + chunk1;
  const lds_u8_t *b0 = lds_b + row_b + chunk0, *b1 = lds_b + row_b + chunk1;
  // Loader: wave instruction l fills the 8-row block wave * L + l; lane l lands at row l / 8,
  // position l % 8 of it and fetches the chunk that belongs there.  Offsets are inside the tile,
  // whose descriptors end with the last row of the operand: rows past it read as zeros.
  lds_u8_t* const wa = lds_a + wave * LA * 1024;
  lds_u8_t* const wb = lds_b + wave * LB * 1024;
  uint32_t va[LA], vb[LB];
  // `chunks`: how many of a row's chunks exist in the slab; the others must arrive as zeros
#define TW_TILE_OFFSETS(chunks)                                                                              \
  do {                                                                                                       \
    _Pragma("unroll") for (int l = 0; l < LA; ++l) {                                                         \
      const int blk = wave * LA + l, c = (lane & 7) ^ (((blk & 1) << 2) | (lane >> 4));                      \
      va[l] = c < (chunks) ? (uint32_t)((blk * 8 + (lane >> 3)) * K + c * 8) * 2u : TILE_OUT_OF_RANGE;       \
    }                                                                                                        \
    _Pragma("unroll") for (int l = 0; l < LB; ++l) {                                                         \
      const int blk = wave * LB + l, c = (lane & 7) ^ (((lane >> 4) & 1) | ((blk & 3) << 1));                \
      vb[l] = c < (chunks) ? (uint32_t)((blk * 8 + (lane >> 3)) * K + c * 8) * 2u : TILE_OUT_OF_RANGE;       \
    }                                                                                                        \
  } while (0)
  // kLines: the same for line `line` of every row: lane position x holds the line's chunk x ^ key ^ flip, so
  // that aligned groups of four lanes fetch aligned 64 bytes.  kc: the chunk of the row that this is.
#define TW_TILE_LINE_OFFSET(v, blk, key, phase, line)                                                        \
  do {                                                                                                       \
    const int row = (blk)*8 + (lane >> 3), j = (lane & 7) ^ (key) ^ (flip & (row << 1));                     \
    const int kc = (line)*8 + j - (((phase) + row * row_chunks) & 7);                                        \
    v = kc >= 0 && kc < row_chunks ? (uint32_t)(row * K + (kc - (line)*8 + 8) * 8) * 2u : TILE_OUT_OF_RANGE; \
  } while (0)
#define TW_TILE_LINE_OFFSETS(line)                                                                           \
  do {                                                                                                       \
    _Pragma("unroll") for (int l = 0; l < LA; ++l)                                                           \
        TW_TILE_LINE_OFFSET(va[l], wave * LA + l, (((wave * LA + l) & 1) << 2) | (lane >> 4), load_phase_a, line); \
    _Pragma("unroll") for (int l = 0; l < LB; ++l) TW_TILE_LINE_OFFSET(                                      \
        vb[l], wave * LB + l, ((lane >> 4) & 1) | (((wave * LB + l) & 3) << 1), load_phase_b, line);         \
  } while (0)
  const int row_chunks = K / 8;
  const int flip = (row_chunks & 2) << 1;  // 4 where rows two apart begin half a line apart
  int load_phase_a = 0, load_phase_b = 0;  // where in a line the product's first row begins, in chunks
  // Load cursor: slab lk of tile lt.  Past the last tile it stays at slab 0 of an empty descriptor:
  // its loads ask memory for nothing.  (The hardware compares with the extent less the slab's offset,
  // which for an extent of 0 must not go below 0.)
  int lt = blockIdx.x, lk = 0;
  __amdgpu_buffer_rsrc_t da, db;
#define TW_TILE_DESCRIPTORS()                                                                                \
  do {                                                                                                       \
    const bool in = lt < num_tiles;                                                                          \
    const TilePlace p = tile_place<TM, TN>(in ? lt : 0, num_tiles, tiles_m, tiles_n);                        \
    const uint16_t *pa = batch.a[p.product] + (size_t)p.m0 * K, *pb = batch.b[p.product] + (size_t)p.n0 * K; \
    if (S::LINES) load_phase_a = line_phase(pa), load_phase_b = line_phase(pb);                              \
    da = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(pa) - (int)AHEAD / 2, 0,                    \
                                           in ? (uint32_t)min(M - p.m0, S::BM) * (uint32_t)K * 2u + AHEAD : 0u, \
                                           0x00020000);                                                      \
    db = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(pb) - (int)AHEAD / 2, 0,                    \
                                           in ? (uint32_t)min(N - p.n0, S::BN) * (uint32_t)K * 2u + AHEAD : 0u, \
                                           0x00020000);                                                      \
  } while (0)
#define TW_TILE_ADVANCE()                                                                                    \
  do {                                                                                                       \
    if (lt < num_tiles) ++lk;                                                                                \
    if (lk == nl) {                                                                                          \
      lk = 0;                                                                                                \
      lt += gridDim.x;                                                                                       \
      TW_TILE_DESCRIPTORS();                                                                                 \
      if (S::LINES) TW_TILE_LINE_OFFSETS(0);                                                                 \
      else if (ROWS == kPartialSlab) TW_TILE_OFFSETS(nk == 1 ? tail_chunks : 8);                             \
    } else if (S::LINES && (lk == 1 || lk >= nk - 1)) {                                                      \
      if (lt < num_tiles) TW_TILE_LINE_OFFSETS(lk);                                                          \
    } else if (ROWS == kPartialSlab && lk == nk - 1) {                                                       \
      TW_TILE_OFFSETS(tail_chunks);                                                                          \
    }                                                                                                        \
  } while (0)
  TW_TILE_DESCRIPTORS();
  if (S::LINES) TW_TILE_LINE_OFFSETS(0);
  else TW_TILE_OFFSETS(nk == 1 ? tail_chunks : 8);
#pragma unroll
  for (int s = 0; s < D; ++s) {
#pragma unroll
    for (int l = 0; l < LA; ++l)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(da, (lds_void_t*)(wa + s * PA + l * 1024), 16, va[l], lk * 128u, 0, 0);
#pragma unroll
    for (int l = 0; l < LB; ++l)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(db, (lds_void_t*)(wb + s * PB + l * 1024), 16, vb[l], lk * 128u, 0, 0);
    TW_TILE_ADVANCE();
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((D - S::NEED) * S::L) : "memory");
  f32x4_t acc[TM][TN];
  bf16x8_t fa0[TM], fb0[TN], fa1[TM], fb1[TN];
  // ring positions: the slab in use and the one being filled
  uint32_t use_a = 0, use_b = 0, fill_a = (D % S::SA) * PA, fill_b = (D % S::SB) * PB;
#define TW_NEXT(x, panel, n) ((x) + (panel) == (n) * (panel) ? 0u : (x) + (panel))
#define TW_RING(x, panel, n) x = TW_NEXT(x, panel, n)
  // kLines: the chunks 8 - phase and up of a row's slab lie in the line behind it.  The fragments of a lane are rows
  // that begin alike in their lines.
  bool next_a0 = false, next_a1 = false, next_b0 = false, next_b1 = false;
  auto place_reader = [&](int t) {
    const TilePlace p = tile_place<TM, TN>(t, num_tiles, tiles_m, tiles_n);
    const int pa = line_phase(batch.a[p.product]) + (r16 & 1) * row_chunks, fa = (pa & 7) ^ (flip & (r16 << 1));
    const int pb = line_phase(batch.b[p.product]) + (r16 & 1) * row_chunks, fb = (pb & 7) ^ (flip & (r16 << 1));
    next_a0 = quad + fa >= 8, next_a1 = 4 + quad + fa >= 8;
    next_b0 = quad + fb >= 8, next_b1 = 4 + quad + fb >= 8;
    a0 = lds_a + row_a + ((((quad + pa) & 7) ^ (r16 >> 1)) << 4);
    a1 = lds_a + row_a + ((((4 + quad + pa) & 7) ^ (r16 >> 1)) << 4);
    b0 = lds_b + row_b + ((((quad + pb) & 7) ^ (r16 >> 1)) << 4);
    b1 = lds_b + row_b + ((((4 + quad + pb) & 7) ^ (r16 >> 1)) << 4);
  };
#define TW_AT(x, ptr, next, panel, n) ((ptr) + (S::LINES && (next) ? TW_NEXT(x, panel, n) : (x)))
#define TW_TILE_READ_FIRST()                                                                                 \
  do {                                                                                                       \
    const lds_u8_t *const pb = TW_AT(use_b, b0, next_b0, PB, S::SB), *const pa = TW_AT(use_a, a0, next_a0, PA, S::SA); \
    _Pragma("unroll") for (int r = 0; r < TN; ++r)                                                           \
        fb0[r] = *(lds_frag_t*)(pb + (r >> 1) * 4096 + (r & 1) * 512);                                       \
    _Pragma("unroll") for (int r = 0; r < TM; ++r) fa0[r] = *(lds_frag_t*)(pa + r * 2048);                   \
  } while (0)
  if (S::LINES) place_reader(blockIdx.x);
  TW_TILE_READ_FIRST();
#define TW_TILE_SLAB(FIRST, AFTER_STORE)                                                                         \
  do {                                                                                                       \
    tile_phase<TM, TN, ROWS, FIRST, 0>(acc, fa0, fb0, fa1, fb1, TW_AT(use_a, a1, next_a1, PA, S::SA),          \
                                       TW_AT(use_b, b1, next_b1, PB, S::SB), \
                                       da, db, va, vb, wa + fill_a, wb + fill_b, lk * 128u);                 \
    if (AFTER_STORE)                                                                                         \
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(S::IN_FLIGHT + S::STORES) : "memory"); \
    else                                                                                                     \
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(S::IN_FLIGHT) : "memory");            \
    TW_RING(use_a, PA, S::SA);                                                                               \
    TW_RING(use_b, PB, S::SB);                                                                               \
    tile_phase<TM, TN, ROWS, false, 1>(acc, fa1, fb1, fa0, fb0, TW_AT(use_a, a0, next_a0, PA, S::SA),          \
                                       TW_AT(use_b, b0, next_b0, PB, S::SB), \
                                       da, db, va, vb, wa + fill_a, wb + fill_b, lk * 128u);                 \
    TW_TILE_ADVANCE();                                                                                       \
    TW_RING(fill_a, PA, S::SA);                                                                              \
    TW_RING(fill_b, PB, S::SB);                                                                              \
  } while (0)

  for (int t = blockIdx.x; t < num_tiles; t += gridDim.x) {
    TW_TILE_SLAB(true, !S::LINES && t != (int)blockIdx.x);
    for (int kt = 1; kt < nk; ++kt) TW_TILE_SLAB(false, false);

    const TilePlace p = tile_place<TM, TN>(t, num_tiles, tiles_m, tiles_n);
    const uint16_t* __restrict__ bias = batch.bias[p.product];
    const __amdgpu_buffer_rsrc_t dc = __builtin_amdgcn_make_buffer_rsrc(
        batch.out[p.product] + (size_t)p.m0 * ldc + p.n0, 0, (uint32_t)min(M - p.m0, S::BM) * (uint32_t)ldc * 2u,
        0x00020000);
    const int col = wn * 16 * TN + quad * 8;
    const uint32_t row_off = (uint32_t)((wm * 16 * TM + r16) * (int)ldc + col) * 2u, row_step = (uint32_t)ldc * 32u;
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last MFMA's result is written
    if (bias) {
      if (wide_store) tile_store<TM, TN, true, true>(acc, dc, row_off, row_step, p.n0 + col, N, bias);
      else tile_store<TM, TN, false, true>(acc, dc, row_off, row_step, p.n0 + col, N, bias);
    } else {
      if (wide_store) tile_store<TM, TN, true, false>(acc, dc, row_off, row_step, p.n0 + col, N, bias);
      else tile_store<TM, TN, false, false>(acc, dc, row_off, row_step, p.n0 + col, N, bias);
    }
    // The tile's rows have one line more than slabs: a slab without products between this tile and the next.
    if (S::LINES && t + (int)gridDim.x < num_tiles) {
      tile_loads<TM, TN, ROWS, 0>(da, db, va, vb, wa + fill_a, wb + fill_b, lk * 128u);
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(S::IN_FLIGHT + S::STORES) : "memory");
      TW_RING(use_a, PA, S::SA);
      TW_RING(use_b, PB, S::SB);
      place_reader(t + gridDim.x);
      TW_TILE_READ_FIRST();
      tile_loads<TM, TN, ROWS, 1>(da, db, va, vb, wa + fill_a, wb + fill_b, lk * 128u);
      TW_TILE_ADVANCE();
      TW_RING(fill_a, PA, S::SA);
      TW_RING(fill_b, PB, S::SB);
    }
  }
#undef TW_TILE_SLAB
#undef TW_TILE_READ_FIRST
#undef TW_AT
#undef TW_NEXT
#undef TW_RING
#undef TW_TILE_ADVANCE
#undef TW_TILE_DESCRIPTORS
#undef TW_TILE_LINE_OFFSETS
#undef TW_TILE_LINE_OFFSET
#undef TW_TILE_OFFSETS
#endif
}

// More than 64 KiB of dynamic LDS must be allowed once per function and device.
static int allow_lds(const void* kernel, std::atomic<bool>* ok, int max_devices, int bytes) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= max_devices)
    return set_error(TW_ERR_LAUNCH, "gemm_bf16_nt: no current device");
  if (!ok[dev].load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess)
      return set_error(TW_ERR_LAUNCH, "gemm_bf16_nt: the device refused %d bytes of LDS", bytes);
    ok[dev].store(true, std::memory_order_release);
  }
  return TW_OK;
}
constexpr int kMaxDevices = 64;

// A K-split launch's tiles: as few rounds of one workgroup per unit as full-width tiles need, and then tiles no
// wider than that many rounds require, so that every unit streams its share of b.  The rounds are the whole batch's:
// with those of one product alone its tiles were up to `count` times too narrow, us: two products [32, 1024] x [2048,
// 1024]^T 6.2 -> 5.0, eight 19.2 -> 9.2, eight [32, 1024] x [6144, 1024]^T 26.2 -> 23.1, four [64, 1024] x [4096,
// 1024]^T 20.1 -> 12.9 (weights from memory).
struct KsTiles { int64_t m, n; int cols; };
static KsTiles ksplit_tiles(int64_t M, int64_t N, int count, int rows, int most_cols, int cus) {
  const int64_t tiles_m = (M + rows - 1) / rows, full = (N + most_cols - 1) / most_cols;
  const int64_t row_tiles = count * tiles_m, rounds = (row_tiles * full + cus - 1) / cus;
  const int64_t per_row_tile = std::max(full, cus * rounds / row_tiles);  // column tiles those rounds have room for
  const int cols = (int)std::min<int64_t>(most_cols, ((N + per_row_tile - 1) / per_row_tile + 3) / 4 * 4);
  return {tiles_m, (N + cols - 1) / cols, cols};
}

template <int MT, int NT, int STAGES, int LA, int BAUX, bool TAIL>
static int launch_ksplit(const GemmBatch& batch, int count, int64_t M, int64_t N, int64_t K, int64_t ldc, int max_cus,
                         int cus, hipStream_t hs) {
  constexpr int LDS = ks_lds_bytes(MT, NT, STAGES);
  static std::atomic<bool> lds_ok[kMaxDevices];
  const auto kernel = gemm_bf16_nt_ksplit_kernel<MT, NT, STAGES, LA, BAUX, TAIL>;
  if (int rc = allow_lds(reinterpret_cast<const void*>(kernel), lds_ok, kMaxDevices, LDS)) return rc;
  const KsTiles tiles = ksplit_tiles(M, N, count, 8 * LA, 32 * NT, cus);
  int64_t grid = count * tiles.m * tiles.n;
  if (max_cus > 0 && grid > max_cus) grid = max_cus;
  launch_kernel(kernel, dim3((unsigned)grid), dim3(KS_THREADS), LDS, hs, batch, count, (int)M, (int)N, (int)K, ldc,
                (int)tiles.m, (int)tiles.n, tiles.cols);
  return TW_OK;
}

// b's loads carry the non-temporal bit (KS_STREAM) where a launch's weights are so large that the last-level
// cache (256 MB) does not keep three of them.  Not beyond 64 rows (128 rows: 37.4 / 37.6, the unit's outstanding lines
// are shared with a), and not where rows of b are not whole lines: the line that two slabs share would be fetched twice
// (8 rows, K = 3696: 11.1 -> 13.4).
// From memory b arrives faster that way at every size, and past the caches too.  us, default / streaming, N = 8192:
//                    weights from memory                       three sets in turn            one set again and again
//   K = 1024 (17 MB)  8 rows 5.43 / 5.11, 32: 5.96 / 5.64    5.22 / 4.65, 5.56 / 5.23      3.59 / 3.60, 3.94 / 3.95
//   K = 2048 (34 MB)  8      8.69 / 7.71, 32: 9.37 / 8.66    7.50 / 7.25, 7.85 / 8.34      4.84 / 5.22, 6.23 / 6.84
//   K = 3584 (59 MB)  8     12.20 / 10.87, 32: 13.63 / 12.65 10.78 / 10.48, 11.24 / 12.47  10.78 / 9.11, 11.19 / 11.49
//   K = 5120 (84 MB)  8     16.30 / 14.76, 32: 19.60 / 18.42 14.06 / 14.37, 14.83 / 18.20  14.04 / 13.13, 14.78 / 17.47
//   K = 7168 (117 MB) 8     21.72 / 19.15, 32: 24.95 / 22.63 21.64 / 18.87, 25.06 / 22.49  18.36 / 17.48, 18.92 / 21.83
// So the line favours weights that are used again before they leave the cache, and costs products below it 5 to 12 %
// where they are not; above it, one product repeated on the same weights pays (64 rows: 22.1 / 28.5).
constexpr int KS_STREAM = 2;  // nt
constexpr double KS_STREAM_BYTES = 96.0 * 1024 * 1024;

// Rows of a tile.  What a unit can have under way is bounded by its L1, so a short tile fetches only the 8-row
// blocks that it has, and two row tiles take even shares of 65 to 96 rows instead of 64 and the rest: the launch
// ends with its longest workgroup.  us, weights of three or four sets in turn, 64-row tiles / this rule:
// [40, 1024] x [8192, 1024]^T 5.77 / 5.52, [40, 3584] 11.67 / 11.37, [40, 3696] 13.50 / 12.91, [33, 7168] 23.9 / 22.9,
// [48, 2048] x [6144, 2048]^T 7.41 / 7.18; [72, 768] x [6144, 768]^T 6.03 / 5.59, [72, 1024] x [8192, 1024]^T 7.05 /
// 6.64, [72, 3584] 13.53 / 12.52, [96, 1024] 7.14 / 6.93.  Even shares gain while the longest workgroup is the bound;
// where the L2s and the memory are, they lose: weights past KS_EVEN_BYTES ([80, 7168] 32.6 / 33.0, [72, 5120] 24.5 /
// 25.3), past 7/8 of it from 73 rows on ([80, 4096] 19.9 / 20.3, weights from memory; [72, 4096] 19.7 / 19.5), past
// half of it for 48-row tiles ([96, 3584] 13.4 / 13.6), or rows of b that are not whole lines ([80, 3696] 16.0 /
// 16.5; 48 rows there: 14.2 / 14.5).  56-row tiles are within 1 % either way and are not built.
//
// Under a grid cap workgroups walk several tiles and the longest one counts for less: from cold weights, 64-row tiles /
// even shares, cap 64: [72, 2048] x [8192, 2048]^T 35.5 / 34.9 us, [80, 2048] 35.9 / 36.0, but [80, 2560] 46.2 / 47.5,
// [80, 3072] 50.1 / 51.8, [80, 2560] x [6144, 2560]^T 41.1 / 41.8; cap 160: [80, 3584] 30.5 / 31.2.  So not past
// KS_EVEN_CAPPED_K there.
constexpr double KS_EVEN_BYTES = 64.0 * 1024 * 1024;
constexpr int64_t KS_EVEN_CAPPED_K = 2048;

// The instantiations: MT, NT, STAGES, LA, stream, tail.
#define TW_KSPLIT_ROWS_32(X, LA) \
  X(1, 1, 2, LA, true, false) X(1, 1, 2, LA, false, false) X(1, 1, 2, LA, false, true) \
  X(1, 1, 3, LA, true, false) X(1, 1, 3, LA, false, false)
#define TW_KSPLIT_FORMS(X)                                                                                   \
  TW_KSPLIT_ROWS_32(X, 1) TW_KSPLIT_ROWS_32(X, 2) TW_KSPLIT_ROWS_32(X, 4)                                      \
  X(1, 1, 3, 1, false, true) X(1, 1, 3, 2, false, true)                                                        \
  X(2, 1, 3, 5, true, false) X(2, 1, 3, 5, false, false) X(2, 1, 2, 5, false, true)                            \
  X(2, 1, 2, 6, true, false) X(2, 1, 2, 6, false, false)                                                       \
  X(2, 1, 2, 8, true, false) X(2, 1, 2, 8, false, false) X(2, 1, 2, 8, false, true)                            \
  X(2, 2, 2, 5, false, false) X(2, 2, 2, 6, false, false) X(2, 2, 2, 8, false, false) X(2, 2, 2, 8, false, true)
struct KsForm { int mt, nt, stages, la; bool stream, tail; };

// No form changes a result bit (see the kernel), so a product has the same bits under every grid cap and in every
// batch, although both are part of the rule.  Up to 32 columns a second column half would be empty LDS and idle
// MFMAs: 256 rows x 16 columns 4.6 -> 4.1 us at K = 128, 13.7 -> 9.5 at 4096.
//
// Up to 32 rows the third stage's 96 KiB leave a compute unit room for one workgroup, two stages for two.  So three
// stages only where no unit has a second tile; us, two / three stages, cold weights: [8, 1024] x [8192, 1024]^T
// 5.52 / 5.39, [32, 4096] x [4096, 4096]^T 10.9 / 10.4, but [32, 1024] x [16384, 1024]^T 9.0 / 10.1, x
// [28672, 1024]^T 14.7 / 17.8, eight products [32, 1024] x [8192, 1024]^T 27.0 / 34.0, [32, 128] 10.5 / 16.4.
// Nor past 16 rows where rows of b are not whole lines, two / three stages, cold weights: [24, 2000] x [8192, 2000]^T
// 9.8 / 10.2, [28, 2000] x [6144, 2000]^T 8.8 / 9.3, [17, 3696] x [8192, 3696]^T 14.7 / 15.2.
static KsForm ksplit_form(int64_t M, int64_t N, int64_t K, int count, int max_cus, int cus) {
  const double b_bytes = (double)count * N * K * 2;
  const bool whole = K % BK == 0, stream = whole && M <= 64 && b_bytes > KS_STREAM_BYTES;
  if (M <= 32) {
    const int la = M <= 8 ? 1 : M <= 16 ? 2 : 4;
    const KsTiles tiles = ksplit_tiles(M, N, count, 8 * la, 32, cus);
    const bool one_each = count * tiles.m * tiles.n <= (max_cus > 0 ? std::min(max_cus, cus) : cus);
    return {1, 1, one_each && (whole || M <= 16) ? 3 : 2, la, stream, !whole};
  }
  if (M <= 40) return {2, 1, whole ? 3 : 2, 5, stream, !whole};
  if (M <= 48 && whole) return {2, 1, 2, 6, stream, false};
  if (M <= 64 || N <= 32) return {2, 1, 2, 8, stream, !whole};
  const bool even = whole && (K <= KS_EVEN_CAPPED_K || max_cus <= 0 || max_cus >= cus);
  if (M <= 80 && even && b_bytes <= KS_EVEN_BYTES * (M <= 72 ? 1.0 : 0.875)) return {2, 2, 2, 5, false, false};
  if (M <= 96 && even && b_bytes < KS_EVEN_BYTES / 2) return {2, 2, 2, 6, false, false};
  return {2, 2, 2, 8, false, !whole};
}

static int launch_ksplit_for(const GemmBatch& batch, int count, int64_t M, int64_t N, int64_t K, int64_t ldc,
                             int max_cus, hipStream_t hs) {
  int cus = device_compute_units();
  if (cus <= 0) cus = 256;
  const KsForm f = ksplit_form(M, N, K, count, max_cus, cus);
#define TW_KSPLIT_LAUNCH(MT, NT, STAGES, LA, STREAM, TAIL)                                                     \
  if (f.mt == MT && f.nt == NT && f.stages == STAGES && f.la == LA && f.stream == STREAM && f.tail == TAIL)      \
    return launch_ksplit<MT, NT, STAGES, LA, STREAM ? KS_STREAM : 0, TAIL>(batch, count, M, N, K, ldc, max_cus, cus, \
                                                                           hs);
  TW_KSPLIT_FORMS(TW_KSPLIT_LAUNCH)
#undef TW_KSPLIT_LAUNCH
  return set_error(TW_ERR_INVALID_ARGUMENT, "gemm_bf16_nt: no kernel for %d rows", (int)M);
}

template <int TM, int TN, TileRows ROWS>
static int launch_tile_kernel(const GemmBatch& batch, int count, int64_t M, int64_t N, int64_t K, int64_t ldc,
                       int max_cus, hipStream_t hs) {
  using S = TileShape<TM, TN, ROWS>;
  static std::atomic<bool> lds_ok[kMaxDevices];
  if (int rc = allow_lds(reinterpret_cast<const void*>(gemm_bf16_nt_tile_kernel<TM, TN, ROWS>), lds_ok, kMaxDevices,
                         S::LDS))
    return rc;
  const int tiles_m = (int)((M + S::BM - 1) / S::BM), tiles_n = (int)((N + S::BN - 1) / S::BN);
  // a workgroup per compute unit at most: it fills the unit and walks its share of the tiles
  int cus = max_cus > 0 ? max_cus : device_compute_units();
  if (cus <= 0) cus = 256;
  const int64_t grid = std::min<int64_t>((int64_t)count * tiles_m * tiles_n, cus);
  // 16-byte stores need 16-byte aligned row segments that end inside the row
  int wide_store = (N % 8 == 0 && ldc % 8 == 0) ? 1 : 0;
  for (int p = 0; p < count; ++p)
    if (reinterpret_cast<uintptr_t>(batch.out[p]) & 15u) wide_store = 0;
  launch_kernel(gemm_bf16_nt_tile_kernel<TM, TN, ROWS>, dim3((unsigned)grid), dim3(TILE_THREADS), S::LDS, hs, batch,
                count, (int)M, (int)N, (int)K, ldc, tiles_m, tiles_n, wide_store);
  return TW_OK;
}

// Whole lines where the shape's ring has room for the panel more and rows are long: a tile costs 0.8 to 1 us more
// (one line more to fetch and every row's place in its lines).  us, kPartialSlab / kLines, 8192 columns, weights from
// memory: [200, 208] 6.1 / 6.9, [200, 528] 8.6 / 8.6, [200, 1040] 12.8 / 11.6, [200, 1552] 17.3 / 14.7; K a multiple
// of 32, where half as many rows lie on two lines: [200, 544] 8.2 / 8.7, [200, 1056] 11.9 / 11.6, [200, 2080] 19.6 /
// 17.7. The same weights again and again, from the last-level cache, gain later, and the lines are drawn between the
// two: [200, 1040] 10.7 / 10.8, [200, 1552] 13.7 / 13.3, [200, 2080] 15.5 / 15.9, [200, 4128] 28.0 / 26.5.  (What the
// L2s hold is not bound by requests: [129, 2064] x [1024, 2064]^T 11.5 / 14.9; from memory 19.9 / 16.7.)
constexpr int64_t LINES_FROM_K = 1280, LINES_FROM_K_32 = 2048;

// The shapes whose ring then is down to the least (TIGHT: 128 x 256 and 96 x 256) cover less of memory's latency and
// are taken only where more than half of the rows lie on two lines: K = 7392, 128 x 256, 800 and 1000 rows 122 / 138
// us with kPartialSlab, 132 / 133 with kLines.
template <int TM, int TN>
static TileRows tile_rows(int64_t K) {
  if (K % BK == 0) return kWholeSlabs;
  if constexpr (TileShape<TM, TN>::TAKES_LINES) {
    if (K % 32 == 16 && K >= LINES_FROM_K) return kLines;
    if (K % 32 == 0 && K >= LINES_FROM_K_32 && !TileShape<TM, TN, kLines>::TIGHT) return kLines;
  }
  return kPartialSlab;
}

template <int TM, int TN>
static int launch_tile(const GemmBatch& batch, int count, int64_t M, int64_t N, int64_t K, int64_t ldc,
                       int max_cus, hipStream_t hs) {
  const TileRows rows = tile_rows<TM, TN>(K);
  if (rows == kWholeSlabs) return launch_tile_kernel<TM, TN, kWholeSlabs>(batch, count, M, N, K, ldc, max_cus, hs);
  if constexpr (TileShape<TM, TN>::TAKES_LINES)
    if (rows == kLines) return launch_tile_kernel<TM, TN, kLines>(batch, count, M, N, K, ldc, max_cus, hs);
  return launch_tile_kernel<TM, TN, kPartialSlab>(batch, count, M, N, K, ldc, max_cus, hs);
}

// The tile shapes, in 32-row and 32-column units, with the time a round of them takes on all
// compute units relative to 256 x 256 tiles, measured at K = 3584 with one tile per unit.  The
// heights and widths are there to make a tile count fit the units: 192 x 256 (M = 1500), 160 x 256
// (M = 2458: 512 tiles) and the 192-wide ones for N = 6144, whose 24 columns of 256 leave a quarter
// of the units idle; the small ones for M <= 512 at N = 8192 (64 x 128, 96 x 128, 128 x 128: 256
// tiles for 256, 384 and 512 rows).
// One column of costs serves every K and every way of fetching rows: of the twelve shapes timed one by one, the
// picked one is the fastest at 112 of 120 points (15 row counts from 129 to 4096; 8192 columns with K = 1024, 2048,
// 3584, 3696, 7168, 7392 and 6144 columns with K = 768, 2048; three sets of operands in turn), 0.3 % from it on
// average and 15 % at worst (640 rows, 6144 columns, K = 768: 11.7 us, 96 x 192 tiles 10.2); with weights from memory
// at 115 points, 0.1 % from it on average and 5 % at worst (2458 rows there: 29.6 us, 192 x 192 tiles 28.3).  At
// K = 3696 and 7392 it misses at two: 800 rows from memory 70.7 us (128 x 128 tiles 67.9), 1000 rows 138 (160 x 256
// 133).
struct TileChoice { int tm, tn; double cost; };
#define TW_TILES(X)                                                                                            \
  X(8, 8, 1.0) X(6, 8, 0.79) X(8, 6, 0.77) X(5, 8, 0.69) X(6, 6, 0.65) X(4, 8, 0.58) X(3, 8, 0.48) X(4, 6, 0.46) \
  X(3, 6, 0.41) X(4, 4, 0.365) X(3, 4, 0.315) X(2, 4, 0.25)
#define TW_TILE_CHOICE(TM, TN, COST) {TM, TN, COST},
constexpr TileChoice kTiles[] = {TW_TILES(TW_TILE_CHOICE)};
#undef TW_TILE_CHOICE

static int launch_tile_shape(int tm, int tn, const GemmBatch& batch, int count, int64_t M, int64_t N, int64_t K,
                             int64_t ldc, int max_cus, hipStream_t hs) {
#define TW_TILE_LAUNCH(TM, TN, COST) \
  if (tm == TM && tn == TN) return launch_tile<TM, TN>(batch, count, M, N, K, ldc, max_cus, hs);
  TW_TILES(TW_TILE_LAUNCH)
#undef TW_TILE_LAUNCH
  return set_error(TW_ERR_INVALID_ARGUMENT, "gemm_bf16_nt: no %d x %d tile", 32 * tm, 32 * tn);
}

// The shape whose rounds over the available units take the least time; ties go to the earlier
// (larger) one.  The shape never changes a result bit: every output element is the same sequence
// of MFMA k-steps whatever tile it lies in.
static const TileChoice& pick_tile(int64_t M, int64_t N, int count, int cus) {
  const TileChoice* best = &kTiles[0];
  double best_cost = 1e300;
  for (const TileChoice& t : kTiles) {
    const int64_t tiles = count * ((M + 32 * t.tm - 1) / (32 * t.tm)) * ((N + 32 * t.tn - 1) / (32 * t.tn));
    const double cost = (double)((tiles + cus - 1) / cus) * t.cost;
    if (cost < best_cost) {
      best_cost = cost;
      best = &t;
    }
  }
  return *best;
}

// Which of the two families runs is decided by M, N and K alone (their sums differ in the order of
// the additions): a product has the same bits under every grid cap and in every batch.
static bool tile_kernel_fits(int64_t M, int64_t N, int64_t K, int64_t ldc) {
  return K <= TILE_MAX_K && ldc <= TILE_MAX_LDC && M > 128 && N >= 64;
}

static int launch_tile_for(const GemmBatch& batch, int count, int64_t M, int64_t N, int64_t K, int64_t ldc,
                           int max_cus, hipStream_t hs) {
  int cus = max_cus > 0 ? max_cus : device_compute_units();
  if (cus <= 0) cus = 256;
  const TileChoice& t = pick_tile(M, N, count, cus);
  return launch_tile_shape(t.tm, t.tn, batch, count, M, N, K, ldc, max_cus, hs);
}

static int check_gemm_shape(const char* what, int64_t M, int64_t N, int64_t K, int64_t ldc) {
  if (M < 0 || N <= 0 || K <= 0 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX || ldc < N)
    return set_error(TW_ERR_INVALID_ARGUMENT, "%s: bad shape M=%lld N=%lld K=%lld ldc=%lld", what, (long long)M,
                     (long long)N, (long long)K, (long long)ldc);
  if (K % 8 != 0 || N % 4 != 0 || ldc % 4 != 0)
    return set_error(TW_ERR_ALIGNMENT, "%s: needs K %% 8 == 0, N %% 4 == 0, ldc %% 4 == 0", what);
  return TW_OK;
}

static int check_gemm_pointers(const char* what, const void* out, const void* a, const void* b,
                               const void* bias) {
  if (!out || !a || !b) return set_error(TW_ERR_INVALID_ARGUMENT, "%s: null pointer argument", what);
  auto al = [](const void* p, unsigned n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; };
  if (!al(a, 16) || !al(b, 16) || !al(out, 8) || !al(bias, 8))
    return set_error(TW_ERR_ALIGNMENT, "%s: needs 16-byte aligned a and b, 8-byte aligned out and bias", what);
  return TW_OK;
}

static int run_products(const char* what, const GemmBatch& batch, int count, int64_t M, int64_t N, int64_t K,
                        int64_t ldc, int max_cus, hipStream_t hs) {
  if (tile_kernel_fits(M, N, K, ldc)) {
    if (int rc = launch_tile_for(batch, count, M, N, K, ldc, max_cus, hs)) return rc;
    return finish_launch(what);
  }
  if (K <= KS_MAX_K) {
    if (int rc = launch_ksplit_for(batch, count, M, N, K, ldc, max_cus, hs)) return rc;
    return finish_launch(what);
  }
  const int tiles_m = (int)((M + BM - 1) / BM), tiles_n = (int)((N + BN - 1) / BN);
  int64_t grid = (int64_t)tiles_m * tiles_n;
  if (max_cus > 0 && grid > max_cus) grid = max_cus;
  if (grid > INT32_MAX) grid = INT32_MAX;
  for (int p = 0; p < count; ++p) {
    launch_kernel(gemm_bf16_nt_kernel, dim3((unsigned)grid), dim3(GEMM_THREADS), 0, hs, batch.out[p], batch.a[p],
                  batch.b[p], batch.bias[p], (int)M, (int)N, (int)K, ldc, tiles_m, tiles_n);
    if (int rc = finish_launch(what)) return rc;
  }
  return TW_OK;
}

int run_gemm_bf16_nt(void* out, const void* a, const void* b, const void* bias, int64_t M, int64_t N,
                     int64_t K, int64_t ldc, int max_cus, void* stream) {
  if (int rc = check_gemm_shape("gemm_bf16_nt", M, N, K, ldc)) return rc;
  if (M == 0) return TW_OK;
  if (int rc = check_gemm_pointers("gemm_bf16_nt", out, a, b, bias)) return rc;
  GemmBatch batch = {};
  batch.out[0] = static_cast<uint16_t*>(out);
  batch.a[0] = static_cast<const uint16_t*>(a);
  batch.b[0] = static_cast<const uint16_t*>(b);
  batch.bias[0] = static_cast<const uint16_t*>(bias);
  return run_products("gemm_bf16_nt", batch, 1, M, N, K, ldc, max_cus, static_cast<hipStream_t>(stream));
}

// outs[p][M, N] (row stride ldc) = as[p][M, K] * bs[p][N, K]^T (+ biases[p] when `biases` and
// that entry are non-null) for p < count, in one launch over count x tiles.
int run_gemm_bf16_nt_partials(void* const* outs, const void* const* as, const void* const* bs,
                              const void* const* biases, int count, int64_t M, int64_t N, int64_t K,
                              int64_t ldc, int max_cus, void* stream) {
  const char* what = "gemm_bf16_nt_partials";
  if (count < 1 || count > TW_MAX_PARTIALS)
    return set_error(TW_ERR_INVALID_ARGUMENT, "%s: number of partials %d not in [1, %d]", what, count,
                     TW_MAX_PARTIALS);
  if (int rc = check_gemm_shape(what, M, N, K, ldc)) return rc;
  if (M == 0) return TW_OK;
  if (!outs || !as || !bs) return set_error(TW_ERR_INVALID_ARGUMENT, "%s: null pointer argument", what);
  GemmBatch batch = {};
  for (int p = 0; p < count; ++p) {
    const void* bias = biases ? biases[p] : nullptr;
    if (int rc = check_gemm_pointers(what, outs[p], as[p], bs[p], bias)) return rc;
    batch.bias[p] = static_cast<const uint16_t*>(bias);
    batch.out[p] = static_cast<uint16_t*>(outs[p]);
    batch.a[p] = static_cast<const uint16_t*>(as[p]);
    batch.b[p] = static_cast<const uint16_t*>(bs[p]);
  }
  return run_products(what, batch, count, M, N, K, ldc, max_cus, static_cast<hipStream_t>(stream));
}

}  // namespace tw
