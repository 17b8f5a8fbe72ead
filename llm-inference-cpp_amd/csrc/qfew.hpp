// The exact product for 2..8 input rows on the matrix cores: one 64-row tile
// of the matrix times up to R (4 or 8) input rows.
//
// v_mfma_f32_4x4x1_16b_f32 holds sixteen 4 x 4 outer products: D[i][lane] =
// fma(A[i], B[lane], C[i][lane]), one IEEE fused multiply-add per result
// (checked bit for bit, as for qrows.hip), where lane l of B belongs to
// block l / 4.  With lane l carrying output row l's code -- the tiled
// layout's own order -- and the A operand broadcast from one block to all
// (cbsz = 4, abid = the block), one instruction advances the reference's
// chain part = fma(x[k], code[k], part) of 64 outputs x 4 input rows by one
// element.  Lane 4a + i of an A register holds x[i][2a + j], so two
// registers feed the 32 steps of a block, and a row's 32 activations are one
// coalesced 128-byte load.
//
// Bound: HBM for the weights at 4 rows; at 8 rows the fp32 units, in part (per
// block of 64 outputs 64 matrix instructions of 4.2 ns and, for Q4_0, 60
// decoding instructions of 1.2 to 1.9: 17 and 5 to 7 of the 33.6 us of
// SmolLM2's 211 products; the other 10 are the barrier, the LDS exchange and
// the loads -- of the wavefronts' time 60 % waits to issue and 28 % at a wait
// or barrier).  The W wavefronts take a tile's blocks in
// turn, one per iteration, loaded kAhead iterations earlier; an iteration's
// block sums and scales meet in one of two LDS buffers, and after its
// barrier wavefront w advances the chains of rows w, w + W, ... over the W
// blocks in order.  Two small buffers instead of a whole row's sums let six
// wavefronts share a SIMD, so one workgroup's barriers run under another's
// arithmetic, and rows of any length take 8 input rows per pass over the
// weights.  Measured, before on the vector ALUs -> here: 151936 x 896 at 8
// rows Q8_0 78.2 -> 36.7 us (4.3 TB/s), Q4_0 51.9 -> 33.5; SmolLM2's 211
// products at batch 8 in one launch, Q4_0, 81.9 -> 33.6 us (decoding a word's
// codes apart from its matrix instructions, to save their wait states, 41.1;
// a whole row's sums in LDS, as batch 1 keeps them, 46.9).
#pragma once

#include <type_traits>

#include "qblock.hpp"

namespace llmi_hip {
namespace few {

constexpr int kAhead = 2;  // iterations a block is loaded ahead

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef std::uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Codes 8j .. 8j + 7 of a block as fp32.  Q4_0: the nibbles of a word as
// signed bytes n - 8 (n + 0x78 never carries out of its byte), then
// converted by byte like Q8_0's.
template <int TYPE>
__device__ __forceinline__ void eight_codes(const Block<TYPE>& b, int j, float* c) {
  if (TYPE == LLMI_TYPE_Q8_0) {
    const uint4 v = b.c[Block<TYPE>::kU == 2 ? j >> 1 : 0];
    const std::uint32_t w[2] = {j & 1 ? v.z : v.x, j & 1 ? v.w : v.y};
#pragma unroll
    for (int e = 0; e < 8; ++e) c[e] = static_cast<float>(static_cast<std::int8_t>(w[e >> 2] >> (8 * (e & 3))));
  } else {
    const std::uint32_t w = j == 0 ? b.c[0].x : j == 1 ? b.c[0].y : j == 2 ? b.c[0].z : b.c[0].w;
    const std::uint32_t lo = ((w & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u;
    const std::uint32_t hi = (((w >> 4) & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      c[e] = static_cast<float>(static_cast<std::int8_t>((e & 1 ? hi : lo) >> (8 * (e >> 1))));
  }
}

template <int K, int H>
__device__ __forceinline__ void step(const float (&xa)[H][2], float code, f32x4 (&part)[H]) {
#pragma unroll
  for (int h = 0; h < H; ++h)
    part[h] = __builtin_amdgcn_mfma_f32_4x4x1f32(xa[h][K & 1], code, part[h], 4, K >> 1, 0);
}

// Rows [0, nr) (nr <= R; row r at x + r * in, results at y + r * out) of one
// tile; the workgroup's W wavefronts all call it.
template <int TYPE, int R, int W>
__device__ __forceinline__ void tile(const GMEM uint4* __restrict__ codes, const GMEM float* __restrict__ scales,
                                     const GMEM float* __restrict__ x, const GMEM float* __restrict__ bias,
                                     GMEM float* __restrict__ y, int in, int nblk, int out, int nr, int accumulate,
                                     std::size_t tile_index) {
  constexpr int H = R / 4;
  constexpr int RW = R > W ? R / W : 1;  // chain rows per wavefront
  __shared__ float ps[2][W][R][kTileRows];
  __shared__ float ss[2][W][kTileRows];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const std::size_t base = tile_index * nblk;
  const int nfull = in / kBlock;
  // The lane's elements 2 (lane / 4), + 1 of rows lane % 4 (+ 4); rows past
  // nr are row nr - 1 again and never stored.  Read through a buffer of the
  // nr rows: past the last row's end it returns zero, and what a partial
  // block reads of the row after is zeroed before use.
  const auto xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>((const float*)x), 0, 4 * nr * in, 0x00020000);
  int xo[H];
#pragma unroll
  for (int h = 0; h < H; ++h) xo[h] = 4 * (min(4 * h + (lane & 3), nr - 1) * in + 2 * (lane >> 2));
  struct Raw {
    u32x2 x[H];
    Block<TYPE> blk;
    float sc;
  };
  // Loads are unconditional, of the last block again past the end (an
  // iteration whose loads depend on a condition makes every later wait a
  // full one); the activations first: loads complete in order, and they come
  // from the caches, the weights from HBM.
  const auto load = [&](Raw& r, int b) {
    b = min(b, nblk - 1);
#pragma unroll
    for (int h = 0; h < H; ++h) r.x[h] = __builtin_amdgcn_raw_buffer_load_b64(xbuf, xo[h], b * (kBlock * 4), 0);
    r.blk = load_block<TYPE, true>(codes, base + b, lane);
    r.sc = loadf<true>(scales + (base + b) * kTileRows + lane);
  };
  float acc[RW];
#pragma unroll
  for (int i = 0; i < RW; ++i) acc[i] = 0.0f;
  const int niter = (nblk + W - 1) / W;
  const auto iteration = [&](int it, auto buf_tag, Raw& r) {
    constexpr int buf = decltype(buf_tag)::value;
    const int b = it * W + wave;
    if (b < nblk) {  // (uniform)
      float xa[H][2];
#pragma unroll
      for (int h = 0; h < H; ++h) {
        xa[h][0] = __uint_as_float(r.x[h][0]);
        xa[h][1] = __uint_as_float(r.x[h][1]);
      }
      if (b >= nfull) {  // activations past `in` are zero: the codes stored there add nothing
        const int left = in - b * kBlock - 2 * (lane >> 2);
#pragma unroll
        for (int h = 0; h < H; ++h) {
          xa[h][0] = left > 0 ? xa[h][0] : 0.0f;
          xa[h][1] = left > 1 ? xa[h][1] : 0.0f;
        }
      }
      f32x4 part[H];
#pragma unroll
      for (int h = 0; h < H; ++h) part[h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#define LLMI_FEW_EIGHT(j)                 \
  {                                       \
    float c[8];                           \
    eight_codes<TYPE>(r.blk, j, c);       \
    step<8 * j + 0, H>(xa, c[0], part);  \
    step<8 * j + 1, H>(xa, c[1], part);   \
    step<8 * j + 2, H>(xa, c[2], part);   \
    step<8 * j + 3, H>(xa, c[3], part);   \
    step<8 * j + 4, H>(xa, c[4], part);   \
    step<8 * j + 5, H>(xa, c[5], part);   \
    step<8 * j + 6, H>(xa, c[6], part);   \
    step<8 * j + 7, H>(xa, c[7], part);   \
  }
      LLMI_FEW_EIGHT(0)
      LLMI_FEW_EIGHT(1)
      LLMI_FEW_EIGHT(2)
      LLMI_FEW_EIGHT(3)
#undef LLMI_FEW_EIGHT
#pragma unroll
      for (int i = 0; i < R; ++i) ps[buf][wave][i][lane] = part[i >> 2][i & 3];
      ss[buf][wave][lane] = r.sc;
    }
    load(r, b + kAhead * W);
    __syncthreads();
    if (R >= W || wave < R) {
      const int end = min(W, nblk - it * W);
      float sv[W], pv[RW][W];
#pragma unroll
      for (int k = 0; k < W; ++k) {  // (blocks past the end: read, not used)
        sv[k] = ss[buf][k][lane];
#pragma unroll
        for (int i = 0; i < RW; ++i) pv[i][k] = ps[buf][k][wave + i * W][lane];
      }
#pragma unroll
      for (int k = 0; k < W; ++k)
        if (k < end) {
#pragma unroll
          for (int i = 0; i < RW; ++i) acc[i] = __builtin_fmaf(pv[i][k], sv[k], acc[i]);
        }
    }
  };
  static_assert(kAhead == 2, "two register sets in turn");
  Raw ra, rb;
  load(ra, wave);
  load(rb, wave + W);
  int it = 0;
  for (; it + 2 <= niter; it += 2) {
    iteration(it, std::integral_constant<int, 0>{}, ra);
    iteration(it + 1, std::integral_constant<int, 1>{}, rb);
  }
  if (it < niter) iteration(it, std::integral_constant<int, 0>{}, ra);
  const std::size_t o = tile_index * kTileRows + lane;
  if (o >= static_cast<std::size_t>(out)) return;
  const float add = bias != nullptr ? bias[o] : 0.0f;
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int r = wave + i * W;
    if (r < nr) {
      GMEM float* dst = y + static_cast<std::size_t>(r) * out + o;
      const float v = acc[i] + add;
      *dst = accumulate ? *dst + v : v;
    }
  }
}

}  // namespace few
}  // namespace llmi_hip
