// Quantized matrix-vector / small-batch product for gfx950.
//
// Reference: src/model/quant.cpp:119-153.  For each output o and input row r
// the reference computes, with the compiler's fused multiply-adds,
//     part_b = fma(x[k], code[k], part_b)   over the block's elements in order
//     acc    = fma(part_b, scale_b, acc)    over the blocks in order
//     y      = acc + bias[o]                (bias 0.0f when absent)
// These kernels perform exactly those operations, so y is bit-identical.
//
// All kernels read the tiled layout (common.hpp): lane l of a wavefront owns
// output row tile*64 + l, so one block of 64 rows is a single coalesced
// 16-byte load per lane (two for Q8_0), and the activations x[k] are the
// same for every lane -- they are read with scalar loads into SGPRs and
// broadcast to the fused multiply-adds.  Every code byte and scale is read
// from HBM once; the kernels are HBM-bound at batch 1.
//
// qgemv_tile (batch 1; 2..8 rows by few_chunk and few_kind): one workgroup
// per (64-row tile, chunk of up to R input rows).  Its W wavefronts split the
// tile's blocks into contiguous ranges; each decodes a block once and forms
// the block sums of every input row of the chunk, which it parks in LDS
// together with the block scales.  After one barrier the wavefronts run the
// sequential chains over all blocks (one chain per input row), add the bias
// and store y.  Splitting the blocks over wavefronts is what fills the GPU
// when a matrix has few tiles.
//
// qgemv_few (2..8 rows): a 64-row tile on the matrix cores (qfew.hpp).
//
// qgemv_narrow (batch 1, matrices with few rows): 16-row tiles, 4x the
// workgroups of qgemv_tile.
//
// qgemv_group, qgemv_group_few: a fixed list of products (each batch 1..8)
// launched together (one kernel per kind of tile present); each workgroup
// runs one tile of one product with the same tile functions.
//
// Batch > 8, and few rows on few tiles, take the multi-row product
// (qrows.hip).
//
// fp32 weights take kernels::matmul instead (f32.hip).
#include <algorithm>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "glue_math.hpp"
#include "qblock.hpp"
#include "qfew.hpp"

namespace llmi_hip {

namespace {

// Q4_0 decode constants, kept in VGPRs (v_and_or_b32 takes no literal).
// Two 4-bit codes n (element value n - 8) are moved into the mantissas of an
// f16 pair whose exponent makes the pair (1024 + n) (nibble at bits 0-3 of a
// half) or (64 + n) (bits 4-7); one packed f16 subtraction of 1032 or 72
// then gives n - 8 exactly, and v_fma_mix_f32 takes the f16 operand into an
// fp32 fused multiply-add with no separate conversion.  The products and
// sums are the same fp32 operations as with an fp32 code operand.
struct Q4Magic {
  std::uint32_t lo_mask, hi_mask, lo_exp, hi_exp;
};
__device__ __forceinline__ Q4Magic q4_magic() {
  Q4Magic k{0x000F000Fu, 0x00F000F0u, 0x64006400u, 0x54005400u};
  asm("" : "+v"(k.lo_mask), "+v"(k.hi_mask), "+v"(k.lo_exp), "+v"(k.hi_exp));
  return k;
}
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ half2_t f16_pair(std::uint32_t w, std::uint32_t mask, std::uint32_t exp_bits) {
  std::uint32_t d;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(d) : "v"(w), "v"(mask), "v"(exp_bits));
  return __builtin_bit_cast(half2_t, d);
}

// Block sum of one full block: part = fma(x[i], code[i], part), i = 0..31;
// XP points to the block's 32 activations (global memory or LDS).  For one
// input row Q4_0 codes go to v_fma_mix_f32 as f16 pairs; the multi-row
// kernels instead convert each code to fp32 once (block_codes) and use it in
// R v_fmac_f32, which issue at twice the rate of the mixed-precision FMA on
// gfx950.
template <int TYPE, typename XP>
__device__ __forceinline__ float full_block_dot(const Block<TYPE>& b, XP __restrict__ xr, const Q4Magic& k) {
  float part = 0.0f;
  if (TYPE == LLMI_TYPE_Q8_0) {
    const std::uint32_t w[8] = {b.c[0].x, b.c[0].y, b.c[0].z, b.c[0].w, b.c[Block<TYPE>::kU - 1].x,
                                b.c[Block<TYPE>::kU - 1].y, b.c[Block<TYPE>::kU - 1].z, b.c[Block<TYPE>::kU - 1].w};
#pragma unroll
    for (int i = 0; i < kBlock; ++i) part = __builtin_fmaf(xr[i], code_of<TYPE>(w, i), part);
    return part;
  }
  // Word j holds elements 8j..8j+7 as nibbles 0..7 (element 8j+2m in the low
  // nibble of byte m, 8j+2m+1 in the high nibble).
  const half2_t lo_off = {static_cast<_Float16>(-1032.0f), static_cast<_Float16>(-1032.0f)};
  const half2_t hi_off = {static_cast<_Float16>(-72.0f), static_cast<_Float16>(-72.0f)};
  const std::uint32_t w[4] = {b.c[0].x, b.c[0].y, b.c[0].z, b.c[0].w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const std::uint32_t s = w[j] >> 8;
    const half2_t e04 = f16_pair(w[j], k.lo_mask, k.lo_exp) + lo_off;  // elements 0, 4 of the word
    const half2_t e15 = f16_pair(w[j], k.hi_mask, k.hi_exp) + hi_off;  // 1, 5
    const half2_t e26 = f16_pair(s, k.lo_mask, k.lo_exp) + lo_off;     // 2, 6
    const half2_t e37 = f16_pair(s, k.hi_mask, k.hi_exp) + hi_off;     // 3, 7
    const XP xj = xr + 8 * j;
    part = __builtin_fmaf(xj[0], static_cast<float>(e04.x), part);
    part = __builtin_fmaf(xj[1], static_cast<float>(e15.x), part);
    part = __builtin_fmaf(xj[2], static_cast<float>(e26.x), part);
    part = __builtin_fmaf(xj[3], static_cast<float>(e37.x), part);
    part = __builtin_fmaf(xj[4], static_cast<float>(e04.y), part);
    part = __builtin_fmaf(xj[5], static_cast<float>(e15.y), part);
    part = __builtin_fmaf(xj[6], static_cast<float>(e26.y), part);
    part = __builtin_fmaf(xj[7], static_cast<float>(e37.y), part);
  }
  return part;
}

// The 32 codes of a full block as fp32 (for the multi-row kernels).
template <int TYPE>
__device__ __forceinline__ void block_codes(const Block<TYPE>& b, float* c) {
  std::uint32_t w[8];
  unpack_words<TYPE>(b, w);
#pragma unroll
  for (int i = 0; i < kBlock; ++i) c[i] = code_of<TYPE>(w, i);
}

template <typename XP>
__device__ __forceinline__ float codes_dot(const float* c, XP __restrict__ xr) {
  float part = 0.0f;
#pragma unroll
  for (int i = 0; i < kBlock; ++i) part = __builtin_fmaf(xr[i], c[i], part);
  return part;
}

// Block sum of the final partial block (len < 32 elements).
template <int TYPE, typename XP>
__device__ __noinline__ float tail_block_dot(const Block<TYPE> blk, XP __restrict__ xr, int len) {
  std::uint32_t w[8];
  unpack_words<TYPE>(blk, w);
  float part = 0.0f;
#pragma unroll
  for (int i = 0; i < kBlock; ++i)
    if (i < len) part = __builtin_fmaf(xr[i], code_of<TYPE>(w, i), part);
  return part;
}

// Block sum of a block whose activation i is in lane i of v.  Not inlined, so
// that the partial block costs the loop over the whole ones no registers
// (SmolLM2's 211 Q4_0 products at batch 1 17.21 us inlined, 17.04 so).
template <int TYPE>
__device__ __noinline__ float lanes_dot(const Block<TYPE> blk, float v) {
  float c[kBlock];
  block_codes<TYPE>(blk, c);
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < kBlock; ++i) sum = __builtin_fmaf(readlane_f32(v, i), c[i], sum);
  return sum;
}

// Block sums of blocks [b_begin, b_end) of one tile for input rows [0, nr)
// (nr <= R; row r starts at x + r*in) into part[(r*nblk + b)*64 + lane], and
// the blocks' scales into scl[b*64 + lane].  Loads run CH blocks ahead.
template <int TYPE, int R, int CH>
__device__ __forceinline__ void block_sums(const GMEM uint4* __restrict__ codes, const GMEM float* __restrict__ scales,
                                           const GMEM float* __restrict__ x, std::size_t tile, int in, int nblk, int nr,
                                           int b_begin, int b_end, int lane, float* part, float* scl) {
  const Q4Magic k = q4_magic();
  const int nfull = in / kBlock;
  const int f_end = min(b_end, nfull);
  const std::size_t base = tile * nblk;
  Block<TYPE> cur[CH];
  float cur_s[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    if (b_begin + j < f_end) {
      cur[j] = load_block<TYPE, true>(codes, base + b_begin + j, lane);
      cur_s[j] = loadf<true>(scales + (base + b_begin + j) * kTileRows + lane);
    }
  }
  for (int b = b_begin; b < f_end; b += CH) {
    Block<TYPE> nxt[CH];
    float nxt_s[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      if (b + CH + j < f_end) {
        nxt[j] = load_block<TYPE, true>(codes, base + b + CH + j, lane);
        nxt_s[j] = loadf<true>(scales + (base + b + CH + j) * kTileRows + lane);
      }
    }
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      if (b + j < f_end) {
        if (R == 1) {
          part[(b + j) * kTileRows + lane] = full_block_dot<TYPE>(cur[j], x + (b + j) * kBlock, k);
        } else {
          float c[kBlock];
          block_codes<TYPE>(cur[j], c);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            if (r < nr)
              part[(r * nblk + b + j) * kTileRows + lane] =
                  codes_dot(c, x + static_cast<std::size_t>(r) * in + (b + j) * kBlock);
          }
        }
        scl[(b + j) * kTileRows + lane] = cur_s[j];
      }
    }
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      cur[j] = nxt[j];
      cur_s[j] = nxt_s[j];
    }
  }
  if (nfull < nblk && nfull >= b_begin && nfull < b_end) {
    // The partial block, its loads issued together.  Lane i carries element i
    // of each row, broadcast by v_readlane; past `in` it is +0, which leaves
    // the chain as it is (its sums are never -0).  Loading element by element
    // in the chain took 2 us a row (6000 x 1087 at 5 rows 13 -> 8 us).
    const int len = in - nfull * kBlock, e = lane & (kBlock - 1);
    const GMEM float* xt = x + nfull * kBlock + min(e, len - 1);
    float xv[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (r < nr) xv[r] = xt[static_cast<std::size_t>(r) * in];
    const Block<TYPE> blk = load_block<TYPE, true>(codes, base + nfull, lane);
    scl[nfull * kTileRows + lane] = loadf<true>(scales + (base + nfull) * kTileRows + lane);
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (r < nr) part[(r * nblk + nfull) * kTileRows + lane] = lanes_dot<TYPE>(blk, e < len ? xv[r] : 0.0f);
  }
}

// The sequential chain over all blocks of one row of a tile, from LDS
// (stride `stride` floats between blocks).  Two register sets of
// kChainRound blocks: the reads of one are issued before the fused
// multiply-adds of the other, so LDS latency overlaps the chain.  The reads
// walk two pointers with constant offsets (an index clamped to the last
// block puts the next address in a register an outstanding read still
// targets, and every round then waits for all reads in flight).  A round's
// look-ahead may read up to kChainRound blocks past the row: inside the
// next row or the scales, or in the padding wide_lds adds after them; those
// values are never used.
constexpr int kChainRound = 4;
__device__ __forceinline__ float chain_lds(const float* part, const float* scl, int nblk, int lane, int stride) {
  const float* pp = part + lane;
  const float* sp = scl + lane;
  float pa[kChainRound], sa[kChainRound], pb[kChainRound], sb[kChainRound];
  const auto read = [&](float* p, float* q, const float* ps, const float* ss) {
#pragma unroll
    for (int u = 0; u < kChainRound; ++u) {
      p[u] = ps[u * stride];
      q[u] = ss[u * stride];
    }
  };
  float acc = 0.0f;
  const auto steps = [&](const float* p, const float* q) {
#pragma unroll
    for (int u = 0; u < kChainRound; ++u) acc = __builtin_fmaf(p[u], q[u], acc);
  };
  read(pa, sa, pp, sp);
  int b = 0;
  for (; b + 2 * kChainRound <= nblk; b += 2 * kChainRound) {
    read(pb, sb, pp + kChainRound * stride, sp + kChainRound * stride);
    __builtin_amdgcn_sched_barrier(0);
    steps(pa, sa);
    read(pa, sa, pp + 2 * kChainRound * stride, sp + 2 * kChainRound * stride);
    __builtin_amdgcn_sched_barrier(0);
    steps(pb, sb);
    pp += 2 * kChainRound * stride;
    sp += 2 * kChainRound * stride;
  }
  // pa holds blocks b .. b + 3 (those below nblk); the rest one by one.
#pragma unroll
  for (int u = 0; u < kChainRound; ++u)
    if (b + u < nblk) acc = __builtin_fmaf(pa[u], sa[u], acc);
  for (int c = b + kChainRound; c < nblk; ++c) acc = __builtin_fmaf(part[c * stride + lane], scl[c * stride + lane], acc);
  return acc;
}

__device__ __forceinline__ void store_out(GMEM float* __restrict__ y, std::size_t o, float v, int accumulate) {
  y[o] = accumulate ? y[o] + v : v;
}

// Load chunk (blocks in flight per wavefront) of the 64-row tile kernels,
// from launch-shape sweeps on MI355X: Q4_0 takes up to 4 blocks (one 16-byte
// load each), Q8_0 one block (two loads).
template <int TYPE>
constexpr int wide_chunk() {
  return TYPE == LLMI_TYPE_Q8_0 ? 1 : 4;
}

// One 64-row tile for input rows [0, nr), nr <= R (x, y already point at the
// chunk's first row).  The workgroup's wavefronts split the blocks, bpw
// each, and park block sums and scales in LDS (part[nr][nblk][64] then
// scale[nblk][64]); wavefront w then runs the chains of rows w, w + W, ...
// Every thread of the workgroup must call it (it has a barrier).
template <int TYPE, int R>
__device__ __forceinline__ void wide_tile(const GMEM uint4* __restrict__ codes, const GMEM float* __restrict__ scales,
                                          const GMEM float* __restrict__ x, const GMEM float* __restrict__ bias,
                                          GMEM float* __restrict__ y, int in, int nblk, int out, int nr, int bpw,
                                          int accumulate, std::size_t tile, float* lds) {
  float* part = lds;
  float* scl = lds + static_cast<std::size_t>(nr) * nblk * kTileRows;
  const int lane = threadIdx.x & (kTileRows - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nwaves = blockDim.x >> 6;
  const int b_begin = wave * bpw;
  const int b_end = min(nblk, b_begin + bpw);
  block_sums<TYPE, R, wide_chunk<TYPE>()>(codes, scales, x, tile, in, nblk, nr, b_begin, b_end, lane, part, scl);
  __syncthreads();
  const std::size_t o = tile * kTileRows + lane;
  for (int r = wave; r < nr; r += nwaves) {
    const float acc = chain_lds(part + static_cast<std::size_t>(r) * nblk * kTileRows, scl, nblk, lane, kTileRows);
    if (o < static_cast<std::size_t>(out))
      store_out(y + static_cast<std::size_t>(r) * out, o, acc + (bias != nullptr ? bias[o] : 0.0f), accumulate);
  }
}

// Stages the activations of a 16-row tile in LDS, applying the prologue
// (see kPlain, kRmsNorm, kSiluUp).  Every thread of the workgroup calls it;
// it ends with a barrier.
// Elements each thread loads per round of stage_x: a round's loads are all
// issued before the first one is used, so a row of `in` activations costs
// one memory round trip while in <= kStageBatch * blockDim.x.
constexpr int kStageBatch = 8;

__device__ __forceinline__ void stage_x(const GMEM float* __restrict__ x, int in, int prologue,
                                        const GMEM float* __restrict__ pw, float eps, float* xs) {
  __shared__ double red[64];
  __shared__ std::uint64_t tab[32];
  const int tid = threadIdx.x, nthreads = blockDim.x;

  const bool one_round = in <= nthreads * kStageBatch;
  float v[kStageBatch], w[kStageBatch];
  double part = 0.0;
  const auto round = [&](int i0) {
#pragma unroll
    for (int u = 0; u < kStageBatch; ++u) {
      const int i = i0 + u * nthreads + tid;
      v[u] = i < in ? x[i] : 0.0f;
      w[u] = prologue != kPlain && i < in ? pw[i] : 0.0f;
    }
    if (prologue == kSiluUp && i0 == 0) {
      if (tid < 32) tab[tid] = exact::kExp2Tab[tid];
      __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < kStageBatch; ++u) {
      const int i = i0 + u * nthreads + tid;
      if (i < in) {
        if (prologue == kSiluUp) {
          xs[i] = silu_exact(v[u], tab) * w[u];
        } else {
          xs[i] = v[u];
          const double d = static_cast<double>(v[u]);
          part = __builtin_fma(d, d, part);
        }
      }
    }
  };
  // The first round outside the loop: a loop header makes the compiler wait
  // for every load in flight (the caller's weight loads, issued just
  // before), which would put the activations' round trip after theirs.
  round(0);
  for (int i0 = nthreads * kStageBatch; i0 < in; i0 += nthreads * kStageBatch) round(i0);
  if (prologue != kRmsNorm) {
    __syncthreads();
    return;
  }
  // RMSNorm: the double sum of squares in any order, taken when the error
  // bound proves the reference's sequential sum gives the same float scale
  // (else summed sequentially), then y = w * (x * scale).
  part = row_sum16_f64(part);
  if ((tid & 15) == 15) red[tid >> 4] = part;
  __syncthreads();
  // Every wave sums the (up to 64) row partials with its lanes, as a tree,
  // and evaluates the three scales of the bound check -- at ss - slack, ss
  // and ss + slack -- on lanes 0, 1 and 2 at once (one double division and
  // square root deep, not three).
  const int lane = tid & 63;
  double rs = lane < (nthreads >> 4) ? red[lane] : 0.0;
  rs = row_sum16_f64(rs);
  const double ss = (readlane_f64(rs, 15) + readlane_f64(rs, 31)) + (readlane_f64(rs, 47) + readlane_f64(rs, 63));
  const double slack = sum_slack(in) * ss;
  const float mine = rms_scale(lane == 0 ? ss - slack : lane == 2 ? ss + slack : ss, in, eps);
  float sc = readlane_f32(mine, 1);
  if (readlane_f32(mine, 0) != readlane_f32(mine, 2)) {
    double seq = 0.0;  // every x is in LDS (the barrier above)
    for (int i = 0; i < in; ++i) {
      const double d = static_cast<double>(xs[i]);
      seq = __builtin_fma(d, d, seq);
    }
    sc = rms_scale(seq, in, eps);
    __syncthreads();  // (uniform branch) xs is read before it is scaled
  }
  if (one_round) {
    // This thread's x and w are still in registers.
#pragma unroll
    for (int u = 0; u < kStageBatch; ++u) {
      const int i = u * nthreads + tid;
      if (i < in) xs[i] = w[u] * (v[u] * sc);
    }
  } else {
    // Each thread scales the elements it staged.
    for (int i = tid; i < in; i += nthreads) xs[i] = pw[i] * (xs[i] * sc);
  }
  __syncthreads();
}

// LDS row stride (floats) of a 16-row tile's (block sum, scale) pairs: nblk
// pairs rounded up to 16, plus 4 floats, so the 16 rows start 4 banks apart.
__host__ __device__ __forceinline__ int pair_stride(int nblk) { return 2 * ((nblk + 15) & ~15) + 4; }

// The sequential chain over the (block sum, scale) pairs of one row, two
// blocks per 16-byte LDS read, eight reads (16 blocks) per round.  Two
// register sets: the reads of one round are issued before the fused
// multiply-adds of the other, and whole rounds run without per-block
// conditions (only the last, partial round has them).  The reads walk one
// pointer with constant offsets; a look-ahead may read up to 15 pairs past
// nblk -- inside the next row, or in the padding narrow_lds adds after the
// last row -- and those values are never used.
constexpr int kPairPad = 32;  // floats of look-ahead padding after the last row
__device__ __forceinline__ float chain_pairs(const float* row, int nblk) {
  const float4* pr = reinterpret_cast<const float4*>(row);
  float4 a[8], c[8];
  const auto read = [&](float4* v, const float4* src) {
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = src[u];
  };
  float acc = 0.0f;
  const auto steps = [&](const float4* v) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      acc = __builtin_fmaf(v[u].x, v[u].y, acc);
      acc = __builtin_fmaf(v[u].z, v[u].w, acc);
    }
  };
  read(a, pr);
  int b = 0;
  for (; b + 32 <= nblk; b += 32) {
    read(c, pr + 8);
    __builtin_amdgcn_sched_barrier(0);
    steps(a);
    read(a, pr + 16);
    __builtin_amdgcn_sched_barrier(0);
    steps(c);
    pr += 16;
  }
  // a holds pairs b .. b + 15; fewer than 32 remain.
  if (b + 16 <= nblk) {
    read(c, pr + 8);
    __builtin_amdgcn_sched_barrier(0);
    steps(a);
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = c[u];
    b += 16;
  }
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    if (b + 2 * u < nblk) acc = __builtin_fmaf(a[u].x, a[u].y, acc);
    if (b + 2 * u + 1 < nblk) acc = __builtin_fmaf(a[u].z, a[u].w, acc);
  }
  return acc;
}

// One 16-row tile (batch 1), for matrices with few rows.  Lane l of a
// wavefront owns row tile16*16 + (l & 15) and one of 4 block groups (l >> 4);
// the W wavefronts give 4W groups of bpg contiguous blocks.  The 16 rows of
// one block are a contiguous 256-byte piece of the 64-row layout, so loads
// stay coalesced.  The first kHoist blocks of a lane are loaded before the
// activations are staged (the two round trips overlap).  The activations sit
// in LDS and are read with broadcast loads (16 lanes per address); block
// sums and scales go to LDS as pairs, and lanes 0-15 run the chains.  LDS:
// x[in (padded to 4)], then 16 rows of pair_stride(nblk) floats.
template <int TYPE>
__device__ __forceinline__ void narrow_tile(const GMEM uint4* __restrict__ codes, const GMEM float* __restrict__ scales,
                                            const GMEM float* __restrict__ x, const GMEM float* __restrict__ bias,
                                            GMEM float* __restrict__ y, int in, int nblk, int out, int bpg, int accumulate,
                                            std::size_t tile16, float* lds, int prologue = kPlain,
                                            const GMEM float* __restrict__ pw = nullptr, float eps = 0.0f) {
  constexpr int kHoist = 4;
  const Q4Magic k = q4_magic();
  float* xs = lds;
  const int stride = pair_stride(nblk);
  float* pairs = lds + ((in + 3) & ~3);
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int group = (threadIdx.x >> 6) * 4 + (lane >> 4);
  const std::size_t row = tile16 * 16 + r;
  const std::size_t tile = row / kTileRows;
  const int sub = static_cast<int>(row % kTileRows);
  const int nfull = in / kBlock;
  const int b_begin = group * bpg;
  const int b_end = min(nblk, b_begin + bpg);
  Block<TYPE> pre[kHoist];
  float pre_s[kHoist];
#pragma unroll
  for (int j = 0; j < kHoist; ++j) {
    const int b = b_begin + j;
    if (b < b_end) {
      pre[j] = load_block<TYPE, true>(codes, tile * nblk + b, sub);
      pre_s[j] = loadf<true>(scales + (tile * nblk + b) * kTileRows + sub);
    }
  }
  // The chain lanes fetch their bias and (accumulating) old y now, so that
  // the store at the end does not wait for them.  y is this product's
  // output only, so reading it early is safe.
  float add = 0.0f, old = 0.0f;
  const bool owner = threadIdx.x < 16 && row < static_cast<std::size_t>(out);
  if (owner) {
    if (bias != nullptr) add = bias[row];
    if (accumulate) old = y[row];
  }
  stage_x(x, in, prologue, pw, eps, xs);
  float2* mine = reinterpret_cast<float2*>(pairs + r * stride);
#pragma unroll
  for (int j = 0; j < kHoist; ++j) {
    const int b = b_begin + j;
    if (b < b_end) {
      const float part = b < nfull ? full_block_dot<TYPE>(pre[j], xs + b * kBlock, k)
                                   : tail_block_dot<TYPE>(pre[j], xs + b * kBlock, in - b * kBlock);
      mine[b] = make_float2(part, pre_s[j]);
    }
  }
  for (int b = b_begin + kHoist; b < b_end; ++b) {
    const Block<TYPE> blk = load_block<TYPE, true>(codes, tile * nblk + b, sub);
    const float sc = loadf<true>(scales + (tile * nblk + b) * kTileRows + sub);
    const float part = b < nfull ? full_block_dot<TYPE>(blk, xs + b * kBlock, k)
                                 : tail_block_dot<TYPE>(blk, xs + b * kBlock, in - b * kBlock);
    mine[b] = make_float2(part, sc);
  }
  __syncthreads();
  if (owner) {
    const float v = chain_pairs(pairs + r * stride, nblk) + add;
    y[row] = accumulate ? old + v : v;
  }
}

// grid (ntiles, ceil(rows / R)).
template <int TYPE, int R>
__global__ void __launch_bounds__(1024) qgemv_tile(const uint4* __restrict__ codes, const float* __restrict__ scales,
                                                   const float* __restrict__ x, const float* __restrict__ bias,
                                                   float* __restrict__ y, int in, int nblk, int out, int rows, int bpw,
                                                   int accumulate) {
  extern __shared__ float lds[];
  const int r0 = blockIdx.y * R;
  const int nr = min(R, rows - r0);
  wide_tile<TYPE, R>(gmem(codes), gmem(scales), gmem(x + static_cast<std::size_t>(r0) * in), gmem(bias),
                     gmem_out(y + static_cast<std::size_t>(r0) * out), in, nblk, out, nr, bpw, accumulate, blockIdx.x,
                     lds);
}

// Up to R = 4 or 8 input rows on the matrix cores (qfew.hpp): one workgroup of W wavefronts per 64-row tile.
template <int TYPE, int R, int W>
__global__ void __launch_bounds__(64 * W, 2) qgemv_few(const uint4* __restrict__ codes, const float* __restrict__ scales,
                                                    const float* __restrict__ x, int in, int nblk, int rows, int out,
                                                    const float* __restrict__ bias, float* __restrict__ y,
                                                    int accumulate) {
  few::tile<TYPE, R, W>(gmem(codes), gmem(scales), gmem(x), gmem(bias), gmem_out(y), in, nblk, out, rows, accumulate,
                        blockIdx.x);
}

template <int TYPE>
__global__ void __launch_bounds__(1024) qgemv_narrow(const uint4* __restrict__ codes, const float* __restrict__ scales,
                                                     const float* __restrict__ x, const float* __restrict__ bias,
                                                     float* __restrict__ y, int in, int nblk, int out, int bpg,
                                                     int accumulate) {
  extern __shared__ float4 lds4[];  // 16-byte aligned: the chains read float4
  narrow_tile<TYPE>(gmem(codes), gmem(scales), gmem(x), gmem(bias), gmem_out(y), in, nblk, out, bpg, accumulate,
                    blockIdx.x, reinterpret_cast<float*>(lds4));
}

// One launch over a group's products that share the weight type and the row
// chunk R (64-row tiles).  Workgroup w runs workgroup (w - first_wg) of
// problem wg_prob[w].
template <int TYPE, int R>
__global__ void __launch_bounds__(1024) qgemv_group(const GroupProblem* __restrict__ probs,
                                                    const std::uint32_t* __restrict__ wg_prob) {
  extern __shared__ float lds[];
  const int wg = blockIdx.x;
  // Uniform by construction; readfirstlane keeps the descriptor in SGPRs.
  const int idx = __builtin_amdgcn_readfirstlane(static_cast<int>(wg_prob[wg]));
  const GroupProblem p = probs[idx];
  const int local = wg - p.first_wg;
  const GMEM uint4* codes = gmem(reinterpret_cast<const uint4*>(p.codes));
  const GMEM float* scales = gmem(p.scales);
  const GMEM float* bias = gmem(p.bias);
  const int tile = local % p.ntiles;
  const int r0 = (local / p.ntiles) * R;
  const int nr = min(R, p.rows - r0);
  const GMEM float* x = gmem(p.x + static_cast<std::size_t>(r0) * p.in);
  GMEM float* y = gmem_out(p.y + static_cast<std::size_t>(r0) * p.out);
  wide_tile<TYPE, R>(codes, scales, x, bias, y, p.in, p.nblk, p.out, nr, p.bpw, p.accumulate, tile, lds);
}

// The same for products on the matrix cores (kinds kFew4 and kFew8).
template <int TYPE, int R, int W>
__global__ void __launch_bounds__(64 * W, 2) qgemv_group_few(const GroupProblem* __restrict__ probs,
                                                          const std::uint32_t* __restrict__ wg_prob) {
  const int wg = blockIdx.x;
  const int idx = __builtin_amdgcn_readfirstlane(static_cast<int>(wg_prob[wg]));
  const GroupProblem p = probs[idx];
  few::tile<TYPE, R, W>(gmem(reinterpret_cast<const uint4*>(p.codes)), gmem(p.scales), gmem(p.x), gmem(p.bias),
                        gmem_out(p.y), p.in, p.nblk, p.out, p.rows, p.accumulate, wg - p.first_wg);
}

// The 16-row tiles of a group (batch 1, optional prologue), in a kernel of
// their own so that their staging registers do not lower the occupancy of
// qgemv_group.
template <int TYPE>
__global__ void __launch_bounds__(1024) qgemv_group_narrow(const GroupProblem* __restrict__ probs,
                                                           const std::uint32_t* __restrict__ wg_prob) {
  extern __shared__ float4 lds4[];  // 16-byte aligned: the chains read float4
  const int wg = blockIdx.x;
  const int idx = __builtin_amdgcn_readfirstlane(static_cast<int>(wg_prob[wg]));
  const GroupProblem p = probs[idx];
  narrow_tile<TYPE>(gmem(reinterpret_cast<const uint4*>(p.codes)), gmem(p.scales), gmem(p.x), gmem(p.bias),
                    gmem_out(p.y), p.in, p.nblk, p.out, p.bpw, p.accumulate, wg - p.first_wg,
                    reinterpret_cast<float*>(lds4), p.prologue, gmem(p.pw), p.eps);
}

// The same 16-row tiles for a launch of at most kFewProblems products whose
// descriptors travel as kernel arguments: the kernel starts without the two
// dependent memory reads (workgroup -> product, then the product) of the
// table-driven launch, which sit in front of every load of the one-token
// step's short kernels.
constexpr int kFewProblems = 3;
struct FewProblems {
  GroupProblem p[kFewProblems];
  int count;
};
template <int TYPE>
__global__ void __launch_bounds__(1024) qgemv_few_narrow(FewProblems f) {
  extern __shared__ float4 lds4[];
  const int wg = blockIdx.x;
  // The product by comparisons (uniform), each field by selects, so the
  // argument block is never indexed dynamically.
  const int i = (f.count > 2 && wg >= f.p[2].first_wg) ? 2 : (f.count > 1 && wg >= f.p[1].first_wg) ? 1 : 0;
#define LLMI_PICK(fld) (i == 2 ? f.p[2].fld : i == 1 ? f.p[1].fld : f.p[0].fld)
  narrow_tile<TYPE>(gmem(reinterpret_cast<const uint4*>(LLMI_PICK(codes))), gmem(LLMI_PICK(scales)),
                    gmem(LLMI_PICK(x)), gmem(LLMI_PICK(bias)), gmem_out(LLMI_PICK(y)), LLMI_PICK(in), LLMI_PICK(nblk),
                    LLMI_PICK(out), LLMI_PICK(bpw), LLMI_PICK(accumulate), wg - LLMI_PICK(first_wg),
                    reinterpret_cast<float*>(lds4), LLMI_PICK(prologue), gmem(LLMI_PICK(pw)), LLMI_PICK(eps));
#undef LLMI_PICK
}

// One 16-row-tile product with its descriptor as scalar arguments, ordered
// so that what the first loads need (the weight pointers and shape, x and
// the prologue operand) is among the first 14 dwords, which arrive
// preloaded in SGPRs (-amdgpu-kernarg-preload-count); the one-token step's
// launches of one product take it.
template <int TYPE>
__global__ void __launch_bounds__(1024)
    qgemv_one_narrow(const uint4* __restrict__ codes, const float* __restrict__ scales, const float* __restrict__ x,
                     const float* __restrict__ pw, int nblk, int bpw, int in, int prologue, float eps, int out,
                     const float* __restrict__ bias, float* __restrict__ y, int accumulate) {
  extern __shared__ float4 lds4[];
  narrow_tile<TYPE>(gmem(codes), gmem(scales), gmem(x), gmem(bias), gmem_out(y), in, nblk, out, bpw, accumulate,
                    blockIdx.x, reinterpret_cast<float*>(lds4), prologue, gmem(pw), eps);
}

// The tolerance-mode one-token product split over K (SplitProduct):
// workgroup (tile, split), one wavefront, computes rows tile * 64 + lane over
// blocks [split * BPS, ...): the prologue's loads (the range's activations,
// and for RMSNorm the row's first batch of squares, for the combine the
// chunk partials) are issued first and the weights of all its blocks right
// after them -- loads complete in issue order, so the prologue then waits for
// its own data only and its arithmetic overlaps the weights' trip from HBM;
// the activations of its range are staged in LDS under the prologue, the
// block sums and the chain over its blocks are the exact kernels', and the
// partial sums go to y by atomic adds.
constexpr int kSplitMaxHeads = 8;  // kAttnCombine: whole heads per split (16 blocks of head_dim 64)
// What the first loads' addresses need comes first in the arguments: their
// first 14 dwords arrive preloaded in SGPRs.
template <int TYPE, int PRO, int BPS>
__global__ void __launch_bounds__(64) tsplit_gemv(const uint4* __restrict__ codes, const float* __restrict__ scales,
                                                  const float* __restrict__ x, const float* __restrict__ pw, int nblk,
                                                  int in, int out, int comb_hd, float eps, int comb_nch,
                                                  const float* __restrict__ bias, float* __restrict__ y,
                                                  float* __restrict__ zero, int nzero,
                                                  const int* __restrict__ npos_dev) {
  __shared__ __attribute__((aligned(16))) float xs[BPS * kBlock];
  __shared__ float wgt[PRO == kAttnCombine ? kSplitMaxHeads * kAttnMaxChunks : 1];
  const int lane = threadIdx.x;
  const int tile = blockIdx.x;
  const int b0 = blockIdx.y * BPS;
  const int nb = min(BPS, nblk - b0);
  const GMEM uint4* cg = gmem(codes);
  const GMEM float* sg = gmem(scales);
  Block<TYPE> blk[BPS];
  float sc[BPS];
  const auto load_weights = [&]() {
    __builtin_amdgcn_sched_barrier(0);  // the prologue's loads stay in front
#pragma unroll
    for (int j = 0; j < BPS; ++j) {
      // Past the range: the range's last block again (unused).
      const std::size_t slot = static_cast<std::size_t>(tile) * nblk + static_cast<std::size_t>(b0 + min(j, nb - 1));
      blk[j] = load_block<TYPE, true>(cg, slot, lane);
      sc[j] = loadf<true>(sg + slot * kTileRows + lane);
    }
  };
  // x' over the range [k0, k0 + n): each lane's elements (and, for
  // RMSNorm, its share of the whole row's squares) are loaded in batches
  // before any is used, so the staging costs one memory round trip per
  // batch rather than one per element.
  constexpr int kPer = (BPS * kBlock + 63) / 64;  // range elements per lane
  static_assert(kPer * 64 == BPS * kBlock, "every lane's slots lie inside xs");
  const int k0 = b0 * kBlock, n = min(nb * kBlock, in - k0);
  const GMEM float* xg = gmem(x);
  const GMEM float* pg = gmem(pw);
  // Every load is unconditional, from an index clamped into the row (a load
  // behind a per-lane condition becomes a branch, and the compiler may then
  // wait for it on the spot); values past the range are never stored.
  if constexpr (PRO == kRmsNorm || PRO == kSiluUp || PRO == kPlain) {
    float xv[kPer], pv[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = min(k0 + u * 64 + lane, in - 1);
      xv[u] = xg[i];
      if constexpr (PRO != kPlain) pv[u] = pg[i];
    }
    if constexpr (PRO == kRmsNorm) {
      // The row's squares in batches of kBatch per lane; the first batch's
      // loads go out before the weights'.
      constexpr int kBatch = 16;
      float v[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int i = u * 64 + lane;
        const float t = xg[min(i, in - 1)];
        v[u] = i < in ? t : 0.0f;
      }
      load_weights();
      float ss = 0.0f;
#pragma unroll
      for (int u = 0; u < kBatch; ++u) ss = __builtin_fmaf(v[u], v[u], ss);
      for (int i0 = 64 * kBatch; i0 < in; i0 += 64 * kBatch) {
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const int i = i0 + u * 64 + lane;
          const float t = xg[min(i, in - 1)];
          v[u] = i < in ? t : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) ss = __builtin_fmaf(v[u], v[u], ss);
      }
      ss = wave_sum_dpp(ss);
      const float scale = 1.0f / __builtin_sqrtf(ss / static_cast<float>(in) + eps);
#pragma unroll
      for (int u = 0; u < kPer; ++u) xv[u] = pv[u] * (xv[u] * scale);
    } else {
      load_weights();
      if constexpr (PRO == kSiluUp) {
#pragma unroll
        for (int u = 0; u < kPer; ++u) xv[u] = xv[u] / (1.0f + __expf(-xv[u])) * pv[u];
      }
    }
    // Every slot is stored (xs holds kPer * 64 = BPS * kBlock floats; the
    // block sums read the first n), so no load is sunk behind a condition.
#pragma unroll
    for (int u = 0; u < kPer; ++u) xs[u * 64 + lane] = xv[u];
  } else {
    // kAttnCombine: the range is whole heads h0 .. h0 + nhh - 1; lanes 16r ..
    // 16r + 15 form the chunk weights of head hb + r.  Every chunk slot's
    // partials are loaded (slots past the step's chunks hold finite values
    // -- zeros or an earlier step's -- and get weight 0), so no load waits
    // for the chunk count, which a graph-replayed step reads from memory.
    // From a graph, comb_nch carries the run's chunk length and the count
    // follows from the positions (read after every load is issued).
    const int hd = comb_hd, nh_all = in / hd, h0 = k0 / hd, nhh = n / hd;
    const GMEM float* ms = xg + static_cast<std::size_t>(kAttnMaxChunks) * nh_all * hd;
    const GMEM float* ls = ms + kAttnMaxChunks * nh_all;
    float ov[kPer][kAttnMaxChunks];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = u * 64 + lane;
      const int hh = i / hd, d = i - hh * hd;
      const GMEM float* oh = xg + static_cast<std::size_t>(h0 + min(hh, nhh - 1)) * kAttnMaxChunks * hd + d;
#pragma unroll
      for (int c = 0; c < kAttnMaxChunks; ++c) ov[u][c] = oh[c * hd];  // a clamped head's for i >= n (unused)
    }
    // m and l of both groups of four heads (at most kSplitMaxHeads = 8),
    // then the weights.
    static_assert(kSplitMaxHeads <= 8, "two groups of four heads");
    float m_all[2], l_all[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int t = (h0 + min(4 * g + (lane >> 4), nhh - 1)) * kAttnMaxChunks + (lane & 15);
      m_all[g] = ms[t];
      l_all[g] = ls[t];
    }
    load_weights();
    if (npos_dev != nullptr) comb_nch = (__builtin_amdgcn_readfirstlane(*npos_dev) + comb_nch - 1) / comb_nch;
    // Both groups always (a lane whose head is past the range is not live
    // and stores nothing), so the loads above have a use on every path.
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int hb = 4 * g;
      const int hh = hb + (lane >> 4), c = lane & 15;
      const bool live = hh < nhh && c < comb_nch;
      const float mv = live ? m_all[g] : -__builtin_inff();
      const float lv = live ? l_all[g] : 0.0f;
      const float mx = row_last_bcast(row_max16_f32(mv), lane);
      const float w = live ? __expf(mv - mx) : 0.0f;
      const float den = row_last_bcast(row_sum16_f32(w * lv), lane);
      if (hh < nhh) wgt[hh * kAttnMaxChunks + c] = live ? w / den : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = u * 64 + lane;
      const float* wh = wgt + min(i / hd, nhh - 1) * kAttnMaxChunks;  // past n: a clamped head's (unused)
      float acc_c = 0.0f;
#pragma unroll
      for (int c = 0; c < kAttnMaxChunks; ++c) acc_c = __builtin_fmaf(wh[c], ov[u][c], acc_c);
      xs[i] = acc_c;
    }
  }
  __syncthreads();
  const Q4Magic k = q4_magic();
  const int nfull = in / kBlock - b0;  // whole blocks of the range
  float acc = 0.0f;
  if (nb == BPS && nfull >= BPS) {
    // A range of BPS whole blocks (uniform): no condition per block, so every
    // block's loads have a use on this path and none is sunk past the prologue.
#pragma unroll
    for (int j = 0; j < BPS; ++j) acc = __builtin_fmaf(full_block_dot<TYPE>(blk[j], xs + j * kBlock, k), sc[j], acc);
  } else {
#pragma unroll
    for (int j = 0; j < BPS; ++j) {
      if (j < nb) {
        const float part = j < nfull ? full_block_dot<TYPE>(blk[j], xs + j * kBlock, k)
                                     : tail_block_dot<TYPE>(blk[j], xs + j * kBlock, in - (b0 + j) * kBlock);
        acc = __builtin_fmaf(part, sc[j], acc);
      }
    }
  }
  const int row = tile * kTileRows + lane;
  if (row < out) {
    if (blockIdx.y == 0 && bias != nullptr) acc += bias[row];
    unsafeAtomicAdd(y + row, acc);
  }
  // Clearing the next product's output (a buffer this launch does not
  // read): last, so that its stores are not ahead of any load in the
  // counter the waits above use.
  if (zero != nullptr) {
    const int wg = static_cast<int>(blockIdx.y * gridDim.x + blockIdx.x);
    const int stride = static_cast<int>(gridDim.x * gridDim.y) * 64;
    for (int i = wg * 64 + lane; i < nzero; i += stride) zero[i] = 0.0f;
  }
}

// ------------------------------------------------------------ planning
// LDS bytes of one workgroup of each kind.
// part[nr][nblk][64], scale[nblk][64], then the chain's look-ahead padding.
std::size_t wide_lds(std::size_t nblk, std::size_t nr) {
  return ((nr + 1) * nblk + 2 * kChainRound) * kTileRows * sizeof(float);
}
// x[in (padded to 4)], 16 rows of pairs, then chain_pairs' look-ahead padding.
std::size_t narrow_lds(std::size_t in, std::size_t nblk) {
  return (((in + 3) & ~std::size_t{3}) + 16 * static_cast<std::size_t>(pair_stride(static_cast<int>(nblk))) +
          kPairPad) *
         sizeof(float);
}

// LDS a wide workgroup aims to stay within, so that several workgroups share
// a CU; longer rows may use up to the per-workgroup maximum.
constexpr std::size_t kLdsTarget = 64 * 1024;

// Whether a 64-row tile's block sums of one input row fit LDS (in up to ~10k).
bool wide_fits(std::size_t nblk) { return wide_lds(nblk, 1) <= max_lds_per_block(); }

// Row chunk R (1, 2 or 4) of a wide workgroup on the vector ALUs, at most
// `want`, halved until its LDS fits.
int pick_chunk(int want, std::size_t rows, std::size_t nblk) {
  for (int r = want; r > 1; r /= 2)
    if (wide_lds(nblk, std::min<std::size_t>(rows, r)) <= kLdsTarget) return r;
  return 1;
}

// Long rows on so few tiles that chunks of the input rows, two or more per
// tile, give each CU at most one workgroup: the smallest such chunk on the
// vector ALUs, 0 if there is none.  A workgroup on the matrix cores takes all
// the rows, which leaves most CUs idle here, and the many blocks make its
// chain long (us, vector ALUs / else, Q8_0): 2048 x 2048 at 3 rows 5.6 / 7.4
// and, in a group, at 8 rows 6.1 / 11.0; 8192 x 2560 at 4 rows 9.1 / 10.9; 144
// x 1712 at 7 rows in a group 5.9 / 9.4; 6000 x 896 at 8 rows 5.6 / 6.3.  Long
// is 33 whole blocks, from 3 rows on 32 in a group of Q4_0 and 28 of Q8_0, and
// 41 with a partial one (us: Q4_0 6000 x 1100 at 5 rows 7.6 / 7.2, 6000 x 896
// at 6 rows in a group 6.4 / 6.0, alone 4096 x 896 at 8 rows 5.3 / 4.8; Q8_0
// 2000 x 896 at 2 rows 4.6 / 4.3).
int few_chunk(const DeviceMatrix& m, std::size_t rows, std::size_t tiles, bool group) {
  constexpr std::size_t kCus = 256;
  const std::size_t lng = m.in % kBlock != 0 ? 41 : rows == 2 ? 33 : m.type == LLMI_TYPE_Q8_0 ? 28 : group ? 32 : 33;
  if (m.nblk < lng) return 0;
  for (std::size_t r = 1; r <= 4 && r < rows; r *= 2)
    if (tiles * ceil_div(rows, r) <= kCus) return r == 1 || wide_lds(m.nblk, r) <= kLdsTarget ? static_cast<int>(r) : 0;
  return 0;
}

// How a launch of `tiles` 64-row tiles runs a product of 2..8 rows that
// few_chunk has no chunk for on 64-row tiles (GroupProblem's kinds), by
// measurement (us, vector ALUs / matrix cores, Q4_0 and Q8_0):
//   rows of more than 64 blocks on up to 128 tiles: row chunks on several
//     workgroups (896 x 4864 10.4 / 15.2);
//   2 rows: the vector ALUs -- half of a 4-row matrix instruction's rows are
//     empty -- (151936 x 896 20.4 / 24.6, 4864 x 896 4.6 / 5.0) except for
//     Q8_0, whose codes decode for less, on many tiles (32.6 / 25.7), and for a
//     partial last block (4864 x 870 5.1 / 4.6, 32000 x 2075 15.5 / 13.7);
//   3 rows of Q4_0 on many tiles: 49152 x 576 6.7 / 7.4;
//   else the matrix cores (151936 x 896 at 8 rows 52.3 / 33.6 and 78.2 /
//     35.6, at 4 27.9 / 24.2 and 41.7 / 26.3).
int few_kind(const DeviceMatrix& m, std::size_t rows, std::size_t tiles) {
  if (m.nblk > 64 && tiles < 128) return pick_chunk(4, rows, m.nblk);
  if (rows == 2 && m.in % kBlock == 0 && (m.type == LLMI_TYPE_Q4_0 || tiles < 512)) return pick_chunk(2, rows, m.nblk);
  if (rows == 3 && m.type == LLMI_TYPE_Q4_0 && tiles >= 512 && pick_chunk(4, rows, m.nblk) == 4) return 4;
  return rows <= 4 ? GroupProblem::kFew4 : GroupProblem::kFew8;
}

// Wavefronts per tile on the matrix cores (4, 8 or 16; us at 8 rows, Q4_0): by
// the tiles, enough to fill the GPU (768 tiles of 576 inputs 9.3 / 10.2 /
// 12.5; 256 of 896 7.5 / 6.8 / 7.3; 76 7.2 / 6.3 / 5.7); long rows keep 16
// for longer (128 of 2560 at 5 rows 17.4 / 13.6 / 12.0).
int few_waves(std::size_t tiles, std::size_t nblk) {
  return tiles >= 512 ? 4 : tiles >= (nblk > 32 ? 192u : 128u) ? 8 : 16;
}

// Wavefronts per 64-row tile: each takes about kBlocksPerWave blocks (4 for
// Q4_0, 2 for Q8_0: about 4 KB of codes and scales in flight per
// wavefront), at most 16.  Measured on MI355X over the 151936x896 lm_head.
int wide_waves(std::size_t nblk, int type) {
  const std::size_t per = type == LLMI_TYPE_Q8_0 ? 2 : 4;
  return static_cast<int>(std::clamp<std::size_t>(ceil_div(nblk, per), 1, 16));
}

// Wavefronts of a 16-row tile: about two blocks per lane group (4 groups per
// wavefront), at most 64 groups.
int narrow_waves(std::size_t nblk) {
  constexpr std::size_t kBlocksPerGroup = 2;
  const std::size_t groups = std::clamp<std::size_t>(ceil_div(nblk, kBlocksPerGroup), 1, 64);
  return static_cast<int>(ceil_div(groups, 4));
}

struct TilePlan {
  int kind = 0;  // 0: the multi-row product (qrows.hip); else a GroupProblem kind
  int waves = 1;
  int bpw = 1;
  std::size_t lds = 0;
};

// Launch shape of a single product.  Batch 1 matrices with fewer than
// kNarrowTiles 64-row tiles use 16-row tiles (more workgroups); otherwise
// the wide tile.
TilePlan plan_single(const DeviceMatrix& m, std::size_t rows) {
  constexpr std::size_t kNarrowTiles = 128;
  const std::size_t nblk = std::max<std::size_t>(m.nblk, 1);
  TilePlan p;
  if (rows > 8) return p;
  if (rows == 1 && m.ntiles < kNarrowTiles && narrow_lds(m.in, nblk) <= max_lds_per_block()) {
    p.kind = GroupProblem::kNarrow;
    p.waves = narrow_waves(nblk);
    p.bpw = static_cast<int>(ceil_div(nblk, static_cast<std::size_t>(p.waves) * 4));
    p.lds = narrow_lds(m.in, nblk);
    return p;
  }
  if (!wide_fits(nblk)) return p;  // rows too long for LDS staging
  const int chunk = rows > 1 ? few_chunk(m, rows, m.ntiles, false) : 0;
  // Few tiles: 16-row x 16-output tiles spread the product over more CUs
  // (qrows.hip; 576 x 576 at 4 rows 3.7 us, on 64-row tiles 4.0), which
  // rows of a partial block take from two rows on (2749 x 1003 4.6, 6.8);
  // 6 rows and more fill them better (4864 x 896 at 8 rows of Q8_0 5.9, 6.8;
  // 6000 x 2048 10.3, 11.0, but 8192 x 1800 at 6 11.4, 9.3).
  const std::size_t few_tiles = rows <= 5 ? 64 : nblk <= 32 ? 128 : 96;
  if (rows > 1 && nblk <= 64 && m.ntiles <= few_tiles && (rows > 2 || m.in % kBlock != 0) &&
      chunk == 0)
    return p;
  p.kind = rows == 1 ? 1 : chunk != 0 ? chunk : few_kind(m, rows, m.ntiles);
  if (p.kind == GroupProblem::kFew4 || p.kind == GroupProblem::kFew8) {
    p.waves = few_waves(m.ntiles, nblk);
    return p;
  }
  p.bpw = static_cast<int>(ceil_div(nblk, wide_waves(nblk, m.type)));
  p.waves = static_cast<int>(ceil_div(nblk, p.bpw));
  p.lds = wide_lds(nblk, std::min<std::size_t>(rows, p.kind));
  return p;
}

template <int TYPE, int R>
void launch_tile(const DeviceMatrix& m, const float* x, std::size_t rows, const float* bias, float* y, int acc,
                 const TilePlan& p, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(m.ntiles), static_cast<unsigned>(ceil_div(rows, R)));
  qgemv_tile<TYPE, R><<<grid, static_cast<unsigned>(p.waves * 64), p.lds, s>>>(
      reinterpret_cast<const uint4*>(m.codes), m.scales, x, bias, y, static_cast<int>(m.in), static_cast<int>(m.nblk),
      static_cast<int>(m.out), static_cast<int>(rows), p.bpw, acc);
}

template <int TYPE, int R>
void launch_few(const DeviceMatrix& m, const float* x, std::size_t rows, const float* bias, float* y, int acc, int waves,
                hipStream_t s) {
  const auto* codes = reinterpret_cast<const uint4*>(m.codes);
  const unsigned grid = static_cast<unsigned>(m.ntiles);
  const int in = static_cast<int>(m.in), nblk = static_cast<int>(m.nblk), out = static_cast<int>(m.out);
  const int nr = static_cast<int>(rows);
  if (waves == 4) qgemv_few<TYPE, R, 4><<<grid, 256, 0, s>>>(codes, m.scales, x, in, nblk, nr, out, bias, y, acc);
  else if (waves == 8) qgemv_few<TYPE, R, 8><<<grid, 512, 0, s>>>(codes, m.scales, x, in, nblk, nr, out, bias, y, acc);
  else qgemv_few<TYPE, R, 16><<<grid, 1024, 0, s>>>(codes, m.scales, x, in, nblk, nr, out, bias, y, acc);
}

template <int TYPE>
void launch_typed(const DeviceMatrix& m, const float* x, std::size_t rows, const float* bias, float* y, int acc,
                  const TilePlan& p, hipStream_t s) {
  switch (p.kind) {
    case GroupProblem::kNarrow:
      qgemv_narrow<TYPE><<<static_cast<unsigned>(ceil_div(m.out, 16)), static_cast<unsigned>(p.waves * 64), p.lds, s>>>(
          reinterpret_cast<const uint4*>(m.codes), m.scales, x, bias, y, static_cast<int>(m.in),
          static_cast<int>(m.nblk), static_cast<int>(m.out), p.bpw, acc);
      break;
    case 1: launch_tile<TYPE, 1>(m, x, rows, bias, y, acc, p, s); break;
    case 2: launch_tile<TYPE, 2>(m, x, rows, bias, y, acc, p, s); break;
    case 4: launch_tile<TYPE, 4>(m, x, rows, bias, y, acc, p, s); break;
    case GroupProblem::kFew4: launch_few<TYPE, 4>(m, x, rows, bias, y, acc, p.waves, s); break;
    default: launch_few<TYPE, 8>(m, x, rows, bias, y, acc, p.waves, s); break;
  }
}

// The kinds of a group's products on 64-row tiles (`total` of them in all).
// Products of different kinds are different launches, one after another, so
// products of one type agree where they can, the heaviest deciding (us, one
// kind each / agreed, Q4_0: 2048 x 2048, 500 x 1024 and 300 x 700 at 2 rows
// 11.0 / 6.9).  Rows of more than 64 blocks go by themselves: few of them, as
// a layer's down projection, would keep a launch of short ones waiting for
// their chains (a Qwen2.5 layer's seven products in one launch / by
// themselves: Q4_0 at 5 rows 24.1 / 17.6, Q8_0 24.3 / 19.8, but at 4 rows of
// Q8_0 17.6 / 18.7).
std::vector<int> group_kinds(const GroupEntry* entries, std::size_t count, std::size_t total) {
  constexpr std::size_t kLong = 64;
  std::vector<int> kinds(count, 1);
  for (int type : {LLMI_TYPE_Q8_0, LLMI_TYPE_Q4_0})
  for (bool lng : {false, true}) {
    std::vector<std::size_t> of;
    std::size_t tiles = 0, heaviest = 0;
    for (std::size_t i = 0; i < count; ++i) {
      const DeviceMatrix& m = *entries[i].m;
      if (entries[i].rows == 1 || m.out == 0 || m.type != type || (m.nblk > kLong) != lng) continue;
      if (of.empty() || m.code_bytes > entries[heaviest].m->code_bytes) heaviest = i;
      of.push_back(i);
      tiles += m.ntiles;
    }
    bool chunked = true;  // few_chunk has the same chunk for all
    for (std::size_t i : of) {
      kinds[i] = few_chunk(*entries[i].m, entries[i].rows, tiles, true);
      chunked = chunked && kinds[i] != 0 && kinds[i] == kinds[of[0]];
    }
    if (chunked) continue;
    for (std::size_t i : of) kinds[i] = few_kind(*entries[i].m, entries[i].rows, lng ? tiles : total);
    if (of.empty()) continue;
    const int k = kinds[heaviest];
    const auto on_cores = [](int kind) { return kind == GroupProblem::kFew4 || kind == GroupProblem::kFew8; };
    for (std::size_t i : of) {
      const GroupEntry& e = entries[i];
      if (on_cores(k)) kinds[i] = e.rows <= 4 ? GroupProblem::kFew4 : GroupProblem::kFew8;
      else if (on_cores(kinds[i]) && pick_chunk(k, e.rows, e.m->nblk) == k) kinds[i] = k;
    }
  }
  return kinds;
}

int check_shape(const DeviceMatrix& m, std::size_t rows) {
  LLMI_REQUIRE(m.in > 0, "matmul: in must be positive");
  LLMI_REQUIRE(m.in <= 0x7FFFFFFFu && m.out <= 0x7FFFFFFFu, "matmul: shape too large");
  LLMI_REQUIRE(ceil_div(rows, 8) <= 65535, "matmul: too many input rows for one launch");
  return LLMI_OK;
}

}  // namespace

int launch_matmul(const DeviceMatrix& m, const float* x, std::size_t rows, const float* bias, float* y, hipStream_t s,
                  bool accumulate) {
  if (rows == 0 || m.out == 0) return LLMI_OK;
  if (m.type == LLMI_TYPE_F32) {
    LLMI_REQUIRE(x != nullptr && y != nullptr, "matmul: null pointer");
    return launch_matmul_f32(m, x, rows, bias, y, s, accumulate);
  }
  if (int rc = check_shape(m, rows)) return rc;
  LLMI_REQUIRE(x != nullptr && y != nullptr, "matmul: null pointer");
  const TilePlan p = plan_single(m, rows);
  if (p.kind == 0) return launch_rows(m, x, rows, bias, y, s, accumulate);
  const int acc = accumulate ? 1 : 0;
  if (m.type == LLMI_TYPE_Q8_0) launch_typed<LLMI_TYPE_Q8_0>(m, x, rows, bias, y, acc, p, s);
  else launch_typed<LLMI_TYPE_Q4_0>(m, x, rows, bias, y, acc, p, s);
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

int plan_group(const GroupEntry* entries, std::size_t count, GroupPlan* plan) {
  // Narrow 16-row tiles for batch-1 products only when the 64-row tiles would
  // leave the GPU mostly idle (fewer than ~4 workgroups per CU), and for long
  // rows (more than kNarrowMaxBlocks blocks) only below one 64-row workgroup
  // per CU: 24 Qwen2.5 down_proj matrices (896 x 4864, 336 64-row tiles) in
  // one launch stream about twice as fast on 64-row tiles, one alone (14
  // tiles) about 1.6x faster on 16-row tiles (measured on MI355X).  A
  // prologue always needs them.
  constexpr std::size_t kNarrowBelow = 1024;
  constexpr std::size_t kNarrowMaxBlocks = 64;
  constexpr std::size_t kLongRowsNarrowBelow = 256;
  *plan = GroupPlan{};
  std::size_t wide_total = 0;
  for (std::size_t i = 0; i < count; ++i) {
    const GroupEntry& e = entries[i];
    LLMI_REQUIRE(e.m != nullptr, "group: null weight");
    LLMI_REQUIRE(e.m->type != LLMI_TYPE_F32, "group: fp32 weights are not part of grouped launches");
    LLMI_REQUIRE(e.rows >= 1 && e.rows <= 8, "group: each product takes 1..8 input rows");
    LLMI_REQUIRE(e.x != nullptr && e.y != nullptr, "group: null x or y");
    if (int rc = check_shape(*e.m, e.rows)) return rc;
    wide_total += e.m->ntiles * ceil_div(e.rows, 8);
  }
  // Products are launched by weight type and row chunk R (one kernel
  // instance each).
  const std::vector<int> kinds = group_kinds(entries, count, wide_total);
  for (int type : {LLMI_TYPE_Q8_0, LLMI_TYPE_Q4_0})
  for (int R : {int{GroupProblem::kNarrow}, 1, 2, 4, int{GroupProblem::kFew4}, int{GroupProblem::kFew8}}) {
    const bool few = R == GroupProblem::kFew4 || R == GroupProblem::kFew8;
    std::vector<GroupProblem> probs;
    std::size_t biggest = 0;
    int waves = 1;
    for (std::size_t i = 0; i < count; ++i) {
      const GroupEntry& e = entries[i];
      const DeviceMatrix& m = *e.m;
      if (m.out == 0) continue;
      const bool fits = narrow_lds(m.in, m.nblk) <= max_lds_per_block();
      const bool narrow =
          e.rows == 1 && fits &&
          (e.prologue != kPlain ||
           (wide_total < kNarrowBelow && (m.nblk <= kNarrowMaxBlocks || wide_total < kLongRowsNarrowBelow)));
      LLMI_REQUIRE(e.prologue == kPlain || narrow, "group: a prologue needs batch 1 and in <= ~20k");
      LLMI_REQUIRE(e.prologue == kPlain || e.prologue == kRmsNorm || e.prologue == kSiluUp,
                   "group: unknown prologue");
      LLMI_REQUIRE(narrow || wide_fits(m.nblk), "group: rows too long for the grouped GEMV (in above ~10k)");
      if (m.type != type) continue;
      const int r = narrow ? int{GroupProblem::kNarrow} : kinds[i];
      if (r != R) continue;
      GroupProblem p{};
      p.codes = m.codes;
      p.scales = m.scales;
      p.x = e.x;
      p.bias = e.bias;
      p.y = e.y;
      p.type = m.type;
      p.kind = r;
      p.in = static_cast<int>(m.in);
      p.nblk = static_cast<int>(m.nblk);
      p.out = static_cast<int>(m.out);
      p.rows = static_cast<int>(e.rows);
      p.ntiles = static_cast<int>(m.ntiles);
      p.accumulate = e.accumulate ? 1 : 0;
      p.prologue = e.prologue;
      p.pw = e.pw;
      p.eps = e.eps;
      probs.push_back(p);
      // The launch's wavefront count: the most any 16-row tile wants, or
      // what the largest product wants for 64-row tiles.
      const std::size_t bytes = m.code_bytes + m.scale_bytes;
      if (narrow) {
        waves = std::max(waves, narrow_waves(m.nblk));
      } else if (bytes > biggest) {
        biggest = bytes;
        waves = wide_waves(m.nblk, m.type);
      }
    }
    if (probs.empty()) continue;
    // Longest workgroups first (most blocks per tile): they start while the
    // short ones fill the GPU around them, and the launch ends on short
    // workgroups.  (Qwen2.5's 24 MLP layers in one launch: 61% / 81% of HBM
    // peak for Q4_0 / Q8_0 against 50% / 71% in layer order.)
    std::stable_sort(probs.begin(), probs.end(),
                     [](const GroupProblem& a, const GroupProblem& b) { return a.nblk > b.nblk; });
    GroupLaunch l;
    l.type = type;
    l.rchunk = R;
    l.waves = waves;
    l.prob_offset = plan->probs.size();
    l.map_offset = plan->wg_prob.size();
    std::size_t wg = 0;
    for (std::size_t j = 0; j < probs.size(); ++j) {
      GroupProblem& p = probs[j];
      std::size_t wgs = 0, need = 0;
      if (p.kind == GroupProblem::kNarrow) {
        p.bpw = static_cast<int>(ceil_div(p.nblk, static_cast<std::size_t>(waves) * 4));
        wgs = ceil_div(p.out, 16);
        need = narrow_lds(p.in, p.nblk);
      } else {
        wgs = static_cast<std::size_t>(p.ntiles) * (few ? 1 : ceil_div(p.rows, R));
        if (!few) {
          p.bpw = static_cast<int>(ceil_div(p.nblk, waves));
          need = wide_lds(p.nblk, std::min(p.rows, R));
        }
      }
      p.first_wg = static_cast<int>(wg);
      wg += wgs;
      LLMI_REQUIRE(wg <= 0x7FFFFFFFu, "group: too many workgroups");
      l.lds = std::max(l.lds, need);
      plan->wg_prob.insert(plan->wg_prob.end(), wgs, static_cast<std::uint32_t>(j));
    }
    if (few) l.waves = few_waves(wg, static_cast<std::size_t>(probs[0].nblk));
    LLMI_REQUIRE(l.lds <= max_lds_per_block(), "group: a product needs more LDS than one workgroup may use");
    l.total_wgs = static_cast<int>(wg);
    l.nprob = static_cast<int>(probs.size());
    plan->probs.insert(plan->probs.end(), probs.begin(), probs.end());
    plan->launches.push_back(l);
  }
  return LLMI_OK;
}

namespace {
template <int TYPE, int R>
void launch_group_few_rows(const GroupProblem* probs, const std::uint32_t* map, const GroupLaunch& l, hipStream_t s) {
  const unsigned grid = static_cast<unsigned>(l.total_wgs);
  if (l.waves == 4) qgemv_group_few<TYPE, R, 4><<<grid, 256, 0, s>>>(probs, map);
  else if (l.waves == 8) qgemv_group_few<TYPE, R, 8><<<grid, 512, 0, s>>>(probs, map);
  else qgemv_group_few<TYPE, R, 16><<<grid, 1024, 0, s>>>(probs, map);
}
template <int TYPE>
void launch_group_wide(const GroupProblem* probs, const std::uint32_t* map, const GroupLaunch& l, hipStream_t s) {
  const unsigned grid = static_cast<unsigned>(l.total_wgs), block = static_cast<unsigned>(l.waves * 64);
  switch (l.rchunk) {
    case 1: qgemv_group<TYPE, 1><<<grid, block, l.lds, s>>>(probs, map); break;
    case 2: qgemv_group<TYPE, 2><<<grid, block, l.lds, s>>>(probs, map); break;
    case 4: qgemv_group<TYPE, 4><<<grid, block, l.lds, s>>>(probs, map); break;
    case GroupProblem::kFew4: launch_group_few_rows<TYPE, 4>(probs, map, l, s); break;
    default: launch_group_few_rows<TYPE, 8>(probs, map, l, s); break;
  }
}
}  // namespace

int launch_group(const GroupProblem* probs_dev, const std::uint32_t* map_dev, const GroupLaunch& l, hipStream_t s) {
  if (l.total_wgs == 0) return LLMI_OK;
  const dim3 grid(static_cast<unsigned>(l.total_wgs)), block(static_cast<unsigned>(l.waves * 64));
  const GroupProblem* probs = probs_dev + l.prob_offset;
  const std::uint32_t* map = map_dev + l.map_offset;
  if (l.rchunk == GroupProblem::kNarrow) {
    if (l.type == LLMI_TYPE_Q8_0) qgemv_group_narrow<LLMI_TYPE_Q8_0><<<grid, block, l.lds, s>>>(probs, map);
    else qgemv_group_narrow<LLMI_TYPE_Q4_0><<<grid, block, l.lds, s>>>(probs, map);
  } else if (l.type == LLMI_TYPE_Q8_0) {
    launch_group_wide<LLMI_TYPE_Q8_0>(probs, map, l, s);
  } else {
    launch_group_wide<LLMI_TYPE_Q4_0>(probs, map, l, s);
  }
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

int DeviceGroup::build(const GroupEntry* entries, std::size_t count) {
  release();
  GroupPlan plan;
  if (int rc = plan_group(entries, count, &plan)) return rc;
  launches = plan.launches;
  host_probs = plan.probs;
  const std::size_t pbytes = plan.probs.size() * sizeof(GroupProblem);
  const std::size_t mbytes = plan.wg_prob.size() * sizeof(std::uint32_t);
  if (pbytes + mbytes == 0) return LLMI_OK;
  LLMI_TRY_HIP(hipMalloc(&table, pbytes + mbytes));
  auto* base = static_cast<std::uint8_t*>(table);
  LLMI_TRY_HIP(hipMemcpy(base, plan.probs.data(), pbytes, hipMemcpyHostToDevice));
  if (mbytes > 0) LLMI_TRY_HIP(hipMemcpy(base + pbytes, plan.wg_prob.data(), mbytes, hipMemcpyHostToDevice));
  probs = reinterpret_cast<const GroupProblem*>(base);
  map = reinterpret_cast<const std::uint32_t*>(base + pbytes);
  return LLMI_OK;
}

int DeviceGroup::launch(hipStream_t s) const {
  for (const GroupLaunch& l : launches) {
    if (l.rchunk == GroupProblem::kNarrow && l.nprob >= 1 && l.nprob <= kFewProblems && l.total_wgs > 0) {
      // Few products: descriptors by value (qgemv_few_narrow).
      FewProblems f{};
      f.count = l.nprob;
      for (int k = 0; k < l.nprob; ++k) f.p[k] = host_probs[l.prob_offset + static_cast<std::size_t>(k)];
      const dim3 grid(static_cast<unsigned>(l.total_wgs)), block(static_cast<unsigned>(l.waves * 64));
      if (l.nprob == 1) {
        // One product: scalar arguments (preloaded), qgemv_one_narrow.
        const GroupProblem& p = f.p[0];
        const auto* codes = reinterpret_cast<const uint4*>(p.codes);
#define LLMI_ONE_ARGS \
  codes, p.scales, p.x, p.pw, p.nblk, p.bpw, p.in, p.prologue, p.eps, p.out, p.bias, p.y, p.accumulate
        if (l.type == LLMI_TYPE_Q8_0) {
          qgemv_one_narrow<LLMI_TYPE_Q8_0><<<grid, block, l.lds, s>>>(LLMI_ONE_ARGS);
        } else {
          qgemv_one_narrow<LLMI_TYPE_Q4_0><<<grid, block, l.lds, s>>>(LLMI_ONE_ARGS);
        }
#undef LLMI_ONE_ARGS
        LLMI_TRY_HIP(hipGetLastError());
        continue;
      }
      if (l.type == LLMI_TYPE_Q8_0) {
        qgemv_few_narrow<LLMI_TYPE_Q8_0><<<grid, block, l.lds, s>>>(f);
      } else {
        qgemv_few_narrow<LLMI_TYPE_Q4_0><<<grid, block, l.lds, s>>>(f);
      }
      LLMI_TRY_HIP(hipGetLastError());
      continue;
    }
    if (int rc = launch_group(probs, map, l, s)) return rc;
  }
  return LLMI_OK;
}

// Splits of a SplitProduct: about kSplitTarget workgroups, BPS (the
// kernel's blocks per split) one of 2, 4, 8, 16, and the power of two is
// taken below max(nblk / (kSplitTarget / tiles), nblk / kSplitMaxPerOutput):
// the atomic adds into one cache line of y are applied one after another
// (152 per output cost ~3 us more than plain stores on MI355X), so long rows
// take wider splits.
constexpr int kSplitTarget = 1024;
constexpr int kSplitMaxPerOutput = 40;

int plan_split(SplitProduct* p) {
  LLMI_REQUIRE(p->m != nullptr && p->x != nullptr && p->y != nullptr, "split product: null operand");
  const DeviceMatrix& m = *p->m;
  LLMI_REQUIRE(m.type == LLMI_TYPE_Q8_0 || m.type == LLMI_TYPE_Q4_0, "split product: Q8_0 or Q4_0 weights only");
  LLMI_REQUIRE(p->prologue == kRmsNorm || p->prologue == kSiluUp || p->prologue == kAttnCombine ||
                   p->prologue == kPlain,
               "split product: unknown prologue");
  LLMI_REQUIRE(p->prologue == kPlain || p->pw != nullptr, "split product: null prologue operand");
  const int nblk = static_cast<int>(m.nblk), ntiles = static_cast<int>(m.ntiles);
  LLMI_REQUIRE(nblk >= 1 && ntiles >= 1, "split product: empty matrix");
  const int want = std::max(1, kSplitTarget / ntiles);
  int bps = static_cast<int>(ceil_div(static_cast<std::size_t>(nblk), static_cast<std::size_t>(want)));
  bps = std::max(bps, static_cast<int>(ceil_div(static_cast<std::size_t>(nblk),
                                                static_cast<std::size_t>(kSplitMaxPerOutput))));
  int unit = 1;
  if (p->prologue == kAttnCombine) {
    LLMI_REQUIRE(p->comb_hd >= 32 && p->comb_hd % kBlock == 0 && m.in % static_cast<std::size_t>(p->comb_hd) == 0,
                 "split product: an attention-combine product needs in = heads * head_dim, head_dim % 32 == 0");
    unit = p->comb_hd / kBlock;
  }
  int pick = 2;
  while (pick < 16 && (2 * pick <= bps || pick % unit != 0)) pick *= 2;
  LLMI_REQUIRE(pick % unit == 0 && (p->prologue != kAttnCombine || pick * kBlock / p->comb_hd <= kSplitMaxHeads),
               "split product: head_dim too large for a split");
  p->bps = pick;
  p->splits = static_cast<int>(ceil_div(static_cast<std::size_t>(nblk), static_cast<std::size_t>(pick)));
  return LLMI_OK;
}

namespace {

template <int TYPE, int PRO>
void launch_split_bps(const SplitProduct& p, hipStream_t s, int comb_nch, const int* npos_dev) {
  const DeviceMatrix& m = *p.m;
  const dim3 grid(static_cast<unsigned>(m.ntiles), static_cast<unsigned>(p.splits));
#define LLMI_SPLIT_ARGS                                                                                            \
  reinterpret_cast<const uint4*>(m.codes), m.scales, p.x, p.pw, static_cast<int>(m.nblk), static_cast<int>(m.in), \
      static_cast<int>(m.out), p.comb_hd, p.eps, comb_nch, p.bias, p.y, p.zero, p.nzero, npos_dev
  switch (p.bps) {
    case 2: tsplit_gemv<TYPE, PRO, 2><<<grid, 64, 0, s>>>(LLMI_SPLIT_ARGS); break;
    case 4: tsplit_gemv<TYPE, PRO, 4><<<grid, 64, 0, s>>>(LLMI_SPLIT_ARGS); break;
    case 8: tsplit_gemv<TYPE, PRO, 8><<<grid, 64, 0, s>>>(LLMI_SPLIT_ARGS); break;
    default: tsplit_gemv<TYPE, PRO, 16><<<grid, 64, 0, s>>>(LLMI_SPLIT_ARGS); break;
  }
#undef LLMI_SPLIT_ARGS
}

template <int TYPE>
void launch_split_type(const SplitProduct& p, hipStream_t s, int comb_nch, const int* npos_dev) {
  switch (p.prologue) {
    case kRmsNorm: launch_split_bps<TYPE, kRmsNorm>(p, s, comb_nch, nullptr); break;
    case kSiluUp: launch_split_bps<TYPE, kSiluUp>(p, s, comb_nch, nullptr); break;
    case kAttnCombine: launch_split_bps<TYPE, kAttnCombine>(p, s, comb_nch, npos_dev); break;
    default: launch_split_bps<TYPE, kPlain>(p, s, comb_nch, nullptr); break;
  }
}

}  // namespace

int launch_split(const SplitProduct& p, hipStream_t s, int comb_nch, const int* npos_dev) {
  LLMI_REQUIRE(p.m != nullptr && p.splits >= 1 && (p.bps == 2 || p.bps == 4 || p.bps == 8 || p.bps == 16),
               "split product: not planned");
  LLMI_REQUIRE(p.prologue != kAttnCombine || npos_dev != nullptr || (comb_nch >= 1 && comb_nch <= kAttnMaxChunks),
               "split product: attention chunks out of range");
  if (p.m->type == LLMI_TYPE_Q8_0) launch_split_type<LLMI_TYPE_Q8_0>(p, s, comb_nch, npos_dev);
  else launch_split_type<LLMI_TYPE_Q4_0>(p, s, comb_nch, npos_dev);
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

void DeviceGroup::release() {
  if (table != nullptr) (void)hipFree(table);
  table = nullptr;
  probs = nullptr;
  map = nullptr;
  launches.clear();
  host_probs.clear();
}

}  // namespace llmi_hip
