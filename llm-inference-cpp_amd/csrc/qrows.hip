// The exact multi-row product (more than 8 input rows) on the matrix cores.
//
// Reference: src/model/quant.cpp:119-153, as gemv.hip describes it:
//     part_b = fma(x[k], code[k], part_b)   over the block's 32 elements in order
//     acc    = fma(part_b, scale_b, acc)    over the blocks in order
//     y      = acc + bias[o]
// v_mfma_f32_16x16x4_f32 computes, for each of its 16 x 16 outputs, exactly
// such a chain: d = fma(a3, b3, fma(a2, b2, fma(a1, b1, fma(a0, b0, c)))),
// one IEEE rounding (to nearest even, subnormals kept) per step.  Checked on
// MI355X against fmaf chains over 3M results (wide exponents, subnormal
// inputs and results, cancellation): no bit differs, and the tests compare
// whole products with the oracle bit for bit.  So eight of them are one
// block's sums for 16 rows x 16 outputs, in the reference's order, at the
// matrix cores' fp32 rate (148 TFLOP/s measured; plain fp32 FMAs without the
// packed forms reach half of that, and the kernels this one replaced 37).
//
// Bound: the fp32 units, which the matrix instructions share with the vector
// ones: measured, every VALU instruction between two v_mfma_f32_16x16x4_f32
// (13.5 ns) adds its own time (fused multiply-add 1.5 ns, conversion or
// v_perm 2.4 ns), in the same wavefront or another.  So the shape of a
// wavefront's work is chosen for few vector instructions per matrix
// instruction: 16 * TT rows x 16 outputs, the lane's eight codes of a block
// decoded once for all rows (Q8_0: 4 v_perm + 8 byte conversions), operands
// from LDS without arithmetic (element 4i + q of a block at [q][i], so a
// lane's eight are two 16-byte reads), uniform bases and constant lane
// offsets, four multiply-adds per 16 x 16 block sums for the chain.  A
// layout that put the workgroup's activations through LDS behind a barrier
// per step ran at half the speed: 0.27 us per barrier, and 20 of 60 us in
// moves and address arithmetic.  LDS is the other part of the bound: each
// wavefront stages its own copy of the rows, and with the bank conflicts of
// kRowStride a CU's LDS is busy for about half of the 47 us of 512 rows of
// 4864 x 896, whose matrix instructions take 28.7.
//
// Measured (Q8_0, before on VALU chains -> here): 512 rows of 4864 x 896
// 88.3 -> 46.9 us (95 TFLOP/s), of 896 x 4864 143 -> 56.6, of 896 x 896
// 21.8 -> 11.9; 128 rows of 576 x 576 6.1 -> 5.3; 9 rows of 896 x 4864 14.7
// -> 13.1; one Qwen2.5 layer's seven products at 512 rows 407 -> 175.
#include <type_traits>

#include "common.hpp"
#include "exact_math.hpp"
#include "qblock.hpp"

namespace llmi_hip {

namespace {

// Up to kMaxShared products of one weight type and input size that share x
// and rows in one launch: 64-row tile t belongs to the product p with
// tile_end[p - 1] <= t < tile_end[p].  The gate_up form takes the gate matrix
// as product 0 and the up matrix as product 1 of the same tiles.
constexpr int kMaxShared = 3;
struct RowsArgs {
  const uint4* codes[kMaxShared];
  const float* scales[kMaxShared];
  const float* bias[kMaxShared];
  float* y[kMaxShared];
  int out[kMaxShared];
  int tile_end[kMaxShared];
  int mode[kMaxShared];  // a SharedEpilogue
  int count, tiles, accumulate;
  RopeCache rope;
};

enum { kProducts = 0, kGateUp = 1 };

// What becomes of a pair of results v0, v1 of one row, outputs c and c + 32
// of tile tl (c < 32): RoPE'd in place (q), RoPE'd into the KV cache (k), or
// copied into it (v).  The modes take a head size of 64, one head per tile;
// RoPE rotates elements (i, i + 32) of a head with the host tables: v[i] =
// fma(a, c, -(b * s)), v[i + 32] = fma(b, c, a * s) (kernels.cpp:122-134).
// kGateUp: v0 is the gate's, v1 the up matrix's output c: silu(gate) * up as
// the reference's MLP does after its two matmuls (kernels.cpp:148,
// transformer.cpp:288-290), whose absent bias is 0.0f: v / (1 + expf(-v)) * u
// with the exact expf.
template <int FORM>
__device__ __forceinline__ void finish_pair(const RowsArgs& g, int p, int tl, int c, int row, float v0, float v1) {
  const int o = tl * kTileRows + c, out = g.out[p], mode = g.mode[p];
  float* __restrict__ y = g.y[p];
  if (FORM == kGateUp) {
    const float gv = v0 + 0.0f, uv = v1 + 0.0f;
    if (o < out) y[static_cast<std::size_t>(row) * out + o] = gv / (1.0f + exact::expf(-gv)) * uv;
    return;
  }
  const float* bias = g.bias[p];
  v0 += bias != nullptr ? bias[o] : 0.0f;
  v1 += bias != nullptr ? bias[o + 32] : 0.0f;
  const int pos = g.rope.base + row;
  if (mode != kStoreCache) {
    const float cs = g.rope.cos_t[static_cast<std::size_t>(pos) * 32 + c];
    const float sn = g.rope.sin_t[static_cast<std::size_t>(pos) * 32 + c];
    const float a = v0, b = v1;
    v0 = __builtin_fmaf(a, cs, -(b * sn));
    v1 = __builtin_fmaf(b, cs, a * sn);
  }
  float* dst = mode == kStoreRope ? y + static_cast<std::size_t>(row) * out + o
                                  : y + (static_cast<std::size_t>(tl) * g.rope.cap + pos) * 64 + c;
  dst[0] = v0;
  dst[32] = v1;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));

// The lane's eight codes of a block as fp32: elements 4i + q, i = 0..7.
template <int TYPE>
__device__ __forceinline__ void lane_codes(const Block<TYPE>& b, int q, float* c) {
  if (TYPE == LLMI_TYPE_Q8_0) {
    // Byte q of words i and i + 1 side by side, then converted by byte.
    const std::uint32_t sel = 0x0400u + 0x0101u * static_cast<std::uint32_t>(q);
    std::uint32_t w[8];
    unpack_words<TYPE>(b, w);
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const std::uint32_t v = __builtin_amdgcn_perm(w[i + 1], w[i], sel);
      c[i] = static_cast<float>(static_cast<std::int8_t>(v & 0xFFu));
      c[i + 1] = static_cast<float>(static_cast<std::int8_t>((v >> 8) & 0xFFu));
    }
  } else {
    // Nibbles q and q + 4 of words j and j + 1: their bytes side by side,
    // the nibbles as signed bytes n - 8 (n + 0x78 never carries out of its
    // byte), then converted by byte.
    const std::uint32_t sel = 0x06040200u + 0x01010101u * static_cast<std::uint32_t>(q >> 1);
    const std::uint32_t w[4] = {b.c[0].x, b.c[0].y, b.c[0].z, b.c[0].w};
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      const std::uint32_t t = __builtin_amdgcn_perm(w[j + 1], w[j], sel) >> (4 * (q & 1));
      const std::uint32_t v = ((t & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u;
#pragma unroll
      for (int e = 0; e < 4; ++e) c[2 * j + e] = static_cast<float>(static_cast<std::int8_t>(v >> (8 * e)));
    }
  }
}

// A 32-bit lane offset that stays one: widened inside the loop (by the load's
// own addressing mode) instead of once before it, where it would cost a
// 64-bit vector addition per load.
__device__ __forceinline__ std::uint32_t opaque(std::uint32_t& v) {
  asm("" : "+v"(v));
  return v;
}

// Memory operations of the wavefront's lanes before this point come before
// those after it; no instruction.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS floats per row: rows start on 16 bytes, eight rows' reads in distinct
// banks; of a store's eight rows the first and the last share four.  Counted:
// 4.0 conflict cycles per LDS instruction, reads and stores together.
constexpr int kRowStride = 36;

// What rows look like: whole blocks; a partial last block; either, with 64-bit
// offsets: from kLongFrom elements 32 rows are out of a 32-bit one's reach.
enum { kWhole, kRagged, kLong };
constexpr int kLongFrom = 1 << 25;

// One wavefront's share of a product: TT groups of 16 rows x 16 outputs, one
// block of 32 elements at a time.  Its loads, its LDS rows and its matrix
// instructions need no other wavefront, so no barrier stands between the
// blocks.  Addresses are a wavefront-uniform base, advanced by scalar
// arithmetic, plus a constant offset per lane.
template <int TYPE, int TT, int ROWS>
struct RowsTile {
  // What a block needs from memory.
  struct Raw {
    f32x4 x[2 * TT];
    Block<TYPE> blk;
    float sc;
  };
  const GMEM char* xb;  // the wavefront's first row (uniform)
  using Offset = std::conditional_t<ROWS == kLong, std::size_t, std::uint32_t>;
  Offset xo[2 * TT];  // the lane's piece of row u * 8 + lane / 8, in bytes
  const GMEM char* cb;           // the tile's codes and scales (uniform)
  const GMEM char* sb;
  float* xs;                     // [16 * TT][kRowStride]
  int in, n, q, lane, sub;
  std::uint32_t co, so;  // lane offsets of the codes and scales, in bytes

  // Rows past the last are the last one again (computed, never stored).
  __device__ __forceinline__ void init(const float* x, int in_, int rows, int r0, int lane_, float* lds) {
    in = in_;
    lane = lane_;
    n = lane & 15;
    q = lane >> 4;
    xs = lds;
    xb = reinterpret_cast<const GMEM char*>(gmem(x + static_cast<std::size_t>(r0) * in));
#pragma unroll
    for (int u = 0; u < 2 * TT; ++u) {
      const int row = min(u * 8 + (lane >> 3), rows - 1 - r0);
      xo[u] = 4u * (static_cast<Offset>(row) * static_cast<Offset>(in) + 4u * (lane & 7));
    }
  }
  // sub_: the matrix row within the tile that lane n's codes come from.
  __device__ __forceinline__ void weights(const uint4* codes, const float* scales, int tl, int nblk, int sub_) {
    const std::size_t base = static_cast<std::size_t>(tl) * nblk * kTileRows;
    cb = reinterpret_cast<const GMEM char*>(gmem(codes) + base * Block<TYPE>::kU);
    sb = reinterpret_cast<const GMEM char*>(gmem(scales) + base);
    sub = sub_;
    co = 16u * sub;
    so = 4u * sub;
  }
  // Where the reads are ordered before the next block's stores: after them,
  // which keeps the next loads below them too, or before the stores (us at 512
  // rows, after / before: Q8_0 896 x 896 12.1 / 13.0, 4864 x 896 44.7 / 45.6,
  // Q4_0 4864 x 896 45.1 / 45.7, but 2048 x 4864 105.3 / 102.2).
  static constexpr bool kOrderAfterReads = TYPE == LLMI_TYPE_Q8_0 || TT == 2;
  // FULL: block b is known to be a whole one.
  template <bool FULL>
  __device__ __forceinline__ void load(Raw& r, int b) {
    const GMEM char* p = xb + static_cast<std::size_t>(b) * kBlock * 4;
    if (FULL || b < in / kBlock) {  // (uniform) four elements at once; a row need only be 4-byte aligned
#pragma unroll
      for (int u = 0; u < 2 * TT; ++u) {
        if constexpr (ROWS != kLong) r.x[u] = *reinterpret_cast<const GMEM f32x4a4*>(p + opaque(xo[u]));
        else r.x[u] = *reinterpret_cast<const GMEM f32x4a4*>(p + xo[u]);
      }
    } else {  // the partial block: past the row, its last element again
      const int last = in - 1 - b * kBlock - 4 * (lane & 7);
#pragma unroll
      for (int u = 0; u < 2 * TT; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          r.x[u][e] = *reinterpret_cast<const GMEM float*>(p + xo[u] + 4 * static_cast<std::ptrdiff_t>(min(e, last)));
    }
    const GMEM char* c = cb + static_cast<std::size_t>(b) * (kTileRows * 16 * Block<TYPE>::kU);
#pragma unroll
    for (int u = 0; u < Block<TYPE>::kU; ++u) {
      const u32x4 v = *reinterpret_cast<const GMEM u32x4*>(c + opaque(co) + u * (kTileRows * 16u));
      r.blk.c[u] = uint4{v.x, v.y, v.z, v.w};
    }
    r.sc = *reinterpret_cast<const GMEM float*>(sb + static_cast<std::size_t>(b) * (kTileRows * 4) + opaque(so));
  }
  // Element 4i + e of the block goes to [e][i].  Activations past `in` (the
  // last block's) become zero: the codes stored there then add nothing.
  template <bool FULL>
  __device__ __forceinline__ void stage(const Raw& r, int b) const {
    if (!kOrderAfterReads) wave_order();
    float* dst = xs + (lane >> 3) * kRowStride + (lane & 7);
    if (FULL || b < in / kBlock) {  // (uniform)
#pragma unroll
      for (int u = 0; u < 2 * TT; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[u * 8 * kRowStride + e * 8] = r.x[u][e];
    } else {
      const int left = in - b * kBlock - 4 * (lane & 7);
#pragma unroll
      for (int u = 0; u < 2 * TT; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[u * 8 * kRowStride + e * 8] = e < left ? r.x[u][e] : 0.0f;
    }
  }
  // The lane's operands, which other lanes of the wavefront staged.  A
  // wavefront's LDS operations execute in order, so no wait stands around
  // the reads, but per lane the addresses differ from the stores': the
  // compiler is told to keep the order too.
  __device__ __forceinline__ void fragments(f32x4 (&a)[TT][2]) const {
    wave_order();
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      const f32x4* src = reinterpret_cast<const f32x4*>(xs + (tt * 16 + n) * kRowStride + q * 8);
      a[tt][0] = src[0];
      a[tt][1] = src[1];
    }
    if (kOrderAfterReads) wave_order();
  }
};

// A block's operands in registers, and its sums.
template <int TT>
struct RowsOps {
  f32x4 a[TT][2];
  float c[8];
  float sc;
  f32x4 part[TT];
  // The sums over the block's first 4 * steps elements.
  __device__ __forceinline__ void products(int steps) {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) part[tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i < steps) {
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
          part[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[tt][i >> 2][i & 3], c[i], part[tt], 0, 0, 0);
      }
    }
  }
};

// Where a workgroup's output groups lie.  kProducts: workgroup column
// blockIdx.x is a 64-row tile, group w its rows 16 w ..; kGateUp: half a
// tile, groups 0 and 1 of the gate matrix and the same rows of the up
// matrix as groups 2 and 3.
template <int FORM>
struct RowsPlace {
  int p, tl;
  __device__ __forceinline__ explicit RowsPlace(const RowsArgs& g) {
    const int t = static_cast<int>(FORM == kGateUp ? blockIdx.x >> 1 : blockIdx.x);
    p = 0;
    if (FORM == kProducts)
      while (p + 1 < g.count && t >= g.tile_end[p]) ++p;
    tl = p == 0 ? t : t - g.tile_end[p - 1];
  }
  __device__ __forceinline__ int column(int group, int n) const {
    return (FORM == kGateUp ? static_cast<int>(blockIdx.x & 1) * 32 + (group & 1) * 16 : group * 16) + n;
  }
  template <class Tile>
  __device__ __forceinline__ void bind(Tile& t, const uint4* codes, const float* scales, const RowsArgs& g, int nblk,
                                       int group) const {
    const int m = FORM == kGateUp ? group >> 1 : p;
    if (m != 0) {
      codes = g.codes[m];
      scales = g.scales[m];
    }
    t.weights(codes, scales, tl, nblk, column(group, t.n));
  }
  // Whether group w + 2's results are needed beside group w's.
  __device__ __forceinline__ bool pairs(const RowsArgs& g) const {
    return FORM == kGateUp || g.mode[p] != kStorePlain;
  }
};

// One output of one row as computed, or added to y.
__device__ __forceinline__ void store_one(const RowsArgs& g, int p, int o, int row, float v) {
  if (o >= g.out[p]) return;
  const float* bias = g.bias[p];
  float* dst = g.y[p] + static_cast<std::size_t>(row) * g.out[p] + o;
  v += bias != nullptr ? bias[o] : 0.0f;
  *dst = g.accumulate ? *dst + v : v;
}

// Launches with enough tiles for the GPU: the workgroup's four wavefronts
// share the rows' cache lines, each runs the chain over the blocks in
// registers.  A block's loads are issued before the matrix instructions of
// the block before it; the previous block's sums are chained while the LDS
// reads of this one's operands are under way.
template <int TYPE, int FORM, int TT, int ROWS>
__global__ void __launch_bounds__(256, 2)
    qgemm_rows(const uint4* __restrict__ codes, const float* __restrict__ scales, const float* __restrict__ x, int in,
               int nblk, int rows, RowsArgs g) {
  __shared__ __attribute__((aligned(16))) float xs[4][16 * TT * kRowStride];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r0 = blockIdx.y * 16 * TT;
  const RowsPlace<FORM> at(g);
  using Tile = RowsTile<TYPE, TT, ROWS>;
  Tile t;
  t.init(x, in, rows, r0, lane, xs[wave]);
  at.bind(t, codes, scales, g, nblk, wave);
  f32x4 acc[TT];
  RowsOps<TT> o;
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) acc[tt] = o.part[tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  o.sc = 0.0f;  // block -1: no sums, scale 0: its chain step leaves +0
  const auto chain = [&]() {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[tt][v] = __builtin_fmaf(o.part[tt][v], o.sc, acc[tt][v]);
  };
  typename Tile::Raw raw;
  const auto operands = [&](int b, auto full) {
    t.template stage<decltype(full)::value>(raw, b);
    t.fragments(o.a);
    lane_codes<TYPE>(raw.blk, t.q, o.c);
    chain();
    o.sc = raw.sc;
  };
  constexpr std::true_type kFull;
  // The whole blocks but, before a partial one, the last: each loads the next
  // (the last of a row without a partial block itself again).  The partial
  // block's element loads stand outside the loop, and its steps past `in` are
  // left out: 24000 x 40 Q8_0 at 424 rows 41 -> 31 us, 8192 x 1003 at 512
  // rows (with 32-bit offsets, as whole rows have) 103 -> 83.
  const int loop = ROWS == kWhole ? nblk : nblk - 2;
  t.template load<ROWS == kWhole>(raw, 0);
  for (int b = 0; b < loop; ++b) {
    operands(b, kFull);
    t.template load<true>(raw, ROWS == kWhole ? min(b + 1, nblk - 1) : b + 1);
    __builtin_amdgcn_sched_barrier(0);
    o.products(8);
  }
  if (ROWS != kWhole) {
    if (nblk > 1) {
      operands(nblk - 2, kFull);
      t.template load<false>(raw, nblk - 1);
      __builtin_amdgcn_sched_barrier(0);
      o.products(8);
    }
    operands(nblk - 1, std::false_type{});  // only its elements' steps
    o.products((in - (nblk - 1) * kBlock + 3) / 4);
  }
  chain();
  if (!at.pairs(g)) {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = r0 + tt * 16 + 4 * t.q + v;
        if (row < rows) store_one(g, at.p, at.tl * kTileRows + t.sub, row, acc[tt][v]);
      }
    return;
  }
  // (uniform) Groups 2 and 3 hand their results to groups 0 and 1.
  __syncthreads();
  float* ex = xs[wave & 1];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (wave >= 2) ex[(tt * 4 + v) * 64 + lane] = acc[tt][v];
  __syncthreads();
  if (wave >= 2) return;
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = r0 + tt * 16 + 4 * t.q + v;
      if (row < rows) finish_pair<FORM>(g, at.p, at.tl, t.sub, row, acc[tt][v], ex[(tt * 4 + v) * 64 + lane]);
    }
}

// Launches with few tiles: KS wavefronts share a group's 16 rows x 16
// outputs; wavefront w takes blocks w, w + KS, ..., U of them in flight.  A
// round of KS * U blocks puts its sums and scales in LDS, and after a
// barrier wavefront v < 4 chains accumulator register v over the round's
// blocks in order.  G = 2: the workgroup holds both groups of a pair.
template <int TYPE, int FORM, int G, int KS, int U, int ROWS>
__global__ void __launch_bounds__(64 * G * KS)
    qgemm_rows_split(const uint4* __restrict__ codes, const float* __restrict__ scales, const float* __restrict__ x,
                     int in, int nblk, int rows, RowsArgs g) {
  constexpr int RB = KS * U;
  __shared__ __attribute__((aligned(16))) float xs[G * KS][16 * kRowStride];
  __shared__ float ps[G][RB][4][64];
  __shared__ float ss[G][RB][16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = wave / KS, kg = wave % KS;
  const int r0 = blockIdx.z * 16;
  const RowsPlace<FORM> at(g);
  using Tile = RowsTile<TYPE, 1, ROWS>;
  Tile t;
  t.init(x, in, rows, r0, lane, xs[wave]);
  at.bind(t, codes, scales, g, nblk, static_cast<int>(blockIdx.y) + 2 * half);
  float acc = 0.0f;
  typename Tile::Raw raw[U];
#pragma unroll
  for (int u = 0; u < U; ++u) t.template load<ROWS == kWhole>(raw[u], min(u * KS + kg, nblk - 1));
  for (int b0 = 0; b0 < nblk; b0 += RB) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int b = b0 + u * KS + kg;
      if (b < nblk) {
        RowsOps<1> o;
        t.template stage<ROWS == kWhole>(raw[u], b);
        t.fragments(o.a);
        lane_codes<TYPE>(raw[u].blk, t.q, o.c);
        if (t.q == 0) ss[half][u * KS + kg][t.n] = raw[u].sc;
        if (b + RB < nblk) t.template load<ROWS == kWhole>(raw[u], b + RB);
        o.products(8);
#pragma unroll
        for (int v = 0; v < 4; ++v) ps[half][u * KS + kg][v][lane] = o.part[0][v];
      }
    }
    __syncthreads();
    if (kg < 4) {
      const int nb = min(RB, nblk - b0);
      const float* pp = &ps[half][0][kg][lane];
      const float* sp = &ss[half][0][t.n];
      int i = 0;
      for (; i + 8 <= nb; i += 8) {
        float pv[8], sv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          pv[u] = pp[(i + u) * 4 * 64];
          sv[u] = sp[(i + u) * 16];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) acc = __builtin_fmaf(pv[u], sv[u], acc);
      }
      for (; i < nb; ++i) acc = __builtin_fmaf(pp[i * 4 * 64], sp[i * 16], acc);
    }
    if (G == 2 || b0 + RB < nblk) __syncthreads();
  }
  const int row = r0 + 4 * t.q + kg;
  if (G == 1 || !at.pairs(g)) {
    if (kg < 4 && row < rows) store_one(g, at.p, at.tl * kTileRows + t.sub, row, acc);
    return;
  }
  if (half == 1 && kg < 4) ps[0][0][kg][lane] = acc;
  __syncthreads();
  if (half == 0 && kg < 4 && row < rows)
    finish_pair<FORM>(g, at.p, at.tl, t.sub, row, acc, ps[0][0][kg][lane]);
}

template <int TYPE, int FORM, int TT>
void launch_tiles(const RowsArgs& g, const float* x, int in, int nblk, int rows, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(g.tiles) * (FORM == kGateUp ? 2 : 1),
                  static_cast<unsigned>(ceil_div(rows, 16 * TT)));
  if (in % kBlock == 0) qgemm_rows<TYPE, FORM, TT, kWhole><<<grid, 256, 0, s>>>(g.codes[0], g.scales[0], x, in, nblk, rows, g);
  else qgemm_rows<TYPE, FORM, TT, kRagged><<<grid, 256, 0, s>>>(g.codes[0], g.scales[0], x, in, nblk, rows, g);
}
// 32-bit offsets measure 2 to 6 % slower in the split form of ragged rows
// (320 x 1003 of Q4_0 at 1000 rows 14.9 us against 14.0), so it takes kLong's.
template <int TYPE, int FORM, int G, int KS, int U>
void launch_split_blocks(const RowsArgs& g, const float* x, int in, int nblk, int rows, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(g.tiles) * (FORM == kGateUp ? 2 : 1), 4 / G,
                  static_cast<unsigned>(ceil_div(rows, 16)));
  if (in % kBlock == 0 && in < kLongFrom)
    qgemm_rows_split<TYPE, FORM, G, KS, U, kWhole><<<grid, 64 * G * KS, 0, s>>>(g.codes[0], g.scales[0], x, in, nblk, rows, g);
  else
    qgemm_rows_split<TYPE, FORM, G, KS, U, kLong><<<grid, 64 * G * KS, 0, s>>>(g.codes[0], g.scales[0], x, in, nblk, rows, g);
}

template <int TYPE, int FORM>
void launch_form(const RowsArgs& g, const float* x, std::size_t in_, std::size_t nblk_, std::size_t rows_,
                 hipStream_t s) {
  const int in = static_cast<int>(in_), nblk = static_cast<int>(nblk_), rows = static_cast<int>(rows_);
  const std::size_t groups = static_cast<std::size_t>(g.tiles) * (FORM == kGateUp ? 8 : 4);
  // By the number of 16 x 16 tiles against the GPU's 1024 SIMDs (times in us,
  // Q8_0).  From 8192: 32 rows per wavefront (4864 x 896 at 512 rows 45.4,
  // 16 rows 47.5; 151936 x 896 at 64 rows 157, 16 rows 176), unless a last
  // half-empty 32 costs more than that saves: few 16-row groups, an odd number
  // of them (151936 x 896 at 9 rows 80.4, 16 rows per wavefront 50.6; at 40
  // 149, 128; 49152 x 576 at 80 50.8, 46.7; but at 176, 11 groups, 98.3,
  // 103.0).  From about 1.4 wavefronts per SIMD: 16 rows, blocks
  // chained in registers (896 x 896 at 512 rows 12.9, split over 8
  // wavefronts 15.1); rows of more than 32 blocks from 2.5 (at 1.75, 896 x
  // 4864: split 53.8, not 56.6), pairs, whose split has half the wavefronts
  // per group, from 0.5.  Below, split: over 8 wavefronts (4864 x 896 at 64
  // rows 10.4, 16 wavefronts 13.6), over 16 when there are at most 256 tiles
  // (896 x 4864 at 64 rows 13.6, 8 wavefronts 15.0).  A Q8_0 wavefront of the
  // 8 has one block in flight: the other waves cover its loads, and two cost
  // registers (896 x 4864 at 256 and 512 rows 32.1 and 53.8, two blocks 35.9
  // and 57.4); Q4_0's smaller blocks measure the same or better in twos (576
  // x 1536 at 256 rows 10.2, one block 10.4).
  const std::size_t groups16 = ceil_div(rows_, 16);
  const std::size_t units = groups * groups16;
  const bool pairs = FORM == kGateUp || g.mode[0] != kStorePlain;
  const bool by32 = groups16 % 2 == 0 || groups16 > 8;
  const bool split = in >= kLongFrom;  // too few tiles fit memory for the others
  if (units >= 8192 && by32 && !split) launch_tiles<TYPE, FORM, 2>(g, x, in, nblk, rows, s);
  else if (units >= (pairs ? 512u : nblk <= 32 ? 1408u : 2560u) && !split) launch_tiles<TYPE, FORM, 1>(g, x, in, nblk, rows, s);
  else if (pairs) launch_split_blocks<TYPE, FORM, 2, 4, 2>(g, x, in, nblk, rows, s);
  else if (units > 256) launch_split_blocks<TYPE, FORM, 1, 8, TYPE == LLMI_TYPE_Q8_0 ? 1 : 2>(g, x, in, nblk, rows, s);
  else launch_split_blocks<TYPE, FORM, 1, 16, 2>(g, x, in, nblk, rows, s);
}

int check_rows(const DeviceMatrix& m, std::size_t rows) {
  LLMI_REQUIRE(m.in > 0, "matmul: in must be positive");
  LLMI_REQUIRE(m.in <= 0x7FFFFFFFu && m.out <= 0x7FFFFFFFu, "matmul: shape too large");
  LLMI_REQUIRE(ceil_div(rows, 8) <= 65535, "matmul: too many input rows for one launch");
  return LLMI_OK;
}

}  // namespace

int launch_rows(const DeviceMatrix& m, const float* x, std::size_t rows, const float* bias, float* y, hipStream_t s,
                bool accumulate) {
  if (int rc = check_rows(m, rows)) return rc;
  RowsArgs g{};
  g.codes[0] = reinterpret_cast<const uint4*>(m.codes);
  g.scales[0] = m.scales;
  g.bias[0] = bias;
  g.y[0] = y;
  g.out[0] = static_cast<int>(m.out);
  g.tile_end[0] = g.tiles = static_cast<int>(m.ntiles);
  g.mode[0] = kStorePlain;
  g.count = 1;
  g.accumulate = accumulate ? 1 : 0;
  if (m.type == LLMI_TYPE_Q8_0) launch_form<LLMI_TYPE_Q8_0, kProducts>(g, x, m.in, m.nblk, rows, s);
  else launch_form<LLMI_TYPE_Q4_0, kProducts>(g, x, m.in, m.nblk, rows, s);
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

int launch_gate_up_silu(const DeviceMatrix& gate, const DeviceMatrix& up, const float* x, std::size_t rows,
                        float* y, hipStream_t s, bool* fused) {
  *fused = false;
  if (rows <= 8 || gate.type == LLMI_TYPE_F32 || gate.type != up.type || gate.in != up.in || gate.out != up.out ||
      gate.out == 0)
    return LLMI_OK;
  if (int rc = check_rows(gate, rows)) return rc;
  LLMI_REQUIRE(x != nullptr && y != nullptr, "gate_up: null pointer");
  RowsArgs g{};
  const DeviceMatrix* ms[2] = {&gate, &up};
  for (int i = 0; i < 2; ++i) {
    g.codes[i] = reinterpret_cast<const uint4*>(ms[i]->codes);
    g.scales[i] = ms[i]->scales;
  }
  g.y[0] = y;
  g.out[0] = static_cast<int>(gate.out);
  g.tiles = static_cast<int>(gate.ntiles);
  if (gate.type == LLMI_TYPE_Q8_0) launch_form<LLMI_TYPE_Q8_0, kGateUp>(g, x, gate.in, gate.nblk, rows, s);
  else launch_form<LLMI_TYPE_Q4_0, kGateUp>(g, x, gate.in, gate.nblk, rows, s);
  LLMI_TRY_HIP(hipGetLastError());
  *fused = true;
  return LLMI_OK;
}

int launch_matmul_shared(const DeviceMatrix* const* ms, const float* const* biases, float* const* ys, int count,
                         const float* x, std::size_t rows, hipStream_t s, const RopeCache* rope, bool* roped) {
  if (roped != nullptr) *roped = false;
  LLMI_REQUIRE(count >= 1 && count <= kMaxShared, "matmul_shared: 1..3 products");
  std::size_t tiles = 0;
  bool grouped = count > 1 && rows > 8;
  for (int i = 0; i < count && grouped; ++i) {
    const DeviceMatrix& m = *ms[i];
    grouped = m.type != LLMI_TYPE_F32 && m.type == ms[0]->type && m.in == ms[0]->in && m.out > 0;
    tiles += m.ntiles;
  }
  if (!grouped || tiles > 0x1FFFFFFFu) {
    for (int i = 0; i < count; ++i)
      if (int rc = launch_matmul(*ms[i], x, rows, biases[i], ys[i], s)) return rc;
    return LLMI_OK;
  }
  if (int rc = check_rows(*ms[0], rows)) return rc;
  LLMI_REQUIRE(x != nullptr, "matmul_shared: null x");
  RowsArgs g{};
  int end = 0;
  for (int i = 0; i < count; ++i) {
    LLMI_REQUIRE(ys[i] != nullptr, "matmul_shared: null y");
    g.codes[i] = reinterpret_cast<const uint4*>(ms[i]->codes);
    g.scales[i] = ms[i]->scales;
    g.bias[i] = biases[i];
    g.y[i] = ys[i];
    g.out[i] = static_cast<int>(ms[i]->out);
    end += static_cast<int>(ms[i]->ntiles);
    g.tile_end[i] = end;
    g.mode[i] = kStorePlain;
  }
  g.count = count;
  g.tiles = end;
  // RoPE and the cache writes ride along for q, k, v of head size 64.
  if (rope != nullptr && roped != nullptr && count == 3 && ms[0]->out % 64 == 0 && ms[1]->out % 64 == 0 &&
      ms[2]->out % 64 == 0) {
    g.rope = *rope;
    g.mode[0] = kStoreRope;
    g.mode[1] = kStoreRopeCache;
    g.mode[2] = kStoreCache;
    g.y[1] = rope->kc;
    g.y[2] = rope->vc;
    *roped = true;
  }
  if (ms[0]->type == LLMI_TYPE_Q8_0) launch_form<LLMI_TYPE_Q8_0, kProducts>(g, x, ms[0]->in, ms[0]->nblk, rows, s);
  else launch_form<LLMI_TYPE_Q4_0, kProducts>(g, x, ms[0]->in, ms[0]->nblk, rows, s);
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

}  // namespace llmi_hip
