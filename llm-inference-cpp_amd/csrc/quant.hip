// Block quantizer (fp32 -> Q8_0 / Q4_0), the planar <-> tiled re-layout, and
// the row dequantizer (embedding gather) for gfx950.
//
// The quantizer restates src/model/quant.cpp:36-102: the block scan, the
// scale and every code have the reference's values (IEEE fp32 divide for the
// scale; the codes as its IEEE fp64 divide and round-half-away-from-zero give
// them), so the packed bytes are bit-identical.  Load-time work: it reads
// each weight once (4 B) and writes 0.625 / 1.125 B, so it is HBM-bound.
#include "common.hpp"

namespace llmi_hip {
namespace {

// C lround: round half away from zero.  |q| <= 128 here (|v| <= amax), so
// q - trunc(q) is exact.
__device__ __forceinline__ int round_half_away(double q) {
  const double t = trunc(q);
  const double frac = q - t;
  double r = t;
  if (frac >= 0.5) r = t + 1.0;
  if (frac <= -0.5) r = t - 1.0;
  return static_cast<int>(r);
}

// The value of a lane's partner within its group of eight lanes: the lane
// with the lowest bit flipped, the second bit flipped, or (all four lanes of
// a quad holding one value) a lane of the group's other quad.
template <int CTRL>
__device__ __forceinline__ std::uint32_t partner(std::uint32_t v) {
  return static_cast<std::uint32_t>(
      __builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xF, 0xF, true));
}
constexpr int kFlip1 = 0xB1, kFlip2 = 0x4E, kOtherQuad = 0x141;  // quad_perm, quad_perm, row_half_mirror

// The reference's code lround(double(v) / double(d)) (quant.cpp:85), without
// the double division where its rounding is not in doubt.  r is 1 / d within
// an ulp, so |v * r| is within 2^-15 of |v / d| <= 128; unless it lies within
// kDoubt of a half it rounds to the same integer.  (The double quotient is a
// half exactly when the real one is: v / d - (n + 1/2) is 0 or, for fp32 v
// and d and n < 128, at least 2^-25.)
constexpr float kDoubt = 0x1p-13f;
__device__ __forceinline__ int code_of_value(float v, float d, float r, bool fast) {
  const float a = v * r;
  const float m = __builtin_fabsf(a) + 0.5f;
  const float f = __builtin_floorf(m);
  const float frac = m - f;
  if (fast && frac >= kDoubt && frac <= 1.0f - kDoubt) {
    const int n = static_cast<int>(f);
    return a < 0.0f ? -n : n;
  }
  return round_half_away(static_cast<double>(v) / static_cast<double>(d));
}

typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));

// Eight lanes per (row, block), four weights each: a block is one coalesced
// 128-byte read, its largest weight three lane exchanges.  The blocks come in
// the order of the output -- planar: by row; tiled: the 64 rows of a tile one
// after another, block by block -- so that the codes of consecutive groups
// are neighbours.  Bound: HBM.  Measured on the 151936 x 896 matrix, against
// one thread per block, whose 128-byte-strided loads and 32 double divisions
// it replaces: Q4_0 355 -> 125 us (5.0 TB/s).
constexpr int kQuantItems = 4;  // blocks per group, their loads issued together

template <int TYPE, bool PLANAR>
__global__ void __launch_bounds__(256) quantize_blocks(const float* __restrict__ w, std::size_t out, int in, int nblk,
                                                       std::uint8_t* __restrict__ codes, float* __restrict__ scales) {
  const int tid = threadIdx.x, e0 = 4 * (tid & 7), group = tid >> 3;
  const bool whole = in % kBlock == 0;
  float v[kQuantItems][4];
  std::size_t row[kQuantItems];
  int block[kQuantItems];
  // Blocks past the last are not stored; they read the last row's.
#pragma unroll
  for (int u = 0; u < kQuantItems; ++u) {
    const std::size_t item = (static_cast<std::size_t>(blockIdx.x) * kQuantItems + u) * 32 + group;
    if (PLANAR) {
      row[u] = item / nblk;
      block[u] = static_cast<int>(item - row[u] * nblk);
    } else {
      const std::size_t slot = (static_cast<std::size_t>(blockIdx.x) * kQuantItems + u) / 2;  // (uniform)
      row[u] = slot / nblk * kTileRows + (item & (kTileRows - 1));
      block[u] = static_cast<int>(slot % nblk);
    }
    const std::size_t r = row[u] < out ? row[u] : out - 1;
    const float* src = w + r * static_cast<std::size_t>(in) + block[u] * kBlock;
    if (whole) {
      const f32x4a4 x = *reinterpret_cast<const f32x4a4*>(src + e0);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[u][e] = x[e];
    } else {
      const int n = in - block[u] * kBlock;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = src[min(e0 + e, n - 1)];
        v[u][e] = e0 + e < n ? x : 0.0f;
      }
    }
  }
#pragma unroll
  for (int u = 0; u < kQuantItems; ++u) {
    // quant.cpp:54-62: the first of the largest |v| (strict '>': NaN never).
    float peak = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (__builtin_fabsf(v[u][e]) > __builtin_fabsf(peak)) peak = v[u][e];
    const auto merge = [&](float other, bool lower) {
      const float a = __builtin_fabsf(peak), b = __builtin_fabsf(other);
      if (b > a || (b == a && lower)) peak = other;
    };
    merge(__uint_as_float(partner<kFlip1>(__float_as_uint(peak))), (tid & 1) != 0);
    merge(__uint_as_float(partner<kFlip2>(__float_as_uint(peak))), (tid & 2) != 0);
    merge(__uint_as_float(partner<kOtherQuad>(__float_as_uint(peak))), (tid & 4) != 0);
    float d = TYPE == LLMI_TYPE_Q4_0 ? peak / -8.0f : __builtin_fabsf(peak) / 127.0f;  // quant.cpp:63-80
    if (d == 0.0f) d = 1.0f;                                                           // quant.cpp:81
    const float size = __builtin_fabsf(d);
    const bool fast = size >= 0x1p-100f && size <= 0x1p100f;  // 1 / d and v / d are normal numbers
    const float r = __builtin_amdgcn_rcpf(d);
    const int left = whole ? kBlock : in - block[u] * kBlock - e0;
    std::uint32_t word = 0u;  // the four codes, in the reference's byte order
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int q = min(max(code_of_value(v[u][e], d, r, fast), TYPE == LLMI_TYPE_Q4_0 ? -8 : -127),
                        TYPE == LLMI_TYPE_Q4_0 ? 7 : 127);
      const std::uint32_t c = TYPE == LLMI_TYPE_Q8_0 ? static_cast<std::uint32_t>(q) & 0xFFu
                                                     : static_cast<std::uint32_t>(q + 8);
      word |= (e < left ? c : 0u) << ((TYPE == LLMI_TYPE_Q8_0 ? 8 : 4) * e);
    }
    // Q4_0: two lanes make a word, stored by the even one.
    if (TYPE == LLMI_TYPE_Q4_0) word |= partner<kFlip1>(word) << 16;
    if (row[u] >= out) continue;
    const bool first = (tid & 7) == 0;
    if (PLANAR) {
      const std::size_t rb = TYPE == LLMI_TYPE_Q4_0 ? (static_cast<std::size_t>(in) + 1) / 2 : static_cast<std::size_t>(in);
      std::uint8_t* dst = codes + row[u] * rb + (block[u] * kBlock + e0) / (TYPE == LLMI_TYPE_Q4_0 ? 2 : 1);
      if (whole && reinterpret_cast<std::uintptr_t>(codes) % 4 == 0) {
        if (TYPE == LLMI_TYPE_Q8_0 || (tid & 1) == 0) *reinterpret_cast<std::uint32_t*>(dst) = word;
      } else {
        const int nbytes = TYPE == LLMI_TYPE_Q4_0 ? (min(left, 4) + 1) / 2 : min(left, 4);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j < nbytes) dst[j] = static_cast<std::uint8_t>(word >> (8 * j));
      }
      if (first) scales[row[u] * nblk + block[u]] = d;
    } else {
      const std::size_t item = (static_cast<std::size_t>(blockIdx.x) * kQuantItems + u) * 32 + group;  // slot * 64 + row
      if (TYPE == LLMI_TYPE_Q4_0) {
        if ((tid & 1) == 0) *reinterpret_cast<std::uint32_t*>(codes + item * 16 + e0 / 2) = word;
      } else {
        const std::size_t slot = item / kTileRows, lane = item % kTileRows;
        *reinterpret_cast<std::uint32_t*>(codes + ((slot * 2 + e0 / 16) * kTileRows + lane) * 16 + e0 % 16) = word;
      }
      if (first) scales[item] = d;
    }
  }
}

// Planar (reference) layout -> tiled device layout, one block per thread.
template <int TYPE>
__global__ void __launch_bounds__(256) planar_to_tiled(const std::uint8_t* __restrict__ pdata,
                                                       const float* __restrict__ pscales, std::size_t out, int in,
                                                       int nblk, std::uint8_t* __restrict__ tcodes,
                                                       float* __restrict__ tscales) {
  const std::size_t gid = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= out * static_cast<std::size_t>(nblk)) return;
  const std::size_t r = gid / nblk;
  const int b = static_cast<int>(gid % nblk);
  const int first = b * kBlock;
  const int n = min(kBlock, in - first);
  const std::size_t rb = TYPE == LLMI_TYPE_Q4_0 ? (static_cast<std::size_t>(in) + 1) / 2 : static_cast<std::size_t>(in);
  const std::uint8_t* src = pdata + r * rb + (TYPE == LLMI_TYPE_Q4_0 ? first / 2 : first);
  const int nbytes = TYPE == LLMI_TYPE_Q4_0 ? (n + 1) / 2 : n;
  constexpr int kBytes = TYPE == LLMI_TYPE_Q4_0 ? 16 : 32;
  std::uint32_t word[kBytes / 4];
#pragma unroll
  for (int k = 0; k < kBytes / 4; ++k) word[k] = 0u;
#pragma unroll
  for (int j = 0; j < kBytes; ++j)
    if (j < nbytes) word[j / 4] |= static_cast<std::uint32_t>(src[j]) << (8 * (j % 4));
  const std::size_t tile = r / kTileRows;
  const int lane = static_cast<int>(r % kTileRows);
  const std::size_t slot = tile * nblk + b;
  uint4* dst = reinterpret_cast<uint4*>(tcodes);
  if (TYPE == LLMI_TYPE_Q4_0) {
    dst[slot * kTileRows + lane] = make_uint4(word[0], word[1], word[2], word[3]);
  } else {
    dst[(slot * 2 + 0) * kTileRows + lane] = make_uint4(word[0], word[1], word[2], word[3]);
    dst[(slot * 2 + 1) * kTileRows + lane] = make_uint4(word[4], word[5], word[6], word[7]);
  }
  tscales[slot * kTileRows + lane] = pscales[r * nblk + b];
}

// IEEE binary16 -> binary32, exactly, as integer operations (src/model/
// safetensors.cpp:249-273 maps the same way: subnormals normalised, the
// infinities and NaNs keep their payload bits unchanged).
__device__ __forceinline__ float half_bits_to_float(std::uint32_t h) {
  const std::uint32_t sign = (h & 0x8000u) << 16;
  const std::uint32_t e = (h >> 10) & 0x1Fu;
  const std::uint32_t m = h & 0x3FFu;
  std::uint32_t bits;
  if (e == 0) {
    if (m == 0) {
      bits = sign;
    } else {
      const int top = 31 - __builtin_clz(m);  // leading one of the mantissa, 0..9: value 2^(top - 24) * 1.f
      bits = sign | (static_cast<std::uint32_t>(top + 103) << 23) | ((m << (23 - top)) & 0x7FFFFFu);
    }
  } else if (e == 0x1F) {
    bits = sign | 0x7F800000u | (m << 13);
  } else {
    bits = sign | ((e + 112u) << 23) | (m << 13);
  }
  return __uint_as_float(bits);
}

// GGUF (ggml) blocks -> tiled device layout, one block per thread
// (gguf.cpp:577-640, to_quantized).  A ggml block is {fp16 d; codes}:
// Q8_0 34 bytes, its 32 signed codes in element order (copied as they are);
// Q4_0 18 bytes, byte j holding element j in the low nibble and element
// j + 16 in the high nibble, re-packed here into this library's pairs of
// neighbours (byte k: element 2k low, 2k + 1 high).  Blocks start 2-byte
// aligned (both sizes are even), so they are read as 16-bit words.
template <int TYPE>
__global__ void __launch_bounds__(256) gguf_to_tiled(const std::uint16_t* __restrict__ raw, std::size_t out, int nblk,
                                                     std::uint8_t* __restrict__ tcodes,
                                                     float* __restrict__ tscales) {
  const std::size_t gid = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= out * static_cast<std::size_t>(nblk)) return;
  const std::size_t r = gid / nblk;
  const int b = static_cast<int>(gid % nblk);
  constexpr int kHalfwords = TYPE == LLMI_TYPE_Q4_0 ? 9 : 17;
  const std::uint16_t* src = raw + gid * kHalfwords;
  std::uint32_t word[TYPE == LLMI_TYPE_Q4_0 ? 4 : 8];
  if (TYPE == LLMI_TYPE_Q8_0) {
#pragma unroll
    for (int k = 0; k < 8; ++k)
      word[k] = static_cast<std::uint32_t>(src[1 + 2 * k]) | (static_cast<std::uint32_t>(src[2 + 2 * k]) << 16);
  } else {
    std::uint8_t q[16];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      q[2 * k] = static_cast<std::uint8_t>(src[1 + k] & 0xFFu);
      q[2 * k + 1] = static_cast<std::uint8_t>(src[1 + k] >> 8);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) word[k] = 0u;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int e0 = 2 * k, e1 = 2 * k + 1;  // elements of engine byte k
      const std::uint32_t n0 = e0 < 16 ? (q[e0] & 0xFu) : (q[e0 - 16] >> 4);
      const std::uint32_t n1 = e1 < 16 ? (q[e1] & 0xFu) : (q[e1 - 16] >> 4);
      word[k / 4] |= (n0 | (n1 << 4)) << (8 * (k % 4));
    }
  }
  const std::size_t tile = r / kTileRows;
  const int lane = static_cast<int>(r % kTileRows);
  const std::size_t slot = tile * nblk + b;
  uint4* dst = reinterpret_cast<uint4*>(tcodes);
  if (TYPE == LLMI_TYPE_Q4_0) {
    dst[slot * kTileRows + lane] = make_uint4(word[0], word[1], word[2], word[3]);
  } else {
    dst[(slot * 2 + 0) * kTileRows + lane] = make_uint4(word[0], word[1], word[2], word[3]);
    dst[(slot * 2 + 1) * kTileRows + lane] = make_uint4(word[4], word[5], word[6], word[7]);
  }
  tscales[slot * kTileRows + lane] = half_bits_to_float(src[0]);
}

// Tiled device layout -> planar (reference) layout, one block per thread.
template <int TYPE>
__global__ void __launch_bounds__(256) tiled_to_planar(const std::uint8_t* __restrict__ tcodes,
                                                       const float* __restrict__ tscales, std::size_t out, int in,
                                                       int nblk, std::uint8_t* __restrict__ pdata,
                                                       float* __restrict__ pscales) {
  const std::size_t gid = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= out * static_cast<std::size_t>(nblk)) return;
  const std::size_t r = gid / nblk;
  const int b = static_cast<int>(gid % nblk);
  const int first = b * kBlock;
  const int n = min(kBlock, in - first);
  const std::size_t tile = r / kTileRows;
  const int lane = static_cast<int>(r % kTileRows);
  const std::size_t slot = tile * nblk + b;
  const uint4* src = reinterpret_cast<const uint4*>(tcodes);
  std::uint32_t word[8];
  uint4 a = TYPE == LLMI_TYPE_Q4_0 ? src[slot * kTileRows + lane] : src[(slot * 2 + 0) * kTileRows + lane];
  word[0] = a.x; word[1] = a.y; word[2] = a.z; word[3] = a.w;
  if (TYPE == LLMI_TYPE_Q8_0) {
    const uint4 c = src[(slot * 2 + 1) * kTileRows + lane];
    word[4] = c.x; word[5] = c.y; word[6] = c.z; word[7] = c.w;
  }
  const std::size_t rb = TYPE == LLMI_TYPE_Q4_0 ? (static_cast<std::size_t>(in) + 1) / 2 : static_cast<std::size_t>(in);
  std::uint8_t* dst = pdata + r * rb + (TYPE == LLMI_TYPE_Q4_0 ? first / 2 : first);
  const int nbytes = TYPE == LLMI_TYPE_Q4_0 ? (n + 1) / 2 : n;
#pragma unroll
  for (int j = 0; j < (TYPE == LLMI_TYPE_Q4_0 ? 16 : 32); ++j)
    if (j < nbytes) dst[j] = static_cast<std::uint8_t>(word[j / 4] >> (8 * (j % 4)));
  pscales[r * nblk + b] = tscales[slot * kTileRows + lane];
}

// quant.cpp:104-117 on the tiled layout: dst[t][k] = code * scale (one
// rounding), for token t's row ids[t].  grid.y = token.
template <int TYPE>
__global__ void __launch_bounds__(256) dequantize_rows(const std::uint8_t* __restrict__ tcodes,
                                                       const float* __restrict__ tscales, int in, int nblk,
                                                       const std::int32_t* __restrict__ ids,
                                                       float* __restrict__ dst) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= in) return;
  const std::size_t row = static_cast<std::size_t>(ids[blockIdx.y]);
  const std::size_t tile = row / kTileRows;
  const int lane = static_cast<int>(row % kTileRows);
  const int b = k / kBlock;
  const int i = k % kBlock;
  const std::size_t slot = tile * nblk + b;
  float code;
  if (TYPE == LLMI_TYPE_Q4_0) {
    const std::uint8_t byte = tcodes[(slot * kTileRows + lane) * 16 + i / 2];
    const int nib = (i & 1) ? (byte >> 4) : (byte & 0xF);
    code = static_cast<float>(nib - 8);
  } else {
    const std::uint8_t byte = tcodes[((slot * 2 + i / 16) * kTileRows + lane) * 16 + (i % 16)];
    code = static_cast<float>(static_cast<std::int8_t>(byte));
  }
  dst[static_cast<std::size_t>(blockIdx.y) * in + k] = code * tscales[slot * kTileRows + lane];
}

unsigned grid_for(std::size_t work, unsigned threads) { return static_cast<unsigned>(ceil_div(work, threads)); }

}  // namespace

int launch_quantize(const float* w, std::size_t out, std::size_t in, int type, std::uint8_t* planar_data,
                    float* planar_scales, DeviceMatrix* tiled, hipStream_t s) {
  const int nblk = static_cast<int>(ceil_div(in, kBlock));
  const std::size_t rows = tiled != nullptr ? ceil_div(out, kTileRows) * kTileRows : out;
  const std::size_t work = rows * static_cast<std::size_t>(nblk);
  if (work == 0) return LLMI_OK;
  const unsigned g = grid_for(work, 32 * kQuantItems);
  const int n = static_cast<int>(in);
  if (tiled != nullptr) {
    if (type == LLMI_TYPE_Q8_0)
      quantize_blocks<LLMI_TYPE_Q8_0, false><<<g, 256, 0, s>>>(w, out, n, nblk, tiled->codes, tiled->scales);
    else
      quantize_blocks<LLMI_TYPE_Q4_0, false><<<g, 256, 0, s>>>(w, out, n, nblk, tiled->codes, tiled->scales);
  } else if (type == LLMI_TYPE_Q8_0) {
    quantize_blocks<LLMI_TYPE_Q8_0, true><<<g, 256, 0, s>>>(w, out, n, nblk, planar_data, planar_scales);
  } else {
    quantize_blocks<LLMI_TYPE_Q4_0, true><<<g, 256, 0, s>>>(w, out, n, nblk, planar_data, planar_scales);
  }
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

int launch_relayout_to_tiled(const std::uint8_t* pdata, const float* pscales, const DeviceMatrix& m, hipStream_t s) {
  const std::size_t work = m.out * m.nblk;
  if (work == 0) return LLMI_OK;
  const unsigned g = grid_for(work, 256);
  if (m.type == LLMI_TYPE_Q8_0) {
    planar_to_tiled<LLMI_TYPE_Q8_0><<<g, 256, 0, s>>>(pdata, pscales, m.out, static_cast<int>(m.in), static_cast<int>(m.nblk), m.codes, m.scales);
  } else {
    planar_to_tiled<LLMI_TYPE_Q4_0><<<g, 256, 0, s>>>(pdata, pscales, m.out, static_cast<int>(m.in), static_cast<int>(m.nblk), m.codes, m.scales);
  }
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

int launch_gguf_to_tiled(const void* raw, const DeviceMatrix& m, hipStream_t s) {
  const std::size_t work = m.out * m.nblk;
  if (work == 0) return LLMI_OK;
  const unsigned g = grid_for(work, 256);
  const auto* src = static_cast<const std::uint16_t*>(raw);
  if (m.type == LLMI_TYPE_Q8_0) {
    gguf_to_tiled<LLMI_TYPE_Q8_0><<<g, 256, 0, s>>>(src, m.out, static_cast<int>(m.nblk), m.codes, m.scales);
  } else {
    gguf_to_tiled<LLMI_TYPE_Q4_0><<<g, 256, 0, s>>>(src, m.out, static_cast<int>(m.nblk), m.codes, m.scales);
  }
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

int launch_relayout_to_planar(const DeviceMatrix& m, std::uint8_t* pdata, float* pscales, hipStream_t s) {
  const std::size_t work = m.out * m.nblk;
  if (work == 0) return LLMI_OK;
  const unsigned g = grid_for(work, 256);
  if (m.type == LLMI_TYPE_Q8_0) {
    tiled_to_planar<LLMI_TYPE_Q8_0><<<g, 256, 0, s>>>(m.codes, m.scales, m.out, static_cast<int>(m.in), static_cast<int>(m.nblk), pdata, pscales);
  } else {
    tiled_to_planar<LLMI_TYPE_Q4_0><<<g, 256, 0, s>>>(m.codes, m.scales, m.out, static_cast<int>(m.in), static_cast<int>(m.nblk), pdata, pscales);
  }
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

int launch_dequantize_rows(const DeviceMatrix& m, const std::int32_t* ids, std::size_t n, float* dst, hipStream_t s) {
  if (m.type == LLMI_TYPE_F32) return launch_gather_f32(m, ids, n, dst, s);
  if (n == 0 || m.in == 0) return LLMI_OK;
  LLMI_REQUIRE(n <= 65535, "dequantize_rows: at most 65535 rows per call");
  const dim3 g(grid_for(m.in, 256), static_cast<unsigned>(n));
  if (m.type == LLMI_TYPE_Q8_0) {
    dequantize_rows<LLMI_TYPE_Q8_0><<<g, 256, 0, s>>>(m.codes, m.scales, static_cast<int>(m.in), static_cast<int>(m.nblk), ids, dst);
  } else {
    dequantize_rows<LLMI_TYPE_Q4_0><<<g, 256, 0, s>>>(m.codes, m.scales, static_cast<int>(m.in), static_cast<int>(m.nblk), ids, dst);
  }
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

}  // namespace llmi_hip
