// fp32 weights on the GPU: the reference's kernels::matmul
// (src/model/kernels.cpp:97-113, y[r][o] = dot(x_r, w_o, in) + bias[o]) and
// the Weight::row copy (src/model/weight.cpp:39-45) for Type::F32 weights.
//
// Storage: row-major [out][in] floats, as the reference keeps them.  One
// group of 16 lanes computes one dot exactly as the AVX2 kernels::dot does:
// lane j accumulates fused products of elements 16c + j over the full
// 16-element chunks, the lanes are reduced by the same tree ((j + j+8),
// (+4), (+2), (+1), as DPP row shifts), and the group's first lane adds the
// scalar part on the fewer than 16 elements left (ref_dot_rest).  The
// result, its bias and the optional residual update are the reference's
// operations in its order, so y is bit-identical.  Weight reads are 64-byte
// pieces per group and lane; x is shared by the workgroup's 16 dots.
#include "common.hpp"
#include "glue_math.hpp"

namespace llmi_hip {

namespace {

template <int N>
__device__ __forceinline__ float add_row_shl(float v) {
  const int src = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + N, 0xF, 0xF, true);
  return v + __int_as_float(src);
}

// grid (ceil(out / 16), rows), 256 threads: group g of 16 lanes computes
// output blockIdx.x * 16 + g of input row blockIdx.y.
__global__ void __launch_bounds__(256) matmul_f32(const float* __restrict__ x, const float* __restrict__ w,
                                                  const float* __restrict__ bias, float* __restrict__ y, int in,
                                                  int out, int accumulate) {
  const int j = threadIdx.x & 15;
  const int o = blockIdx.x * 16 + (threadIdx.x >> 4);
  const int r = blockIdx.y;
  const bool live = o < out;
  const float* xr = x + static_cast<std::size_t>(r) * in;
  const float* wr = w + static_cast<std::size_t>(live ? o : 0) * in;
  const int nfull = in / 16;
  float lane = 0.0f;
#pragma unroll 4
  for (int c = 0; c < nfull; ++c) lane = __builtin_fmaf(xr[16 * c + j], wr[16 * c + j], lane);
  lane = add_row_shl<8>(lane);
  lane = add_row_shl<4>(lane);
  lane = add_row_shl<2>(lane);
  lane = add_row_shl<1>(lane);
  if (j == 0 && live) {
    const float d = lane + ref_dot_rest(xr + 16 * nfull, wr + 16 * nfull, in - 16 * nfull);
    const float v = d + (bias != nullptr ? bias[o] : 0.0f);
    float* dst = y + static_cast<std::size_t>(r) * out + o;
    *dst = accumulate ? *dst + v : v;
  }
}

// The same dots for many rows, on the matrix cores.  v_mfma_f32_16x16x4_f32
// adds to each of 16 x 16 results an ascending chain of four IEEE fused
// multiply-adds (see qrows.hip), so with lane j's elements of four
// consecutive chunks as its four k, sixteen of them -- one accumulator per
// lane j of the AVX2 dot -- advance 16 rows x 16 outputs by 64 elements; the
// tree over the lanes is then fifteen additions in registers.  Bound: the
// fp32 matrix rate.  The workgroup's wavefronts share 16 * RW rows and
// 16 * 4 / RW outputs of both operands through LDS (two buffers, 64 elements
// a step); fetched per wavefront, the operands would take the L1's whole
// bandwidth.  Chunks past the last whole one are staged as -0 * 0, which
// leaves every accumulator as it is.  4864 x 896 at 128 rows: 120 -> 17.1 us (65 TFLOP/s).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));

template <int RW>
__global__ void __launch_bounds__(256, 2) matmul_f32_rows(const float* __restrict__ x, const float* __restrict__ w,
                                                          const float* __restrict__ bias, float* __restrict__ y, int in,
                                                          int out, int rows, int accumulate) {
  constexpr int OW = 4 / RW, kRows = 16 * (RW + OW), kStep = 64;
  constexpr int kStride = kStep + 4;  // 16 rows' 16-byte reads in distinct banks
  constexpr int kPer = kRows * (kStep / 4) / 256;
  __shared__ __attribute__((aligned(16))) float lds[2][kRows][kStride];  // 16 * RW rows of x, then of w
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = blockIdx.y * 16 * RW, o0 = blockIdx.x * 16 * OW;
  const int whole = in / 16 * 16;  // elements of whole chunks
  const int nstep = (whole + kStep - 1) / kStep;
  // Piece u of this thread: row u * 16 + tid / 16 of the workgroup's (rows of
  // x, then of w), elements 4 * (tid % 16) .. of the step.  Rows past the
  // last are the last one again (computed, never stored).
  const float* src[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int t = u * 16 + (tid >> 4);
    src[u] = u < RW ? x + static_cast<std::size_t>(min(r0 + t, rows - 1)) * in
                    : w + static_cast<std::size_t>(min(o0 + t - 16 * RW, out - 1)) * in;
    src[u] += 4 * (tid & 15);
  }
  struct Pieces {
    f32x4 v[kPer];
  };
  const auto load = [&](Pieces& p, int s) {
    const int k = min(s, nstep - 1) * kStep;
    if (k + kStep <= whole) {  // (uniform)
#pragma unroll
      for (int u = 0; u < kPer; ++u) p.v[u] = *reinterpret_cast<const f32x4a4*>(src[u] + k);
      return;
    }
    const bool inside = k + 4 * (tid & 15) < whole;  // a piece lies in one chunk
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const f32x4a4 t = *reinterpret_cast<const f32x4a4*>(src[u] + (inside ? k : -4 * (tid & 15)));
      const float pad = u < RW ? -0.0f : 0.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e) p.v[u][e] = inside ? t[e] : pad;
    }
  };
  const auto store = [&](const Pieces& p, int buf) {
#pragma unroll
    for (int u = 0; u < kPer; ++u)
      *reinterpret_cast<f32x4*>(&lds[buf][u * 16 + (tid >> 4)][4 * (tid & 15)]) = p.v[u];
  };
  const int rg = wave % RW, og = wave / RW;
  f32x4 acc[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // Step s computes from LDS buffer s % 2, then stores step s + 1 (loaded two
  // steps earlier) and loads step s + 3 in its place.
  Pieces pa, pb;
  load(pa, 0);
  load(pb, 1);
  store(pa, 0);
  load(pa, 2);
  __syncthreads();
  const auto step = [&](int s, int buf, Pieces& next) {
    const f32x4* a = reinterpret_cast<const f32x4*>(&lds[buf][rg * 16 + n][q * 16]);
    const f32x4* b = reinterpret_cast<const f32x4*>(&lds[buf][16 * RW + og * 16 + n][q * 16]);
#pragma unroll
    for (int j = 0; j < 16; ++j)
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j >> 2][j & 3], b[j >> 2][j & 3], acc[j], 0, 0, 0);
    store(next, buf ^ 1);
    load(next, s + 3);
    __syncthreads();
  };
  int s = 0;
  for (; s + 2 <= nstep; s += 2) {
    step(s, 0, pb);
    step(s + 1, 1, pa);
  }
  if (s < nstep) step(s, 0, pb);
#pragma unroll
  for (int h = 8; h > 0; h /= 2)
#pragma unroll
    for (int j = 0; j < h; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[j][e] = acc[j][e] + acc[j + h][e];
  const int o = o0 + og * 16 + n;
  if (o >= out) return;
  const float add = bias != nullptr ? bias[o] : 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = r0 + rg * 16 + 4 * q + e;
    if (r < rows) {
      const float d = acc[0][e] + ref_dot_rest(x + static_cast<std::size_t>(r) * in + whole,
                                               w + static_cast<std::size_t>(o) * in + whole, in - whole);
      const float t = d + add;
      float* dst = y + static_cast<std::size_t>(r) * out + o;
      *dst = accumulate ? *dst + t : t;
    }
  }
}

// dst[i] = rows ids[i] of w (the fp32 embedding gather).
__global__ void __launch_bounds__(256) gather_rows_f32(const float* __restrict__ w, const std::int32_t* __restrict__ ids,
                                                       std::size_t n, int in, float* __restrict__ dst) {
  const std::size_t e = static_cast<std::size_t>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= n * static_cast<std::size_t>(in)) return;
  const std::size_t i = e / in;
  const int k = static_cast<int>(e % in);
  dst[e] = w[static_cast<std::size_t>(ids[i]) * in + k];
}

}  // namespace

int launch_matmul_f32(const DeviceMatrix& m, const float* x, std::size_t rows, const float* bias, float* y,
                      hipStream_t s, bool accumulate) {
  LLMI_REQUIRE(rows <= 65535, "matmul (f32): at most 65535 input rows per call");
  const float* w = reinterpret_cast<const float*>(m.codes);
  const int in = static_cast<int>(m.in), out = static_cast<int>(m.out), nr = static_cast<int>(rows);
  // One dot per 16 lanes reads its row of w once per input row, from the
  // caches; a step of the matrix-core form takes 0.4 us however few rows it
  // has.  The line lies where the two met (us, dots / matrix cores): 896 x 896
  // at 32 rows 7.7 / 8.3, at 64 12.9 / 8.4; 576 x 576 at 64 7.0 / 6.4; 4864 x
  // 896 at 8 10.5 / 8.8; 896 x 4864 at 32 34.9 / 33.7; 49152 x 576 at 2 rows
  // 30.9 / 18.9; not below the 24576 dots that give every CU six workgroups:
  // 2048 x 12000 at 12 rows 68.9 / 94.4.
  if (m.in >= 16 && rows > 1 && rows * m.out > 24600 + 5600000 / m.in) {
    if (rows <= 16) {
      const dim3 grid(static_cast<unsigned>(ceil_div(m.out, 64)), 1);
      matmul_f32_rows<1><<<grid, 256, 0, s>>>(x, w, bias, y, in, out, nr, accumulate ? 1 : 0);
    } else {
      const dim3 grid(static_cast<unsigned>(ceil_div(m.out, 32)), static_cast<unsigned>(ceil_div(rows, 32)));
      matmul_f32_rows<2><<<grid, 256, 0, s>>>(x, w, bias, y, in, out, nr, accumulate ? 1 : 0);
    }
    LLMI_TRY_HIP(hipGetLastError());
    return LLMI_OK;
  }
  const dim3 grid(static_cast<unsigned>(ceil_div(m.out, 16)), static_cast<unsigned>(rows));
  matmul_f32<<<grid, 256, 0, s>>>(x, reinterpret_cast<const float*>(m.codes), bias, y, static_cast<int>(m.in),
                                  static_cast<int>(m.out), accumulate ? 1 : 0);
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

int launch_gather_f32(const DeviceMatrix& m, const std::int32_t* ids, std::size_t n, float* dst, hipStream_t s) {
  const std::size_t total = n * m.in;
  if (total == 0) return LLMI_OK;
  gather_rows_f32<<<static_cast<unsigned>(ceil_div(total, 256)), 256, 0, s>>>(
      reinterpret_cast<const float*>(m.codes), ids, n, static_cast<int>(m.in), dst);
  LLMI_TRY_HIP(hipGetLastError());
  return LLMI_OK;
}

}  // namespace llmi_hip
