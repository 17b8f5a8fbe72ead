// Device helpers shared by the kernels that read the tiled weight layout
// (common.hpp): typed global pointers, block loads and code extraction.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "common.hpp"

namespace llmi_hip {

// Signed bit-field extract (v_bfe_i32).  The builtin is declared with an
// unsigned result, so the value is reinterpreted as int before any
// conversion to float.
__device__ __forceinline__ int sfield(std::uint32_t w, int offset, int width) {
  return static_cast<int>(__builtin_amdgcn_sbfe(w, offset, width));
}

// Global-memory pointers.  The grouped kernel reads its pointers from a
// table, where the compiler cannot see that they point to global memory;
// typing them keeps global (not flat) loads for the weights and scalar
// loads for the activations.
#define GMEM __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ const GMEM T* gmem(const T* p) {
  return (const GMEM T*)p;
}
template <typename T>
__device__ __forceinline__ GMEM T* gmem_out(T* p) {
  return (GMEM T*)p;
}

template <int TYPE>
struct Block {
  static constexpr int kU = TYPE == LLMI_TYPE_Q8_0 ? 2 : 1;  // 16-byte loads per lane per block
  uint4 c[kU];
};

// Weights are streamed through once per product, so the batch 1..8 kernels
// load them with the nontemporal hint (they are not kept in the caches for
// reuse); the multi-row prefill kernel re-reads a tile per row chunk and uses
// ordinary loads.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
template <bool NT>
__device__ __forceinline__ uint4 load16(const GMEM uint4* p) {
  const GMEM u32x4* q = reinterpret_cast<const GMEM u32x4*>(p);
  const u32x4 v = NT ? __builtin_nontemporal_load(q) : *q;
  return uint4{v.x, v.y, v.z, v.w};
}
template <bool NT>
__device__ __forceinline__ float loadf(const GMEM float* p) {
  if (NT) return __builtin_nontemporal_load(p);
  return *p;
}

template <int TYPE, bool NT>
__device__ __forceinline__ Block<TYPE> load_block(const GMEM uint4* __restrict__ codes, std::size_t slot, int lane) {
  Block<TYPE> b;
#pragma unroll
  for (int u = 0; u < Block<TYPE>::kU; ++u) b.c[u] = load16<NT>(codes + (slot * Block<TYPE>::kU + u) * kTileRows + lane);
  return b;
}

// The code of element i of a block as float, exactly.
//   Q4_0: element i is nibble i%8 of word i/8 with +8 bias; XOR-ing every
//         nibble with 8 turns it into the 4-bit two's complement of n - 8.
//   Q8_0: element i is signed byte i%4 of word i/4.
template <int TYPE>
__device__ __forceinline__ float code_of(const std::uint32_t* w, int i) {
  if (TYPE == LLMI_TYPE_Q4_0) return static_cast<float>(sfield(w[i >> 3], (i & 7) * 4, 4));
  return static_cast<float>(sfield(w[i >> 2], (i & 3) * 8, 8));
}

template <int TYPE>
__device__ __forceinline__ void unpack_words(const Block<TYPE>& b, std::uint32_t* w) {
  if (TYPE == LLMI_TYPE_Q4_0) {
    w[0] = b.c[0].x ^ 0x88888888u;
    w[1] = b.c[0].y ^ 0x88888888u;
    w[2] = b.c[0].z ^ 0x88888888u;
    w[3] = b.c[0].w ^ 0x88888888u;
  } else {
    w[0] = b.c[0].x; w[1] = b.c[0].y; w[2] = b.c[0].z; w[3] = b.c[0].w;
    w[4] = b.c[Block<TYPE>::kU - 1].x; w[5] = b.c[Block<TYPE>::kU - 1].y;
    w[6] = b.c[Block<TYPE>::kU - 1].z; w[7] = b.c[Block<TYPE>::kU - 1].w;
  }
}

}  // namespace llmi_hip
