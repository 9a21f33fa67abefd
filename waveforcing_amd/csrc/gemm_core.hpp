// Pieces shared by the matrix-core GEMM kernels: the MFMA forms of the three operand types, the LDS DMA of
// 1 KB blocks and the wait counts around it.
#pragma once

#include <atomic>
#include <utility>

#include "wf_common.hpp"

namespace wf {
namespace gemm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int BK = 128;  // K bytes per step
constexpr int GROUP_M = 8;
constexpr int NUM_XCD = 8;
// Word 3 of a raw (untyped, stride 0) buffer resource on gfx9-family parts:
// DATA_FORMAT = 32 bit.  With it, offsets >= num_records read as zero.
constexpr int kBufferRsrcWord3 = 0x00020000;
constexpr int kOutOfRange = 0x7ffffff0;

// int8 x int8 -> int32, K = 32 per MFMA (one 16-byte piece per lane).
struct OpI8 {
  static constexpr int SUB = 4;
  static constexpr int PIECES = 1;
  typedef v16i acc_t;
  __device__ static acc_t mfma(const v4i* w, const v4i* a, acc_t c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(w[0], a[0], c, 0, 0, 0);
  }
};
// e4m3 x e4m3 -> fp32, K = 64 per MFMA (two 16-byte pieces per lane).  Zero
// scale operands select the unscaled v_mfma_f32_32x32x64_f8f6f4; format 0
// is OCP e4m3 for both operands.
struct OpFp8 {
  static constexpr int SUB = 2;
  static constexpr int PIECES = 2;
  typedef v16f acc_t;
  __device__ static acc_t mfma(const v4i* w, const v4i* a, acc_t c) {
    const v8i wv = __builtin_shufflevector(w[0], w[1], 0, 1, 2, 3, 4, 5, 6, 7);
    const v8i av = __builtin_shufflevector(a[0], a[1], 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wv, av, c, 0, 0, 0, 0, 0, 0);
  }
};

// bf16 x bf16 -> fp32, K = 16 per MFMA (one 16-byte piece per lane).
struct OpBf16 {
  static constexpr int SUB = 4;
  static constexpr int PIECES = 1;
  typedef v16f acc_t;
  __device__ static acc_t mfma(const v4i* w, const v4i* a, acc_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, w[0]), __builtin_bit_cast(v8bf, a[0]), c,
                                                   0, 0, 0);
  }
};

template <typename F, int... I>
__device__ inline void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ inline void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}
template <int V>
using ic = std::integral_constant<int, V>;

// s_waitcnt with vmcnt(VM), lgkmcnt(LGKM) (15 = no wait), expcnt unchanged.
template <int VM, int LGKM>
__device__ inline void wait_counts() {
  static_assert(VM >= 0 && VM < 64 && LGKM >= 0 && LGKM < 16, "wait counts");
  __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | 0x70 | (LGKM << 8));
}

__device__ inline void dma16(__amdgpu_buffer_rsrc_t rsrc, uint8_t* lds_block, int offset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, lds_block, 16, offset, 0, 0, 0);
}
__device__ inline void dma4(__amdgpu_buffer_rsrc_t rsrc, uint8_t* lds_block, int offset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, lds_block, 4, offset, 0, 0, 0);
}

// Compute units of the current device (one workgroup per CU at a time), cached per device (host threads may
// call concurrently; each stores the same value).
inline int device_cus() {
  static std::atomic<int> cus[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int v = cus[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    int n = 0;
    v = (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0) ? n : 256;
    cus[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

// Tile plan: -1 the product's rule; settable only in the instrumented libraries, for A/B runs (0 / 1 the 128- /
// 256-row W8A8 tile for the whole output, 2 + i the small tile i of gemm_small.hpp).
inline int g_tile_policy = -1;

}  // namespace gemm
}  // namespace wf
