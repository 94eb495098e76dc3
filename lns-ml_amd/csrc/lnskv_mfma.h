// Types and lane exchanges shared by the matrix-core kernels (decode and
// prefill) over f16 and Q8A pages.
#pragma once

#include "lnskv_device.h"

namespace lnskv {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef unsigned int uint2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) short4v lds_short4v;
typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) half8 lds_half8;

// Heads of 128 dims (Llama-3 / Mixtral) and of 256 (lns-ml's Qwen3.5
// full-attention layers, model_config.rs:563-593): a 256-wide head is two
// 128-dim halves (NH = 2) that share one softmax; every per-half layout below
// (K operand lanes, V slot, transposed reads, output lanes) is the 128-dim one.
constexpr int kD = 128;                    // dims of one half
constexpr int kRowBytes = kD * 2;         // one half-row of f16
constexpr int kVSlot = kPage * kRowBytes;  // one half-page of V in LDS (swizzled rows)
constexpr float kRescaleSlack = 8.0f;     // log2 units the running max may lag
// Buffer resource word 3 for raw dword access on gfx9-family parts
// (DATA_FORMAT = 32-bit; no swizzle, no index stride).
constexpr int kBufferFormat = 0x00020000;

// A max or sum across halves / across adjacent 16-lane rows on the VALU.
__device__ __forceinline__ float max_xor32(float x) {
  const float2 p = swap_xor32(x);
  return fmaxf(p.x, p.y);
}
__device__ __forceinline__ float max_xor16(float x) {
  const float2 p = swap_xor16(x);
  return fmaxf(p.x, p.y);
}
__device__ __forceinline__ float sum_xor32(float x) {
  const float2 p = swap_xor32(x);
  return p.x + p.y;
}
__device__ __forceinline__ float sum_xor16(float x) {
  const float2 p = swap_xor16(x);
  return p.x + p.y;
}

__device__ __forceinline__ uint32_t v_swz(int R) { return 2u * (uint32_t)(((R >> 2) & 3) | ((R & 1) << 2)); }

// Waits until at most N vector-memory loads of this wave are outstanding
// (gfx9 s_waitcnt: vmcnt bits [3:0] and [15:14]; expcnt and lgkmcnt left open).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// Exact int8 -> f16 of the four signed bytes of w: the f16 with bits
// 0x6400 | (b + 128) is 1024 + b + 128, and subtracting 1152 leaves b.
__device__ __forceinline__ half4 i8x4_to_f16(uint32_t w) {
  typedef _Float16 half2q __attribute__((ext_vector_type(2)));
  const uint32_t u = w ^ 0x80808080u;
  const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);  // bytes u0, 0x64, u1, 0x64
  const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);  // bytes u2, 0x64, u3, 0x64
  const half2q c = {(_Float16)1152.0f, (_Float16)1152.0f};
  const half2q x = __builtin_bit_cast(half2q, lo) - c;
  const half2q y = __builtin_bit_cast(half2q, hi) - c;
  return half4{x[0], x[1], y[0], y[1]};
}

__device__ __forceinline__ half8 i8x8_to_f16(uint2v w) {
  const half4 a = i8x4_to_f16(w[0]), b = i8x4_to_f16(w[1]);
  return half8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

__device__ __forceinline__ int wave_incl_scan(int x) {
  const int lane = (int)(threadIdx.x & (kWave - 1));
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int y = __shfl_up(x, d, kWave);
    if (lane >= d) x += y;
  }
  return x;
}

}  // namespace
}  // namespace lnskv
