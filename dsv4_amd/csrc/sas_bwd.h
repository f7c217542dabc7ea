// Shared pieces of the backward kernels (sas_bwd.hip: per-token kernels and
// the window pass; sas_bwd_pre.hip: the prefill path).
#pragma once

#include <type_traits>
#include <utility>

#include "sas_kern.h"

namespace sas {

struct BwdParams {
  FwdParams f;
  const uint8_t* out;   // [T, H, 512] q dtype
  const uint8_t* dout;  // [T, H, 512] q dtype
  float* dq;            // [T, H, D] fp32
  float* d_ori;         // [ori rows, D] fp32, accumulated
  float* d_cmp;         // [cmp rows, D] fp32, accumulated (null for SWA)
  float* d_sinks;       // [H] fp32, accumulated
  int win_pass;         // 1: window rows' gradients come from sas_bwd_win_kernel (the per-token kernels skip them)
  int win_tiles;        // sas_bwd_win_kernel: 64-position row tiles per batch
  // key-major path (sas_bwd_pre.hip)
  float* delta;         // [T, H] fp32 workspace: Delta = dO . O
  uint8_t* nonfinite;   // [T, H / 16, 2] workspace: 1 if the heads' q (in that half of the channels) or dO has a NaN or Inf
  int npass;            // sas_bwd_dq_kernel: slot ranges of slots_per_split a workgroup walks
  int dq_direct;        // 1: dq is in the query dtype and written whole
  int dense_thr;        // tokens with a causal threshold up to this have their compressed rows' gradients
                        // summed by the key-major pass; the others add per token
  int sparse_only;      // per-token kernels: 1 takes only the tokens beyond dense_thr
  int key_seg;          // key-major pass: tokens per segment
  int seg_groups;       // key-major pass: (batch, segment) slots of the grid
  int cmp_tiles;        // key-major pass: compressed row tiles per segment
  int win_tiles_seg;    // key-major pass: window row tiles per segment
};

// f(integral_constant<int, j>) for j = 0 .. N-1, with no loop: arrays
// indexed this way are split into registers, while an array indexed inside a
// loop (even one unrolled later) is first moved to LDS or scratch memory by
// the compiler, which made each row-chunk prefetch a load waited for at once.
template <typename F, int... I>
__device__ __forceinline__ void unroll_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void unroll(F&& f) {
  unroll_impl(f, std::make_integer_sequence<int, N>{});
}
template <typename QT>
__device__ __forceinline__ float to_f(uint16_t v) {
  return (float)__builtin_bit_cast(QT, v);
}

// c + a.x * b.x + a.y * b.y for two packed 16-bit pairs (v_dot2c_f32_bf16 /
// v_dot2c_f32_f16)
template <typename QT>
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  typedef QT v2 __attribute__((ext_vector_type(2)));
  if constexpr (std::is_same<QT, __bf16>::value)
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c, false);
  else
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c, false);
}

// two packed 16-bit values (low half first) -> floats
template <typename QT>
__device__ __forceinline__ float2 unpack2(uint32_t w) {
  return make_float2(to_f<QT>((uint16_t)(w & 0xffffu)), to_f<QT>((uint16_t)(w >> 16)));
}

// Sum over the 16 lanes of a DPP row (a head's lanes), returned in every
// lane: quad_perm [1,0,3,2] and [2,3,0,1] (lane xor 1, xor 2), then
// row_half_mirror and row_mirror pair the quads and the halves.
__device__ __forceinline__ float sum16(float x) {
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1, 0xF, 0xF, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x4E, 0xF, 0xF, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x141, 0xF, 0xF, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x140, 0xF, 0xF, false));
  return x;
}

// The prefill path: dq by sas_bwd_dq_kernel (one workgroup per token and head
// group), then every cache row's gradient by sas_bwd_keys_kernel.
int launch_bwd_prefill(const BwdParams& bp, int D, int q_dtype, hipStream_t st);
// heads per workgroup of sas_bwd_dq_kernel
inline int bwd_dq_heads(int H) { return H % 64 == 0 ? 64 : 32; }
constexpr int kKeyRows = 64;   // rows per tile of the key-major pass

}  // namespace sas
