// Pieces shared by the qrow kernels (qs_qrow.hip, qs_batched.hip, qs_prefill.hip).
#pragma once

#include "qs_common.h"

namespace qs {

template <bool F16>
struct Half;
template <>
struct Half<false> {
  typedef bf16x8 vec;
  static __device__ __forceinline__ void deq(i32x4 w, float s, vec& lo, vec& hi) { deq16_bf16(w, s, lo, hi); }
  static __device__ __forceinline__ f32x4 mma(vec a, vec b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint16_t out(float v) { return f32_to_bf16_bits(v); }
};
template <>
struct Half<true> {
  typedef f16x8 vec;
  static __device__ __forceinline__ void deq(i32x4 w, float s, vec& lo, vec& hi) { deq16_f16(w, s, lo, hi); }
  static __device__ __forceinline__ f32x4 mma(vec a, vec b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint16_t out(float v) { return f32_to_f16_bits(v); }
};

__device__ __forceinline__ float silu(float g) { return g * (1.0f / (1.0f + expf(-g))); }

// Epilogue of one output: plane sums -> bf16/f16 (P = 1) or the paired SwiGLU (P = 2).
template <int P, bool F16>
__device__ __forceinline__ uint16_t w8a16_out(const float (&v)[P]) {
  if constexpr (P == 2) {
    const float gt = bf16_bits_to_f32(f32_to_bf16_bits(v[0]));
    const float ut = bf16_bits_to_f32(f32_to_bf16_bits(v[1]));
    const float sl = bf16_bits_to_f32(f32_to_bf16_bits(silu(gt)));
    return f32_to_bf16_bits(sl * ut);
  } else {
    return Half<F16>::out(v[0]);
  }
}

constexpr int kLdsBudget = 64 * 1024;  // activation rows staged by the VALU kernels

// Activation rows per VALU launch: the largest of 4/2/1 whose LDS copy fits.
inline int valu_mb(int x_dtype, int64_t K, int64_t M) {
  const int es = x_dtype == QS_F32 ? 4 : 2;
  const int cap = x_dtype == QS_F32 ? 4 : 2;
  for (int mb = cap; mb >= 1; mb /= 2)
    if ((int64_t)mb * K * es <= kLdsBudget && (mb <= M || mb == 1)) return mb;
  return 0;
}

// One linear of a call with many activation rows (qs_prefill.hip).
struct QrowPrefillLin {
  const int8_t* codes;
  const float* scales;
  void* y;
  int64_t ldy;
  int64_t N;
};
bool prefill_faster(int x_dtype, int64_t M, int n_lin, const int64_t* N, int64_t K, int P, bool split);
int run_prefill(const void* x, int x_dtype, int64_t ldx, int n_lin, const QrowPrefillLin* lin, int P, int64_t M,
                int64_t K, void* workspace, size_t workspace_bytes, hipStream_t s);

}  // namespace qs
