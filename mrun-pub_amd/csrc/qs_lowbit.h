// Pieces shared by the packed int3 / int2 kernels (qs_lowbit.hip, qs_lowbit_gemm.hip).
#pragma once

#include "qs_common.h"

namespace qs {

struct LowbitParams {
  const uint16_t* x;   // bf16 [M, K] (M <= 16)
  int64_t ldx;
  const float* s0;     // [M, ng] group sums of x
  const uint8_t* packed;
  int64_t row_bytes;
  const void* scales;  // [N, ng] f32 or f16
  const void* zeros;   // [N, ng] f16/f32, nullable
  int scale_f16, zero_f16;
  float offset;        // used when zeros == nullptr
  float* y;            // [M, N]
  int64_t ldy;
  int M, N, K, ng;
  uint32_t pair_mask, pair_base;  // code-pair -> bf16x2 (OFF + c) masks, set by pair_consts()
};

// (t * spread) & mask | base turns the 2*BITS-bit code pair t into two bf16 (OFF + c).
// mask/base travel as kernel arguments (scalar registers) so that the and/or is a single
// v_bitop3_b32 (table 0xEA = (a & b) | c).
template <int BITS>
__device__ __forceinline__ uint32_t pair_bf16(uint32_t t, uint32_t mask, uint32_t base) {
  constexpr uint32_t spread = BITS == 3 ? 0x20010u : 0x80020u;
  return __builtin_amdgcn_bitop3_b32(t * spread, mask, base, 0xEA);
}

inline void pair_consts(LowbitParams& p, int bits) {
  p.pair_mask = bits == 3 ? 0x00700070u : 0x00600060u;
  p.pair_base = bits == 3 ? 0x41004100u : 0x40804080u;
}

// 2 codes starting at bit position bp of the field -> packed bf16 pair (OFF + c).
template <int BITS>
__device__ __forceinline__ uint32_t code_pair(const uint32_t (&f)[3], int bp, uint32_t mask, uint32_t base) {
  const int w = bp >> 5, o = bp & 31;
  uint32_t t;
  if (o + 2 * BITS <= 32)
    t = __builtin_amdgcn_ubfe(f[w], o, 2 * BITS);
  else
    t = __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(f[w + 1], f[w], o), 0, 2 * BITS);
  return pair_bf16<BITS>(t, mask, base);  // int3: 8 + c at bits 4-6 / 20-22; int2: 4 + c at 5-6 / 21-22
}

// Many activation rows (qs_lowbit_gemm.hip).
struct LowbitGemm {
  const void* x;  // BF16 or F32 [M, ldx]
  int x_dtype;
  int64_t ldx;
  const uint8_t* packed;
  int64_t row_bytes;
  const void* scales;  // F16 with F16 zeros, or F32 without
  const void* zeros;
  bool scale_f16;
  float offset;
  int bits, G;
  float* y;
  int64_t ldy;
  int64_t M, N, K;
};
size_t lowbit_gemm_workspace(int x_dtype, int64_t M, int64_t N, int64_t K, int G);
// QS_ERR_UNSUPPORTED (nothing launched, no message) for operands or a workspace it does not take.
int run_lowbit_gemm(const LowbitGemm& a, void* workspace, size_t workspace_bytes, hipStream_t s);
// x -> bf16 rows, an fp32 row as its three terms (qs_lowbit.hip)
void launch_lowbit_prep(const void* x, int x_dtype, int64_t ldx, int M, int K, uint16_t* xb, hipStream_t s);

}  // namespace qs
