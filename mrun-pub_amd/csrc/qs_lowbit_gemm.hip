// Packed int3 / int2 products of many activation rows on gfx950.
//
//   k_lowbit_gemm    y[m, n] = sum_k x[m, k] w[n, k] for a tile of 16 * MT bf16 rows and
//                    64 weight rows x one K slice, the formula of k_lowbit_gk per group
//   k_lowbit_sum     the slices' (and, for fp32 activations, the three bf16 terms') partial
//                    sums added in order
#include "qs_lowbit.h"

#include <limits.h>

#include <algorithm>

namespace qs {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct LgParams {
  const uint16_t* x;  // bf16 [M, ldx]
  int64_t ldx;
  const uint8_t* packed;
  int64_t row_bytes;
  const void* scales;
  const void* zeros;
  float offset;
  float* out;  // [S][M][ldo]
  int64_t ldo;
  int M, N, K, ng;
  int T, TS, S;  // 128-k steps, steps per slice, slices
  int tiles_m, tiles_n;
  uint32_t pair_mask, pair_base;
};

__device__ __forceinline__ int lg_sgpr(int v) {  // see to_sgpr (qs_prefill.hip)
  asm("" : "+v"(v));
  return __builtin_amdgcn_readfirstlane(v);
}

__device__ __forceinline__ void lg_copy16(__amdgpu_buffer_rsrc_t r, uint8_t* dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
}

template <int N>
__device__ __forceinline__ void lg_wait_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// What bounds it: per group and 16 x 16 tile, 2 or 4 MFMAs (as many again per 16 activation
// rows for the group sums), 8 VALU operations to apply the zero point and the scale in fp32
// (the weights are fp32: folding the scale into the bf16 operand would round them), the
// unpacking of the wave's codes (19 VALU operations per 16 int2 codes, 24 per 16 int3) and the
// scale gathers; no single one dominates (by counter, 131 rows: the matrix pipe is busy 36% of
// the time at G = 128 and 22% at G = 64, half of it with the group sums; LDS reads take 37% at
// G = 128, half of it bank conflicts).  Activations reach LDS by DMA in 128-k steps shared by
// four waves, codes and scales go global -> VGPR, both two steps ahead.  k_lowbit_gk, one launch
// per 16 rows, reads and unpacks all codes for each of them.  Measured against it: int2 G = 128
// 131 x 4096 x 11008 124 -> 38 us, int3 G = 64 131 x 11008 x 4096 110 -> 60,
// 393 x 4096 x 11008 360 -> 109, 17 rows 26 -> 21 / 29 -> 17.  A step's two G = 64 scales (and
// zero points) in one load each: 74 -> 60 us at 131 rows.
template <int BITS, int G, int SZ, int MT>
__global__ __launch_bounds__(256, 2) void k_lowbit_gemm(LgParams p) {
  constexpr float OFF = BITS == 3 ? 8.f : 0.f;
  constexpr int TM = 16 * MT, TN = 64;
  constexpr int D = 2;             // steps in flight
  constexpr int GPS = 128 / G;     // groups per step
  constexpr int NJ = G / 32;       // MFMAs per group
  constexpr int CB = BITS * G / 8;  // code bytes of a row per group
  constexpr int QB = CB / 4;       // of a lane's quarter
  constexpr int NWD = BITS == 2 ? QB / 4 : (QB + 3) / 4;  // dwords read for it
  constexpr int STAGE = TM * 256;
  constexpr int XD = MT;           // 1 KiB copies per wave per stage
  constexpr int SW = GPS * (SZ ? 2 : 4) / 4 > 0 ? GPS * (SZ ? 2 : 4) / 4 : 1;  // scale words per step
  constexpr bool PAIR = GPS == 2;  // a step's two groups: their scales are loaded together
  constexpr int GROUP = XD + GPS + (SZ ? 2 : 1);
  __shared__ __attribute__((aligned(1024))) uint8_t lds[(D + 1) * STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, q = lane >> 4;

  // contiguous runs of tiles per XCD, the activation tile fastest (as k_prefill)
  const int Gr = (int)gridDim.x;
  const int q8 = Gr >> 3, r8 = Gr & 7, xcd = (int)blockIdx.x & 7;
  const int lid = xcd * q8 + min(xcd, r8) + ((int)blockIdx.x >> 3);
  const int ls = lg_sgpr(lid / p.S);
  const int s = lid - ls * p.S;
  const int tn = lg_sgpr(ls / p.tiles_m);
  const int tm = ls - tn * p.tiles_m;
  const int tb = tn * TN, bm = tm * TM;
  const int t0 = s * p.TS;
  const int T = min(p.TS, p.T - t0);
  const int ng = p.ng, K = p.K;

  // operands through buffers from the tile's first row: rows past the operand, steps past the
  // slice and groups past the row read out of range (zero codes, scales and activations)
  const int xrows = min(TM, p.M - bm), wrows = min(TN, p.N - tb);
  const int xlim = (int)(((int64_t)(xrows - 1) * p.ldx + K) * 2);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(p.x + (int64_t)bm * p.ldx), (short)0, xlim, 0x00020000);
  const int wlim = wrows * (int)p.row_bytes;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(p.packed + (int64_t)tb * p.row_bytes), (short)0, wlim, 0x00020000);
  constexpr int ES = SZ ? 2 : 4;
  const int slim = wrows * ng * ES;
  const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(static_cast<const char*>(p.scales) + (int64_t)tb * ng * ES), (short)0, slim, 0x00020000);
  const __amdgpu_buffer_rsrc_t zr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(static_cast<const char*>(SZ ? p.zeros : p.scales) + (int64_t)tb * ng * ES), (short)0, slim,
      0x00020000);

  // copy e: 4 rows x 256 bytes; lane l lands in row l >> 4, slot l & 15, which holds chunk
  // slot ^ (row & 15)
  int xoff[XD], xk[XD], xdst[XD];
#pragma unroll
  for (int e = 0; e < XD; ++e) {
    const int c = wave * XD + e, r = 4 * c + (lane >> 4);
    const int ch = (lane & 15) ^ (r & 15);
    xoff[e] = r * (int)p.ldx * 2 + 16 * ch;
    xk[e] = 8 * ch;
    xdst[e] = 1024 * c;
  }
  auto copy_x = [&](int i, int st) {
    const int k0 = (t0 + i) * 128;
    const int room = i < T ? K - k0 : 0;  // k left in the row
#pragma unroll
    for (int e = 0; e < XD; ++e)
      lg_copy16(xr, lds + st * STAGE + xdst[e], xk[e] < room ? xoff[e] : xlim, i < T ? k0 * 2 : 0);
  };
  uint32_t cw[D][GPS][NWD];
  uint32_t sw[D][SW], zw[D][SW];
  const int qoff = BITS == 3 && G == 64 ? (6 * q) & ~3 : QB * q;
  auto load_w = [&](int b, int i) {
    const int r = 16 * wave + col;
#pragma unroll
    for (int gi = 0; gi < GPS; ++gi) {
      const int g = (t0 + i) * GPS + gi;
      const bool live = i < T && g < ng;
      const int wo = live ? r * (int)p.row_bytes + g * CB + qoff : wlim;
      if constexpr (NWD == 1) {
        cw[b][gi][0] = __builtin_amdgcn_raw_buffer_load_b32(wr, wo, 0, 0);
      } else if constexpr (NWD == 2) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(wr, wo, 0, 0);
        cw[b][gi][0] = v[0];
        cw[b][gi][1] = v[1];
      } else {
        const auto v = __builtin_amdgcn_raw_buffer_load_b96(wr, wo, 0, 0);
        cw[b][gi][0] = v[0];
        cw[b][gi][1] = v[1];
        cw[b][gi][2] = v[2];
      }
    }
    // (an even group count keeps both groups of a step on one side of the row's end)
    const int g = (t0 + i) * GPS;
    const int so = i < T && g < ng ? (r * ng + g) * ES : slim;
    if constexpr (SZ) {
      sw[b][0] = PAIR ? __builtin_amdgcn_raw_buffer_load_b32(sr, so, 0, 0) : __builtin_amdgcn_raw_buffer_load_b16(sr, so, 0, 0);
      zw[b][0] = PAIR ? __builtin_amdgcn_raw_buffer_load_b32(zr, so, 0, 0) : __builtin_amdgcn_raw_buffer_load_b16(zr, so, 0, 0);
    } else if constexpr (PAIR) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(sr, so, 0, 0);
      sw[b][0] = v[0];
      sw[b][1] = v[1];
    } else {
      sw[b][0] = __builtin_amdgcn_raw_buffer_load_b32(sr, so, 0, 0);
    }
  };

  // the lane's quarter of a group as NJ fragments of OFF + code
  auto unpack = [&](const uint32_t (&c)[NWD], u32x4 (&f)[NJ]) {
    if constexpr (BITS == 2) {
      typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
      for (int wd = 0; wd < NJ / 2; ++wd) {  // 16 codes: FP4 conversions give pairs (c, c + 2)
        const uint32_t lo = c[wd] & 0x33333333u, hi = (c[wd] >> 2) & 0x33333333u;
        const bf16x2 pl[4] = {__builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(lo, 2.f, 0),
                              __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(lo, 2.f, 1),
                              __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(lo, 2.f, 2),
                              __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(lo, 2.f, 3)};
        const bf16x2 ph[4] = {__builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(hi, 2.f, 0),
                              __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(hi, 2.f, 1),
                              __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(hi, 2.f, 2),
                              __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(hi, 2.f, 3)};
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const uint32_t a = __builtin_bit_cast(uint32_t, pl[2 * h + e]), b = __builtin_bit_cast(uint32_t, ph[2 * h + e]);
            f[2 * wd + h][2 * e] = __builtin_amdgcn_perm(b, a, 0x05040100u);
            f[2 * wd + h][2 * e + 1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
          }
      }
    } else {
      uint32_t w[3] = {c[0], c[1], 0};
      if constexpr (NWD == 3) {
        w[2] = c[2];
      } else {  // 48 bits that start 0 or 16 bits into the dwords
        const int sh = (6 * q & 3) * 8;
        w[0] = __builtin_amdgcn_alignbit(c[1], c[0], sh);
        w[1] = c[1] >> sh;
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) f[j][e] = code_pair<3>(w, 3 * (8 * j + 2 * e), p.pair_mask, p.pair_base);
    }
  };

  const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});
  f32x4 y[MT], sum[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) y[m] = sum[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mul = [&](int b, int i, int st) {
    const uint8_t* xs = lds + st * STAGE + col * 256;
#pragma unroll
    for (int gi = 0; gi < GPS; ++gi) {
      u32x4 f[NJ];
      unpack(cw[b][gi], f);
      f32x4 s0[MT], d[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) s0[m] = d[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < NJ; ++e) {
        const int ch = (G == 64 ? 8 * gi + 2 * q : 4 * q) + e;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const bf16x8 x = *reinterpret_cast<const bf16x8*>(xs + 4096 * m + 16 * (ch ^ col));
          s0[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, ones, s0[m], 0, 0, 0);
          d[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, __builtin_bit_cast(bf16x8, f[e]), d[m], 0, 0, 0);
        }
      }
      const float sc = SZ ? f16_bits_to_f32((uint16_t)(sw[b][0] >> (16 * gi))) : __uint_as_float(sw[b][gi % SW]);
      const float cz = OFF + (SZ ? f16_bits_to_f32((uint16_t)(zw[b][0] >> (16 * gi))) : p.offset);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) y[m][r] = fmaf(sc, fmaf(-cz, s0[m][r], d[m][r]), y[m][r]);
    }
    load_w(b, i + D);
  };

#pragma unroll
  for (int d = 0; d < D; ++d) {
    copy_x(d, d);
    __builtin_amdgcn_sched_barrier(0);
    load_w(d, d);
    __builtin_amdgcn_sched_barrier(0);
  }
  int st = 0;
  auto step = [&](int b, int i) {
    lg_wait_barrier<(D - 1) * GROUP>();
    copy_x(i + D, st == 0 ? D : st - 1);
    __builtin_amdgcn_sched_barrier(0);
    mul(b, i, st);
    st = st == D ? 0 : st + 1;
  };
  // the running sums join the totals every four steps: a chain over all of a row's groups
  // would be less exact than k_lowbit_gk's short ones (11008 k, 172 groups: 2.4e-7 against
  // 1.1e-7 of 64-bit sums)
  auto flush = [&]() {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      sum[m] += y[m];
      y[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  for (int i = 0;;) {  // the loop's shape keeps the load counts exact (see k_prefill)
    step(0, i);
    if (++i >= T) break;
    step(1, i);
    if (++i >= T) break;
    step(0, i);
    if (++i >= T) break;
    step(1, i);
    if (++i >= T) break;
    flush();
  }
  flush();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copies past the slice

  // lane holds D[m = 4 q + r][n = col] of each tile
  float* out = p.out + (int64_t)s * p.M * p.ldo;
  const int n = tb + 16 * wave + col;
  if (n >= p.N) return;
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = bm + 16 * m + 4 * q + r;
      if (row < p.M) out[(int64_t)row * p.ldo + n] = sum[m][r];
    }
}

// y[m, n] = sum over the rpx terms of row m of the sum over slices s of part[s][rpx m + t][n]
__global__ __launch_bounds__(256) void k_lowbit_sum(const float* __restrict__ part, int S, int rpx, int M, int N,
                                                    float* __restrict__ y, int64_t ldy) {
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  if (i >= (int64_t)M * N) return;
  const int64_t m = i / N, n = i - m * N;
  const int64_t plane = (int64_t)rpx * M * N;
  float acc = 0.f;
  for (int t = 0; t < rpx; ++t) {
    const float* q = part + (rpx * m + t) * N + n;
    float v = q[0];
#pragma unroll 4
    for (int s = 1; s < S; ++s) v = add_rn(v, q[s * plane]);
    acc = t == 0 ? v : add_rn(acc, v);
  }
  y[m * ldy + n] = acc;
}

// One launch's tile rows MT, and in microseconds, fitted to 300 timings (int2 / int3; M 17..393;
// 4096x11008, 11008x4096, 4096x4096 and 2141x2048; 7% rms): `lat` a 128-k step of one
// workgroup alone on a CU, `thr` the same per workgroup when a CU has several, `end` its start
// and epilogue.  The first two are G = 64, the others G = 128 (half the scales to apply).
struct LgShape {
  int MT;
  float lat, thr, end;
};
constexpr LgShape kLgShapes[4] = {{2, 0.18f, 0.44f, 0.22f}, {4, 0.71f, 0.61f, 0.f}, {2, 0.21f, 0.30f, 0.f}, {4, 0.58f, 0.44f, 0.f}};
constexpr float kLgReduce = 1.1f;         // the launch that adds the slices,
constexpr float kLgReduceBytes = 5.2e6f;  // and its partial bytes (written and read) per microsecond
constexpr int kLgMaxS = 8;
constexpr int64_t kLgMaxPart = (int64_t)128 << 20;  // bytes of partial sums

struct LgPlan {
  int MT, S;
};

// The shape and slice count with the smallest modelled time, with at most `part_cap` bytes of
// partial sums.  1.2% slower than the best choice on average over the timings, 10% at worst.
LgPlan lg_plan(int64_t rows, int64_t N, int64_t K, int G, int64_t part_cap) {
  const int64_t T = cdiv(K, 128), tiles_n = cdiv(N, 64);
  LgPlan best{0, 1};
  float best_t = 0.f;
  for (int k = G == 64 ? 0 : 2, end = k + 2; k < end; ++k) {
    const LgShape& sh = kLgShapes[k];
    const int64_t tiles = cdiv(rows, 16 * sh.MT) * tiles_n;
    for (int S = 1; S <= kLgMaxS; ++S) {
      // a slice has at least three steps, and none is empty
      if (S > 1 && (T / S < 3 || (S - 1) * cdiv(T, S) >= T || S * rows * N * 4 > part_cap)) continue;
      const float per_cu = (float)cdiv(tiles * S, 256);
      float t = (float)cdiv(T, S) * std::max(sh.lat, sh.thr * per_cu) + sh.end * per_cu;
      if (S > 1) t += kLgReduce + 2.f * (float)(S * rows * N * 4) / kLgReduceBytes;
      if (best.MT == 0 || t < best_t) {
        best = LgPlan{sh.MT, S};
        best_t = t;
      }
    }
  }
  return best;
}

template <int BITS, int G, int SZ>
void lg_launch(const LgParams& p, int mt, hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)p.tiles_m * p.tiles_n * p.S));
  if (mt == 2) hipLaunchKernelGGL((k_lowbit_gemm<BITS, G, SZ, 2>), grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL((k_lowbit_gemm<BITS, G, SZ, 4>), grid, dim3(256), 0, s, p);
}

// Activation rows per launch.  fp32 (three bf16 rows each): at most 512, and no more than keep
// the terms' partial sums within 256 MB and the terms within 64 MB (147 rows of a
// 151,936 x 1536 head, where 512 would take 0.9 GB), but 32 in any case (384 bytes per weight
// row, less than the 512 of a single row's workspace).  bf16: a grid has fewer than 2^32
// threads (a K split's partial sums, at most kLgMaxPart, keep it far below).
int64_t lg_chunk_rows(bool f32, int64_t N, int64_t K) {
  if (!f32) return (int64_t)UINT32_MAX / 256 / cdiv(N, 64) * 32;
  const int64_t rows = std::min(((int64_t)256 << 20) / (12 * N), ((int64_t)64 << 20) / (6 * K));
  return std::min<int64_t>(512, std::max<int64_t>(32, rows));
}

}  // namespace

size_t lowbit_gemm_workspace(int x_dtype, int64_t M, int64_t N, int64_t K, int G) {
  if (G != 64 && G != 128) return 0;
  if (x_dtype == QS_F32) {
    const int64_t rows = 3 * std::min(M, lg_chunk_rows(true, N, K));
    const LgPlan plan = lg_plan(rows, N, K, G, kLgMaxPart);
    return (size_t)((rows * K * 2 + 255) / 256 * 256) + (size_t)plan.S * rows * N * 4;
  }
  const LgPlan plan = lg_plan(M, N, K, G, kLgMaxPart);
  return plan.S > 1 ? (size_t)plan.S * M * N * 4 : 0;
}

int run_lowbit_gemm(const LowbitGemm& a, void* workspace, size_t workspace_bytes, hipStream_t s) {
  const bool f32 = a.x_dtype == QS_F32;
  const bool sz = a.scale_f16;
  const int ng = (int)(a.K / a.G);
  if ((a.G == 64 && ng % 2 != 0) || a.K % 8 != 0 || a.row_bytes % 4 != 0 || !aligned(a.packed, 4) ||
      !aligned(a.scales, 4) || (a.zeros && !aligned(a.zeros, 4)) || !aligned(workspace, 16))
    return QS_ERR_UNSUPPORTED;
  if (!f32 && (!aligned(a.x, 16) || a.ldx % 8 != 0)) return QS_ERR_UNSUPPORTED;
  // offsets inside a tile are 31-bit
  if (64 * a.row_bytes >= INT_MAX || 64 * std::max(a.ldx, a.K) * 2 >= INT_MAX) return QS_ERR_UNSUPPORTED;
  LgParams p{};
  p.packed = a.packed;
  p.row_bytes = a.row_bytes;
  p.scales = a.scales;
  p.zeros = a.zeros;
  p.offset = a.offset;
  p.N = (int)a.N;
  p.K = (int)a.K;
  p.ng = ng;
  p.T = (int)cdiv(a.K, 128);
  p.tiles_n = (int)cdiv(a.N, 64);
  LowbitParams pc{};
  pair_consts(pc, a.bits);
  p.pair_mask = pc.pair_mask;
  p.pair_base = pc.pair_base;
  const int rpx = f32 ? 3 : 1;
  const int64_t chunk = std::min(a.M, lg_chunk_rows(f32, a.N, a.K));
  if (chunk == 0 || chunk * rpx > INT_MAX) return QS_ERR_UNSUPPORTED;
  const int64_t xb_bytes = f32 ? (3 * chunk * a.K * 2 + 255) / 256 * 256 : 0;
  if ((int64_t)workspace_bytes < xb_bytes) return QS_ERR_UNSUPPORTED;
  const int64_t room = (int64_t)workspace_bytes - xb_bytes;
  float* part = reinterpret_cast<float*>(static_cast<char*>(workspace) + xb_bytes);
  for (int64_t m0 = 0; m0 < a.M; m0 += chunk) {
    const int64_t mm = std::min(chunk, a.M - m0), rows = rpx * mm;
    if (f32 && room < rows * a.N * 4) return m0 ? fail(QS_ERR_INVALID, "lowbit_gemv: workspace too small") : QS_ERR_UNSUPPORTED;
    const LgPlan plan = lg_plan(rows, a.N, a.K, a.G, std::min(room, kLgMaxPart));
    p.M = (int)rows;
    p.S = plan.S;
    p.TS = (int)cdiv(p.T, plan.S);
    p.tiles_m = (int)cdiv(rows, 16 * plan.MT);
    float* y = a.y + m0 * a.ldy;
    const void* xm = static_cast<const char*>(a.x) + m0 * a.ldx * (f32 ? 4 : 2);
    if (f32) {
      uint16_t* xb = static_cast<uint16_t*>(workspace);
      launch_lowbit_prep(xm, a.x_dtype, a.ldx, (int)mm, (int)a.K, xb, s);
      p.x = xb;
      p.ldx = a.K;
    } else {
      p.x = static_cast<const uint16_t*>(xm);
      p.ldx = a.ldx;
    }
    const bool direct = plan.S == 1 && !f32;
    p.out = direct ? y : part;
    p.ldo = direct ? a.ldy : a.N;
    if (a.bits == 3 && a.G == 64) sz ? lg_launch<3, 64, 1>(p, plan.MT, s) : lg_launch<3, 64, 0>(p, plan.MT, s);
    else if (a.bits == 3) sz ? lg_launch<3, 128, 1>(p, plan.MT, s) : lg_launch<3, 128, 0>(p, plan.MT, s);
    else if (a.G == 64) sz ? lg_launch<2, 64, 1>(p, plan.MT, s) : lg_launch<2, 64, 0>(p, plan.MT, s);
    else sz ? lg_launch<2, 128, 1>(p, plan.MT, s) : lg_launch<2, 128, 0>(p, plan.MT, s);
    if (!direct)
      hipLaunchKernelGGL(k_lowbit_sum, dim3((unsigned)cdiv(mm * a.N, 256)), dim3(256), 0, s, part, plan.S, rpx, (int)mm,
                         (int)a.N, y, a.ldy);
  }
  return hip_check(hipGetLastError(), "k_lowbit_gemm launch");
}

}  // namespace qs

using namespace qs;

extern "C" int qs_lowbit_many_plan(int x_dtype, int64_t M, int64_t N, int64_t K, int group_size, int32_t* tile) {
  const bool f32 = x_dtype == QS_F32;
  if (!tile || N < 1 || K < 1) return fail(QS_ERR_INVALID, "lowbit_many_plan: bad arguments");
  if (M <= (f32 ? 5 : 16) || (group_size != 64 && group_size != 128))
    return fail(QS_ERR_UNSUPPORTED, "lowbit_many_plan: more than 16 BF16 or 5 F32 rows, groups of 64 or 128");
  const int64_t chunk = std::min(M, lg_chunk_rows(f32, N, K));
  const LgPlan plan = lg_plan((f32 ? 3 : 1) * chunk, N, K, group_size, kLgMaxPart);
  tile[0] = 16 * plan.MT;
  tile[1] = plan.S;
  tile[2] = (int32_t)std::min<int64_t>(chunk, INT_MAX);
  return QS_OK;
}
