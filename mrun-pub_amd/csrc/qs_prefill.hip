// qrow linears for many activation rows (prefill) on gfx950: W8A16 and fp32.
//
// Kernels
//   k_prefill<P, MT, NT, WN, WK, XT> : one workgroup = a tile of 16 * MT activation rows
//                               and 16 * NT * WN weight rows (of P planes; P = 2 pairs the
//                               gate and up rows of a SwiGLU) x one K slice.
//   k_prefill_reduce<P, XT>   : the K slices' fp32 partial sums added in slice order, and the
//                               epilogue.
#include "qs_w8a16.h"

#include <limits.h>

#include <algorithm>

namespace qs {
namespace {

struct PfLin {
  const int8_t* codes;
  const float* scales;
  void* y;
  int64_t ldy;
  int N;
  int tile_begin;  // first weight tile of this linear
  int n_begin;     // first output column of this linear in the partial rows (a multiple of 4)
};

struct PfParams {
  const void* x;
  int64_t ldx;
  int M, K;
  int T, TS;  // 64-k steps, and steps per slice
  int S;      // slices
  int tiles_m, tiles_n;
  int n_lin, n_total;  // columns of a partial row: every linear's N rounded up to 4
  int vec;  // outputs allow 8-byte stores
  PfLin lin[4];
  float* part;  // [S][P][M][n_total] when S > 1
};

// A uniform value that the compiler computed on the vector ALU (an integer quotient), moved to
// an SGPR.  Left alone it keeps everything derived from it in VGPRs, the buffer descriptors
// included, and every buffer access then runs in a waterfall loop over the lanes.  The empty
// asm hides that the value is uniform, so that the read is not folded away.
__device__ __forceinline__ int to_sgpr(int v) {
  asm("" : "+v"(v));
  return __builtin_amdgcn_readfirstlane(v);
}

// One wave's 1 KiB global -> LDS copy: lane l's 16 bytes at buffer offset voff + soff land at
// dst + 16 l.  Not a template (see bd2_copy16).
__device__ __forceinline__ void pf_copy16(__amdgpu_buffer_rsrc_t r, uint8_t* dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
}

// At most N vector-memory operations of this wave outstanding, its LDS reads done, barrier.
template <int N>
__device__ __forceinline__ void pf_wait_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// A wave's accumulators go to separate sums every six of its 64-k steps (12 MFMAs): one
// fp32 chain over a whole row of 1536..8960 k would be less exact than the short chains of
// the batched kernels' K splits (outputs of 1531 x 1536 x 8960 that round differently from
// the exact sum: rel-L2 4.7e-5 in one chain, 1.8e-5 with the flushes, 1.9e-5 batched; they
// cost 2-3% of the time).
//
// What bounds it and why this split: the dequantized weight element costs 2.5 VALU operations,
// so it is made once per 16 * MT activation rows, in the registers of the one wave (of its
// K part) that owns the weight row: weights go global -> VGPR, and only activations pass
// through LDS, copied by DMA and read by all WN waves.  Measured in graph replays (1531 rows,
// one launch, before: 32-row batches of the batched kernel): paired SwiGLU 8960 x 1536
// 497 -> 113 us (745 TFLOP/s; traced 113 to 124 on several cards), 1536 x 8960 481 -> 70 us
// with its reduce, 1536 x 1536 213 -> 20 us.  At MT = 8 the loop's conversion instructions
// take 62% of the issue time of the MFMAs they feed, the other VALU ones 22%; the matrix pipe
// is busy 32% of the SwiGLU's time by counter, and LDS reads 33%, half of those cycles bank
// conflicts.  Timing probes of the 128-row tile on one box, 114 us whole: no conversion 101, no
// LDS reads 103, no copies 100, no weight loads 105, MFMAs and epilogue alone 63: no single
// phase bounds it, the phases of a CU's two or three workgroups overlap only in part.  Pinning
// the conversions between the MFMAs (one pair of codes per two MFMAs) was 10% slower, as was a
// third group in flight.
//
// fp32 activations run on v_mfma_f32_16x16x4 (a sixteenth of the bf16 rate), so there the
// matrix pipe is the bound and the tiles are small (16 or 32 rows) to keep every CU's busy:
// 149 x 1536 x 8960 785 -> 54 us (75 TFLOP/s of the 135 that a 4096^3 library product reaches,
// the pipe busy half of the time; before: one launch of the one-row VALU kernel per row),
// 64 x 8960 x 1536 148 -> 29 us, 16 x 4096 x 1024 19.3 -> 8.8 us.  Error against 64-bit sums 1.0e-7..1.2e-7 (VALU: 1.0e-7 at
// K = 1024 to 2.3e-7 at K = 8960).
template <int P, int MT, int NT, int WN, int WK, int XT>
__global__ __launch_bounds__(WN * WK * 64, 2) void k_prefill(PfParams p) {
  constexpr bool F32 = XT == QS_F32;
  typedef Half<XT == QS_F16> H;
  typedef typename H::vec hvec;
  constexpr int D = 2;  // iterations in flight
  constexpr int NW = WN * WK;
  constexpr int TM = 16 * MT, TN = 16 * NT * WN;
  constexpr int ES = F32 ? 4 : 2;
  constexpr int ROW = 64 * ES;     // bytes of one activation row's 64-k step
  constexpr int SL = ROW / 16;     // its 16-byte chunks
  constexpr int SUB = TM * ROW;    // bytes of one 64-k step's activations
  constexpr int STAGE = SUB * WK;
  constexpr int XD = STAGE / 1024 / NW;  // 1 KiB copies per wave per stage
  static_assert(XD * NW * 1024 == STAGE, "whole copies per wave");
  constexpr int RED = WK > 1 ? (WK - 1) * WN * MT * 64 * 16 : 0;
  constexpr int LDS = (D + 1) * STAGE > RED ? (D + 1) * STAGE : RED;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wk = wave / WN;
  const int col = lane & 15, grp = lane >> 4;

  // workgroups go to the 8 XCDs round robin; each XCD takes a contiguous run of tiles, the
  // activation tile fastest, so the tiles sharing a weight slab share an L2
  const int G = (int)gridDim.x;
  const int q8 = G >> 3, r8 = G & 7, xcd = (int)blockIdx.x & 7;
  const int lid = xcd * q8 + min(xcd, r8) + ((int)blockIdx.x >> 3);
  const int ls = to_sgpr(lid / p.S);
  const int s = lid - ls * p.S;
  const int tn = to_sgpr(ls / p.tiles_m);
  const int tm = ls - tn * p.tiles_m;
  int li = 0;
  if (P == 1) {
#pragma unroll
    for (int j = 1; j < 4; ++j)
      if (j < p.n_lin && tn >= p.lin[j].tile_begin) li = j;
  }
  const PfLin& L0 = p.lin[li];
  const int N = L0.N;
  const int tb = (tn - L0.tile_begin) * TN;  // first weight row of the tile
  const int bm = tm * TM;                    // first activation row
  const int K = p.K;
  const int t0 = s * p.TS;
  const int T = min(p.TS, p.T - t0);  // 64-k steps of this slice
  const int I = (T + WK - 1) / WK;

  // row scales
  float sc[P][NT];
#pragma unroll
  for (int pl = 0; pl < P; ++pl)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = tb + 16 * (NT * wn + j) + col;
      sc[pl][j] = p.lin[P == 2 ? pl : li].scales[n < N ? n : N - 1];
    }

  // operands through buffers that start at the tile's first row: rows past the operand and
  // steps past the slice read out of range (zero, no memory access)
  const int xrows = min(TM, p.M - bm);
  const int xlim = (int)(((int64_t)(xrows - 1) * p.ldx + K) * ES);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(static_cast<const char*>(p.x) + (int64_t)bm * p.ldx * ES), (short)0, xlim, 0x00020000);
  const int wlim = min(TN, N - tb) * K;
  __amdgpu_buffer_rsrc_t wr[P];
#pragma unroll
  for (int pl = 0; pl < P; ++pl)
    wr[pl] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(p.lin[P == 2 ? pl : li].codes + (int64_t)tb * K), (short)0, wlim, 0x00020000);

  // copy e of a stage: whole rows of one 64-k step; lane l lands in row l / SL, slot l % SL,
  // which holds 16-byte chunk slot ^ (a hash of the row): the 16 rows that 16 lanes of a
  // fragment read touch fall in distinct bank groups
  auto swz = [](int r) { return F32 ? r & 15 : (r >> 1) & 7; };
  int xoff[XD], xsub[XD], xdst[XD];
#pragma unroll
  for (int e = 0; e < XD; ++e) {
    const int c = wave * XD + e;
    const int r = (64 / SL) * (c % (SUB / 1024)) + lane / SL;
    xsub[e] = c / (SUB / 1024);
    xdst[e] = 1024 * c;
    xoff[e] = r * (int)p.ldx * ES + 16 * ((lane % SL) ^ swz(r));
  }
  auto copy_x = [&](int i, int st) {  // iteration i -> stage st
#pragma unroll
    for (int e = 0; e < XD; ++e) {
      const int t = i * WK + xsub[e];
      pf_copy16(xr, lds + st * STAGE + xdst[e], t < T ? xoff[e] : xlim, t < T ? (t0 + t) * ROW : 0);
    }
  };
  const int wlane = (16 * NT * wn + col) * K + 16 * grp;
  auto load_w = [&](i32x4 (&w)[P][NT], int i) {
    const int t = i * WK + wk;
#pragma unroll
    for (int pl = 0; pl < P; ++pl)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        w[pl][j] = __builtin_bit_cast(
            i32x4, __builtin_amdgcn_raw_buffer_load_b128(wr[pl], t < T ? wlane + 16 * j * K : wlim,
                                                         t < T ? (t0 + t) * 64 : 0, 0));
  };

  f32x4 acc[P][NT][MT], sum[P][NT][MT];
#pragma unroll
  for (int pl = 0; pl < P; ++pl)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[pl][j][m] = sum[pl][j][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  // iteration i from stage st; its weight registers take the weights of iteration i + D as
  // soon as they are dequantized.  16-bit: the lane's 16 codes make two MFMA fragments.
  const int sw = swz(col);
  auto mul16 = [&](i32x4 (&w)[P][NT], int i, int st) {
    const uint8_t* xs = lds + st * STAGE + wk * SUB + col * ROW;
    const uint8_t* x0 = xs + 16 * ((2 * grp) ^ sw);
    const uint8_t* x1 = xs + 16 * ((2 * grp + 1) ^ sw);
    hvec xa[MT], xb[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) xa[m] = *reinterpret_cast<const hvec*>(x0 + 16 * ROW * m);
    hvec wb[P][NT][2];
#pragma unroll
    for (int pl = 0; pl < P; ++pl)
#pragma unroll
      for (int j = 0; j < NT; ++j) H::deq(w[pl][j], sc[pl][j], wb[pl][j][0], wb[pl][j][1]);
    load_w(w, i + D);
#pragma unroll
    for (int pl = 0; pl < P; ++pl)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[pl][j][m] = H::mma(wb[pl][j][0], xa[m], acc[pl][j][m]);
#pragma unroll
    for (int m = 0; m < MT; ++m) xb[m] = *reinterpret_cast<const hvec*>(x1 + 16 * ROW * m);
#pragma unroll
    for (int pl = 0; pl < P; ++pl)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[pl][j][m] = H::mma(wb[pl][j][1], xb[m], acc[pl][j][m]);
  };
  // fp32: each of the lane's 16 codes is one k of a 16x16x4 MFMA (four k per instruction, one
  // from each lane group), weights float(code) * scale, products and sums in fp32.  Sums of 16
  // k start from zero and the four of a step are added in pairs before they join the
  // accumulators: short chains, as exact as the row's sum over a wave's lanes.
  auto mul32 = [&](i32x4 (&w)[P][NT], int i, int st) {
    const uint8_t* xs = lds + st * STAGE + wk * SUB + col * ROW;
    f32x4 part[2][NT][MT];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      f32x4 x[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) x[m] = *reinterpret_cast<const f32x4*>(xs + 16 * ((4 * grp + c) ^ sw) + 16 * ROW * m);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int d = w[0][j][c];
        const float wf[4] = {sbyte_f32<0>(d) * sc[0][j], sbyte_f32<1>(d) * sc[0][j], sbyte_f32<2>(d) * sc[0][j],
                             sbyte_f32<3>(d) * sc[0][j]};
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          f32x4 t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int q = 0; q < 4; ++q) t = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[q], x[m][q], t, 0, 0, 0);
          if (c % 2 == 0) part[c / 2][j][m] = t;
          else part[c / 2][j][m] += t;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m) sum[0][j][m] += part[0][j][m] + part[1][j][m];
    load_w(w, i + D);
  };
  auto mul = [&](i32x4 (&w)[P][NT], int i, int st) {
    if constexpr (F32) mul32(w, i, st);
    else mul16(w, i, st);
  };

  // Group i: the activation copies, then the weights, of iteration i.  D groups are in
  // flight: iteration i waits until only the D - 1 newer ones are outstanding; the barrier
  // also ends every wave's reads of the stage that group i + D overwrites.
  constexpr int GROUP = XD + P * NT;
  i32x4 w[D][P][NT];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    copy_x(d, d);
    __builtin_amdgcn_sched_barrier(0);
    load_w(w[d], d);
    __builtin_amdgcn_sched_barrier(0);
  }
  // The weight registers of an even and an odd iteration alternate in the loop body, and
  // every exit leaves it whole: the compiler then counts the loads still in flight exactly
  // (paths that join with another order of requests make it wait for the newest ones).
  auto flush = [&]() {
    if constexpr (!F32) {
#pragma unroll
      for (int pl = 0; pl < P; ++pl)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            sum[pl][j][m] += acc[pl][j][m];
            acc[pl][j][m] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
    }
  };
  int st = 0;
  auto step = [&](int d, int i) {
    pf_wait_barrier<(D - 1) * GROUP>();
    copy_x(i + D, st == 0 ? D : st - 1);
    __builtin_amdgcn_sched_barrier(0);
    mul(w[d], i, st);
    st = st == D ? 0 : st + 1;
  };
  for (int i = 0;;) {
    step(0, i);
    if (++i >= I) break;
    step(1, i);
    if (++i >= I) break;
    if constexpr (!F32) {
      step(0, i);
      if (++i >= I) break;
      step(1, i);
      if (++i >= I) break;
      step(0, i);
      if (++i >= I) break;
      step(1, i);
      if (++i >= I) break;
      flush();
    }
  }
  flush();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copies past the slice

  // the WK parts are added in order through LDS, one 16-row block of weights at a time
  if constexpr (WK > 1) {
    f32x4* red = reinterpret_cast<f32x4*>(lds);  // [WK - 1][WN][MT][64]
#pragma unroll
    for (int pl = 0; pl < P; ++pl)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        pf_wait_barrier<0>();  // copies landed and earlier reads done
        if (wk > 0) {
#pragma unroll
          for (int m = 0; m < MT; ++m) red[(((wk - 1) * WN + wn) * MT + m) * 64 + lane] = sum[pl][j][m];
        }
        pf_wait_barrier<0>();
        if (wk == 0) {
#pragma unroll
          for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int k2 = 1; k2 < WK; ++k2) sum[pl][j][m] += red[(((k2 - 1) * WN + wn) * MT + m) * 64 + lane];
        }
      }
    if (wk != 0) return;
  }

  // lane holds D[n = nb + q][m = 16 t + col]
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int nb = tb + 16 * (NT * wn + j) + 4 * grp;
    if (nb >= N) continue;
    const bool full = p.vec && nb + 3 < N;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = bm + 16 * t + col;
      if (m >= p.M) continue;
      if (p.S == 1 && F32) {
        float* yr = static_cast<float*>(L0.y) + (int64_t)m * L0.ldy + nb;
        if (full) {
          *reinterpret_cast<f32x4*>(yr) = sum[0][j][t];
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (nb + q < N) yr[q] = sum[0][j][t][q];
        }
      } else if (p.S == 1) {
        uint16_t o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float v[P];
#pragma unroll
          for (int pl = 0; pl < P; ++pl) v[pl] = sum[pl][j][t][q];
          o[q] = w8a16_out<P, XT == QS_F16>(v);
        }
        uint16_t* yr = static_cast<uint16_t*>(L0.y) + (int64_t)m * L0.ldy + nb;
        if (full) {
          *reinterpret_cast<uint2*>(yr) = make_uint2(o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16);
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (nb + q < N) yr[q] = o[q];
        }
      } else {
#pragma unroll
        for (int pl = 0; pl < P; ++pl) {
          // columns past N land in the row's padding
          *reinterpret_cast<f32x4*>(p.part + (((int64_t)s * P + pl) * p.M + m) * p.n_total + L0.n_begin + nb) =
              sum[pl][j][t];
        }
      }
    }
  }
}

// Slice sums in slice order and the epilogue: one thread per (row m, 4 columns of the
// partial row).  Partial rows hold every linear's columns rounded up to 4, so that any N can
// be split (three fp32 rows of 1001 x 8960: 61 us in one slice, 15 in ten); the columns past N
// are not stored.
template <int P, int XT>
__global__ __launch_bounds__(256) void k_prefill_reduce(PfParams p) {
  const int q4 = p.n_total / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int m = (int)(i / q4);
  if (m >= p.M) return;
  const int ncol = 4 * (int)(i - (int64_t)m * q4);
  int li = 0;
  if (P == 1) {
#pragma unroll
    for (int j = 1; j < 4; ++j)
      if (j < p.n_lin && ncol >= p.lin[j].n_begin) li = j;
  }
  f32x4 a[P];
#pragma unroll
  for (int pl = 0; pl < P; ++pl) {
    const float* pr = p.part + ((int64_t)pl * p.M + m) * p.n_total + ncol;
    const int64_t step = (int64_t)P * p.M * p.n_total;
    a[pl] = *reinterpret_cast<const f32x4*>(pr);
    for (int s = 1; s < p.S; ++s) a[pl] += *reinterpret_cast<const f32x4*>(pr + s * step);
  }
  const PfLin& L = p.lin[li];
  const int n = ncol - L.n_begin;
  const bool full = p.vec && n + 3 < L.N;
  if constexpr (XT == QS_F32) {
    float* yr = static_cast<float*>(L.y) + (int64_t)m * L.ldy + n;
    if (full) {
      *reinterpret_cast<f32x4*>(yr) = a[0];
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (n + q < L.N) yr[q] = a[0][q];
    }
    return;
  }
  uint16_t o[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float v[P];
#pragma unroll
    for (int pl = 0; pl < P; ++pl) v[pl] = a[pl][q];
    o[q] = w8a16_out<P, XT == QS_F16>(v);
  }
  uint16_t* yr = static_cast<uint16_t*>(L.y) + (int64_t)m * L.ldy + n;
  if (full) {
    *reinterpret_cast<uint2*>(yr) = make_uint2(o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (n + q < L.N) yr[q] = o[q];
  }
}

// Tile shapes: MT, NT * P, WN, WK, and three times in microseconds fitted to timings of these
// shapes: `lat` a round of WK 64-k steps of one workgroup alone on a CU, `thr` the same per
// workgroup when a CU has several, `end` its start and epilogue per workgroup.  16-bit: 600
// timings (M 33..1531; 2048x1536, 1536x8960, 6144x4096, 4096x14336 and 1024x2816 plain,
// 8960x1536, 14336x4096 and 2816x1024 paired; 8% rms).  fp32: 600 timings (M 2..500;
// 1536x8960, 4096x1024, 8960x1536, 2500x320, 3000x1536, 4096x4096, 4096x14336; 6% rms).
struct PfShape {
  int MT, NTP, WN, WK;
  float lat, thr, end;
};
constexpr PfShape kPfShapes[] = {
    {2, 2, 4, 2, 0.14f, 0.59f, 0.47f}, {4, 2, 4, 2, 0.73f, 0.65f, 0.70f},
    {8, 2, 4, 1, 0.61f, 0.48f, 0.36f}, {8, 2, 4, 2, 0.32f, 0.90f, 2.81f},
    {1, 1, 4, 2, 0.91f, 0.75f, 0.30f}, {2, 1, 4, 2, 1.42f, 1.27f, 0.93f},  // fp32
};
constexpr int kPfShapes16 = 4, kPfShapesAll = 6;
constexpr float kPfLaunch = 4.1f;         // a launch
constexpr float kPfReduce = 2.7f;         // the reduce launch,
constexpr float kPfReduceBytes = 4.8e6f;  // and its partial bytes (written and read) per microsecond
constexpr int kPfMaxS = 16;
constexpr int64_t kPfMaxWorkspace = (int64_t)256 << 20;

struct PfPlan {
  int shape, S;
  int64_t tiles_n, n_total;
  float us;  // modelled time
};

// The shape and slice count with the smallest modelled time: a large tile reuses its operands
// best, a small one (or a K split, which costs a reduce launch) fills the chip when the
// product has few tiles.  Over the products timed for the fits, the choice is 2% (16-bit) and
// 3% (fp32) slower than the best shape on average and 21% at worst.
PfPlan pf_plan(bool f32, int64_t M, int n_lin, const int64_t* N, int64_t K, int P, bool split) {
  const int64_t T = K / 64;
  int64_t n_total = 0;
  for (int i = 0; i < (P == 2 ? 1 : n_lin); ++i) n_total += cdiv(N[i], 4) * 4;
  PfPlan best{0, 1, 0, n_total, 0.f};
  for (int k = f32 ? kPfShapes16 : 0; k < (f32 ? kPfShapesAll : kPfShapes16); ++k) {
    const PfShape& sh = kPfShapes[k];
    int64_t tiles_n = 0;
    for (int i = 0; i < (P == 2 ? 1 : n_lin); ++i) tiles_n += cdiv(N[i], 16 * sh.NTP / P * sh.WN);
    const int64_t tiles = cdiv(M, 16 * sh.MT) * tiles_n;
    for (int S = 1; S <= (split ? kPfMaxS : 1); ++S) {
      const int64_t part = (int64_t)S * P * M * n_total * 4;
      // a slice has at least four 64-k steps and two rounds, and none is empty
      if (S > 1 && (T / S < 4 || T / S < 2 * sh.WK || (S - 1) * cdiv(T, S) >= T || part > kPfMaxWorkspace)) continue;
      const float per_cu = (float)cdiv(tiles * S, 256);
      const float rounds = (float)cdiv(cdiv(T, S), sh.WK);
      float t = kPfLaunch + rounds * std::max(sh.lat, sh.thr * per_cu) + sh.end * per_cu;
      if (S > 1) t += kPfReduce + 2.f * (float)part / kPfReduceBytes;
      if (best.tiles_n == 0 || t < best.us) best = PfPlan{k, S, tiles_n, n_total, t};
    }
  }
  return best;
}

template <int P, int XT>
void pf_launch(const PfParams& p, int shape, hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)p.tiles_m * p.tiles_n * p.S));
#define QS_PF(K_)                                                                                               \
  if (shape == K_) {                                                                                            \
    constexpr PfShape h = kPfShapes[K_];                                                                        \
    hipLaunchKernelGGL((k_prefill<P, h.MT, h.NTP / P, h.WN, h.WK, XT>), grid, dim3(h.WN * h.WK * 64), 0, s, p); \
  }
  if constexpr (XT == QS_F32) {
    QS_PF(4) QS_PF(5)
  } else {
    QS_PF(0) QS_PF(1) QS_PF(2) QS_PF(3)
  }
#undef QS_PF
  if (p.S > 1) {
    const dim3 rg((unsigned)cdiv((int64_t)p.M * (p.n_total / 4), 256));
    hipLaunchKernelGGL((k_prefill_reduce<P, XT>), rg, dim3(256), 0, s, p);
  }
}

// Activation rows that one launch of a plan takes: a grid has fewer than 2^32 threads (32-row
// fp32 tiles of one column reach that at 2^28 rows).  0: not even one tile row.
int64_t pf_launch_rows(const PfPlan& plan) {
  const PfShape& sh = kPfShapes[plan.shape];
  return (int64_t)UINT32_MAX / (sh.WN * sh.WK * 64) / (plan.tiles_n * plan.S) * 16 * sh.MT;
}

}  // namespace

// Whether the prefill kernel is expected to beat the launches that qs_qrow_matmul_multi and
// qs_qrow_swiglu otherwise make, from `split` or unsplit plan times against their times in
// microseconds (graph replays, 2 to 512 rows of the shapes below and their K and N in other
// pairs).  Rows longer than those kernels take run one wave per weight row there: always prefill.
bool prefill_faster(int x_dtype, int64_t M, int n_lin, const int64_t* N, int64_t K, int P, bool split) {
  if (M < 2) return false;
  float rows = 0.f;  // millions of weights
  for (int i = 0; i < (P == 2 ? 1 : n_lin); ++i) rows += (float)N[i];
  const float k = (float)K * 1e-3f, nk = rows * k * 1e-3f;
  if (x_dtype == QS_F32) {
    // One launch of the VALU kernel per 4, 2 or 1 rows that fit its 64 KiB (none past 12288):
    // 13% rms over 91 products.  It keeps rows of a single launch, two rows and, beside a split, those
    // the plan does not win by 4 us: a split call asks for a workspace and launches twice, 6 us
    // more of host time than the plain call (eager calls of 8 rows of 4096 x 1024 12.6 against
    // 18.4 us for 10.2 and 9.1 on the GPU; 6 rows of 4096 x 4096 21.6 against 18.7; 3 rows of
    // 1536 x 8960 16.2 against 18.9, and 61 on the GPU unsplit).
    if (K > 12288) return true;
    const int mb = valu_mb(x_dtype, K, M);
    const float L = (float)cdiv(M, mb);
    if (L < 2.f || M < 3) return false;
    const float valu = 0.65f + L * (2.6f + nk * (0.115f * mb - 0.019f) + 0.149f * mb * k);
    return pf_plan(true, M, n_lin, N, K, P, split).us + (split ? 4.f : 0.f) < valu;
  }
  // 16-bit: 32-row batches.  Past two of them, with a split, for a SwiGLU (33 rows of
  // 8960 x 1536 28 -> 14.5 us; at worst 37 -> 39, 33 rows of 301 x 8192 unsplit) and for rows
  // they do not take the prefill kernel is faster; unsplit it is bound by its K steps up to 64
  // rows (33 rows of 1536 x 8960 42 us against 33, of 4096 x 4096 22 against 20, of
  // 14336 x 4096 29 against 62), where a batch takes 2.7 us and its K steps or its weights.
  // Weights past the L2s' 32 MB slow the steps of the plan by a fifth (48 rows of
  // 4096 x 14336 82 us against 68).
  if (M <= 32) return false;
  if (M > 64 || split || P == 2 || K % 128 != 0) return true;
  const float body = std::max(2.4f * k, 0.7f * nk);
  const int tail = (int)M - 32;
  const float batches = 5.4f + body * (tail > 16 ? 2.f : 1.33f + 0.022f * (float)tail);
  return pf_plan(false, M, n_lin, N, K, P, false).us * (nk > 32.f ? 1.2f : 1.f) < batches;
}

// y = x @ W^T over the linears' shared x: `lin` holds the P planes of a SwiGLU (P = 2, y in lin[0])
// or n_lin linears.  `workspace` null: no K split.  Returns QS_ERR_UNSUPPORTED, without a
// message, for operands the kernel does not take (the callers' other kernels do).
int run_prefill(const void* x, int x_dtype, int64_t ldx, int n_lin, const QrowPrefillLin* lin, int P, int64_t M,
                int64_t K, void* workspace, size_t workspace_bytes, hipStream_t s) {
  const bool f32 = x_dtype == QS_F32;
  const int es = f32 ? 4 : 2;
  if (K % 64 != 0 || ldx * es % 16 != 0 || !aligned(x, 16)) return QS_ERR_UNSUPPORTED;
  if (128 * ldx * 4 >= INT_MAX || 128 * K >= INT_MAX) return QS_ERR_UNSUPPORTED;  // tile offsets are 31-bit
  PfParams p{};
  int64_t N[4];
  bool vec = true;
  for (int i = 0; i < n_lin; ++i) {
    if (!aligned(lin[i].codes, 16)) return QS_ERR_UNSUPPORTED;
    N[i] = lin[i].N;
    if (lin[i].y) vec = vec && lin[i].ldy % 4 == 0 && aligned(lin[i].y, 4 * es);
  }
  const PfPlan plan = pf_plan(f32, M, n_lin, N, K, P, workspace != nullptr);
  const PfShape& sh = kPfShapes[plan.shape];
  if (plan.S > 1) {
    if (workspace_bytes < (size_t)plan.S * P * M * plan.n_total * 4)
      return fail(QS_ERR_INVALID, "qrow prefill: workspace smaller than qs_qrow_prefill_workspace_bytes()");
    if (!aligned(workspace, 16)) return fail(QS_ERR_INVALID, "qrow prefill: workspace must be 16-byte aligned");
  }
  const int64_t rows = pf_launch_rows(plan);
  if (rows == 0 || plan.n_total > INT_MAX) return QS_ERR_UNSUPPORTED;
  p.ldx = ldx;
  p.K = (int)K;
  p.T = (int)(K / 64);
  p.S = plan.S;
  p.TS = (int)cdiv(p.T, plan.S);
  p.tiles_n = (int)plan.tiles_n;
  p.n_lin = n_lin;
  p.n_total = (int)plan.n_total;
  p.vec = vec;
  p.part = static_cast<float*>(workspace);
  int64_t tb = 0, nb = 0;
  for (int i = 0; i < n_lin; ++i) {
    p.lin[i] = PfLin{lin[i].codes, lin[i].scales, lin[i].y, lin[i].ldy, (int)N[i], (int)tb, (int)nb};
    if (P == 1) {
      tb += cdiv(N[i], 16 * sh.NTP * sh.WN);
      nb += cdiv(N[i], 4) * 4;
    }
  }
  for (int64_t m0 = 0; m0 < M; m0 += rows) {
    p.M = (int)std::min(rows, M - m0);
    p.tiles_m = (int)cdiv(p.M, 16 * sh.MT);
    p.x = static_cast<const char*>(x) + m0 * ldx * es;
    for (int i = 0; i < n_lin; ++i)
      if (lin[i].y) p.lin[i].y = static_cast<char*>(lin[i].y) + m0 * lin[i].ldy * es;
    if (P == 2) pf_launch<2, QS_BF16>(p, plan.shape, s);
    else if (f32) pf_launch<1, QS_F32>(p, plan.shape, s);
    else if (x_dtype == QS_F16) pf_launch<1, QS_F16>(p, plan.shape, s);
    else pf_launch<1, QS_BF16>(p, plan.shape, s);
  }
  return hip_check(hipGetLastError(), "k_prefill launch");
}

}  // namespace qs

using namespace qs;

extern "C" int64_t qs_qrow_prefill_plan(int x_dtype, int64_t M, int n_linear, const int64_t* N, int64_t K, int swiglu,
                                        int split, int32_t* tile) {
  if (!N || n_linear < 1 || n_linear > 4 || M < 1 || K < 64) return -1;
  const int P = swiglu ? 2 : 1;
  const PfPlan plan = pf_plan(x_dtype == QS_F32, M, n_linear, N, K, P, split != 0);
  if (tile) {
    const PfShape& sh = kPfShapes[plan.shape];
    tile[0] = 16 * sh.MT;
    tile[1] = 16 * sh.NTP / P * sh.WN;
    tile[2] = sh.WK;
    tile[3] = plan.S;
  }
  if (pf_launch_rows(plan) == 0 || plan.n_total > INT_MAX) return -1;
  if (!prefill_faster(x_dtype, M, n_linear, N, K, P, split != 0)) return -1;
  return plan.S > 1 ? plan.S * P * M * plan.n_total * 4 : 0;
}

extern "C" size_t qs_qrow_prefill_workspace_bytes(int x_dtype, int64_t M, int n_linear, const int64_t* N, int64_t K,
                                                  int swiglu) {
  if (!N || n_linear < 1 || n_linear > 4 || M < 1 || K < 64) return 0;
  const int P = swiglu ? 2 : 1;
  const PfPlan plan = pf_plan(x_dtype == QS_F32, M, n_linear, N, K, P, true);
  return plan.S > 1 ? (size_t)plan.S * P * M * plan.n_total * 4 : 0;
}

namespace {

int prefill_check(const void* x, int x_dtype, int64_t ldx, int64_t M, int64_t K) {
  if (!x) return fail(QS_ERR_INVALID, "qrow prefill: null activations");
  if (x_dtype != QS_BF16 && x_dtype != QS_F16 && x_dtype != QS_F32)
    return fail(QS_ERR_INVALID, "qrow prefill: activations BF16, F16 or F32");
  if (M < 1 || K < 1 || ldx < K) return fail(QS_ERR_INVALID, "qrow prefill: bad M, K or ldx");
  if (M > (int64_t)1 << 30 || K > (int64_t)1 << 30) return fail(QS_ERR_LIMIT, "qrow prefill: dimension exceeds 2^30");
  return QS_OK;
}

int prefill_status(int st) {
  if (st != QS_ERR_UNSUPPORTED) return st;
  return fail(QS_ERR_UNSUPPORTED, "qrow prefill: needs K %% 64 == 0 and 16-byte aligned activation and weight rows");
}

}  // namespace

extern "C" int qs_qrow_matmul_prefill(const void* x, int x_dtype, int64_t ldx, int n_linear,
                                      const int8_t* const* codes, const float* const* scales, void* const* y,
                                      const int64_t* ldy, const int64_t* N, int64_t M, int64_t K, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  int st = prefill_check(x, x_dtype, ldx, M, K);
  if (st) return st;
  if (n_linear < 1 || n_linear > 4) return fail(QS_ERR_LIMIT, "qrow prefill: 1..4 linears");
  if (!codes || !scales || !y || !ldy || !N) return fail(QS_ERR_INVALID, "qrow prefill: null array");
  QrowPrefillLin lin[4];
  for (int i = 0; i < n_linear; ++i) {
    if (!codes[i] || !scales[i] || !y[i]) return fail(QS_ERR_INVALID, "qrow prefill: null pointer in linear %d", i);
    if (N[i] <= 0 || N[i] > ((int64_t)1 << 30) || ldy[i] < N[i])
      return fail(QS_ERR_INVALID, "qrow prefill: bad N/ldy for linear %d", i);
    lin[i] = QrowPrefillLin{codes[i], scales[i], y[i], ldy[i], N[i]};
  }
  return prefill_status(run_prefill(x, x_dtype, ldx, n_linear, lin, 1, M, K,
                                    workspace_bytes ? workspace : nullptr, workspace_bytes,
                                    static_cast<hipStream_t>(stream)));
}

extern "C" int qs_qrow_swiglu_prefill(const void* x, int64_t ldx, const int8_t* gate_codes, const float* gate_scales,
                                      const int8_t* up_codes, const float* up_scales, void* y, int64_t ldy, int64_t M,
                                      int64_t N, int64_t K, void* workspace, size_t workspace_bytes, void* stream) {
  int st = prefill_check(x, QS_BF16, ldx, M, K);
  if (st) return st;
  if (!gate_codes || !gate_scales || !up_codes || !up_scales || !y)
    return fail(QS_ERR_INVALID, "swiglu prefill: null pointer");
  if (N <= 0 || N > ((int64_t)1 << 30) || ldy < N) return fail(QS_ERR_INVALID, "swiglu prefill: bad N/ldy");
  const QrowPrefillLin lin[2] = {{gate_codes, gate_scales, y, ldy, N}, {up_codes, up_scales, nullptr, 0, N}};
  return prefill_status(run_prefill(x, QS_BF16, ldx, 2, lin, 2, M, K, workspace_bytes ? workspace : nullptr,
                                    workspace_bytes, static_cast<hipStream_t>(stream)));
}
