// Linears with 16-bit weights and 2 to 15 fp32 activation rows (src/kernels.c:
// 129-151), above all the language-model head of batched decoding: the
// activations in registers.
//
//   C[m][n] = sum_k A[m][k] * B[n][k], fp32 FMAs
//
// The fused GEMV (gemv_impl.h) reads the activations of every weight chunk
// again, 32 bytes per row and 16-byte chunk: at 8 rows the L1 delivers 16 bytes
// for each byte of weights, and the head of 151936 x 896 took 153 us where its
// 272 MB take about 45 us.  Here a lane keeps the MT rows' values of its CH
// 8-element chunks (chunk lane + 64 c of a row), so a weight row costs its
// 1 KB loads, one convert per weight and MT FMAs; two rows per step, the next
// two rows' loads in flight.  A wave's MT sums of a row meet by half-wave
// swaps, which also spread them: 18 instructions for 8 sums where a tree each
// would take 48.  Every lane adds at most 8 CH products in order before the
// tree (the fused GEMV up to 64), so the error against 64 bits is no larger:
// 9.8e-8 of the result against 1.46e-7 at K = 896, 1.12e-7 both at 1536.  The
// matrix cores would need the rows' 16-bit parts, whose products' sums come
// out further off (2.8e-7 and 3.6e-7).
//
// 151936 x 896 fp16, 8 rows: 153 -> 64 us (4.3 TB/s), where a step's 300
// vector instructions per two weight rows are about 30 us and the loads of 2
// waves per SIMD (170 registers) bound it; 4 rows: 99 -> 48 us (5.7 TB/s).
#include "ec_device.h"
#include "ec_kernels.h"

namespace ec {

namespace {

constexpr int kRxRows = 2;  // weight rows per wave and step

// a and b with a's upper (odd) half exchanged for b's lower (even) one, halves
// of 32 (16) lanes: the sum holds a's total of both in one half and b's in the other
__device__ __forceinline__ float swap_add32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float swap_add16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}

// the wave's sums of acc[0 .. MT): lane l ends with that of row
// (l >> 5 & 1) + 2 (l >> 4 & 1) + 4 (l >> 3 & 1) (MT 4: without the last)
template <int MT>
__device__ __forceinline__ float spread_sum(const float (&acc)[MT], int lane) {
  float h[MT / 2];
#pragma unroll
  for (int i = 0; i < MT / 2; i++) h[i] = swap_add32(acc[2 * i], acc[2 * i + 1]);
  float q[MT / 4];
#pragma unroll
  for (int i = 0; i < MT / 4; i++) q[i] = swap_add16(h[2 * i], h[2 * i + 1]);
  float v;
  if constexpr (MT == 8) {
    const bool up = lane & 8;
    v = (up ? q[1] : q[0]) + dpp_mov<0x128>(up ? q[0] : q[1]);  // row_ror:8
  } else {
    v = q[0] + dpp_mov<0x128>(q[0]);
  }
  v = v + dpp_mov<0xB1>(v);    // quad_perm [1,0,3,2]
  v = v + dpp_mov<0x4E>(v);    // quad_perm [2,3,0,1]
  return v + dpp_mov<0x141>(v);  // row_half_mirror
}

// one block: 4 waves, each on its own pairs of weight rows, grid-stride;
// blockIdx.y: a tile of MT activation rows
template <bool BF16, int MT, int CH>
__global__ __launch_bounds__(256, 2) void gemv_regs_kernel(GemvArgs a) {
  constexpr int R = kRxRows;
  const int t = threadIdx.x, lane = t & 63;
  const int K = a.K, N = a.N, nch = K / 8;
  const int m0 = blockIdx.y * MT, mc = min(MT, a.M - m0);
  const int step = 4 * R * gridDim.x;
  const int n0 = __builtin_amdgcn_readfirstlane(R * (4 * blockIdx.x + (t >> 6)));
  const uint16_t *W = (const uint16_t *)a.W;

  // chunks past the row are loaded clamped and count as zero
  int ko[CH];
  bool in[CH];
#pragma unroll
  for (int c = 0; c < CH; c++) {
    in[c] = lane + 64 * c < nch;
    ko[c] = 8 * min(lane + 64 * c, nch - 1);
  }
  v4u wn[R][CH];
  auto load = [&](int n) {
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int c = 0; c < CH; c++)
        wn[r][c] = __builtin_nontemporal_load(
            reinterpret_cast<const v4u *>(W + (size_t)min(n + r, N - 1) * K + ko[c]));
  };
  load(min(n0, N - 1));
  float x[CH][8][MT];
#pragma unroll
  for (int c = 0; c < CH; c++)
#pragma unroll
    for (int m = 0; m < MT; m++) {
      const float *p = (const float *)a.A + (size_t)(m0 + min(m, mc - 1)) * a.lda + ko[c];
      const float4 u = *reinterpret_cast<const float4 *>(p), v = *reinterpret_cast<const float4 *>(p + 4);
      const float e[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 8; i++) x[c][i][m] = in[c] ? e[i] : 0.0f;
    }
  const int om = ((lane >> 5) & 1) + 2 * ((lane >> 4) & 1) + (MT == 8 ? 4 * ((lane >> 3) & 1) : 0);
  const bool writes = (lane & (MT == 8 ? 7 : 15)) == 0 && om < mc;
  float *out = a.out + (size_t)(m0 + min(om, mc - 1)) * a.ldo;

#pragma unroll 1
  for (int n = n0; n < N; n += step) {
    v4u w[R][CH];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int c = 0; c < CH; c++) w[r][c] = in[c] ? wn[r][c] : v4u{0, 0, 0, 0};
    load(min(n + step, N - 1));
#pragma unroll
    for (int r = 0; r < R; r++) {
      float acc[MT];
#pragma unroll
      for (int m = 0; m < MT; m++) acc[m] = 0.0f;
#pragma unroll
      for (int c = 0; c < CH; c++) {
        const uint32_t hw[4] = {w[r][c].x, w[r][c].y, w[r][c].z, w[r][c].w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const float f = w2f<BF16>((uint16_t)(i & 1 ? hw[i / 2] >> 16 : hw[i / 2] & 0xffffu));
#pragma unroll
          for (int m = 0; m < MT; m++) acc[m] = __builtin_fmaf(x[c][i][m], f, acc[m]);
        }
      }
      const float v = spread_sum<MT>(acc, lane);
      if (writes && n + r < N) out[n + r] = v;
    }
  }
}

template <bool BF16, int MT, int CH>
hipError_t launch(const GemvArgs &a, hipStream_t s) {
  const int pairs = (a.N + 4 * kRxRows - 1) / (4 * kRxRows), mt = (a.M + MT - 1) / MT;
  // resident blocks: 2 per CU by registers
  const int gx = min(pairs, max(1, 512 / mt));
  klaunch((gemv_regs_kernel<BF16, MT, CH>), dim3(gx, mt), dim3(256), 0, s, a);
  return hipGetLastError();
}

template <bool BF16>
hipError_t launch_wt(const GemvArgs &a, hipStream_t s) {
  const int ch = (a.K / 8 + 63) / 64;
  if (a.M <= 4) {
    switch (ch) {
      case 1: return launch<BF16, 4, 1>(a, s);
      case 2: return launch<BF16, 4, 2>(a, s);
      case 3: return launch<BF16, 4, 3>(a, s);
    }
  } else {
    switch (ch) {
      case 1: return launch<BF16, 8, 1>(a, s);
      case 2: return launch<BF16, 8, 2>(a, s);
      case 3: return launch<BF16, 8, 3>(a, s);
    }
  }
  return hipErrorInvalidValue;
}

}  // namespace

bool gemv_regs_ok(const GemvArgs &a, int wt) {
  return (wt == WT_F16 || wt == WT_BF16) && a.M >= 1 && a.N >= 1 && a.K >= 8 && a.K <= 3 * 512 && a.K % 8 == 0 &&
         a.lda % 4 == 0 && !((uintptr_t)a.A & 15u) && !((uintptr_t)a.W & 15u) && !a.cand && !a.bias;
}

// From 4 rows on, and from 2 for wide outputs, of rows that give most lanes of a
// wave a chunk (a row has 64 lanes here, in the fused GEMV as few as it needs).
// Fused GEMV and this kernel, us, K x N: 1536 x 4096 5.0 and 6.2 (2 rows), 5.8
// and 6.3 (3), 6.5 and 6.3 (4), 9.7 and 7.8 (8), 17.5 and 9.5 (15); 896 x 896
// 5.9 and 4.3 (4), 9.8 and 4.8 (8); 896 x 9728 6.6 and 5.9 (2), 13.7 and 8.1 (8);
// 896 x 151936 62 and 47 (2), 99 and 48 (4), 153 and 64 (8), 282 and 124 (15);
// 128 x 20000 4.8 and 5.9 (2), 6.3 and 7.9 (5), 11.2 and 12.6 (12).
bool gemv_regs_faster(const GemvArgs &a, int wt) {
  return gemv_regs_ok(a, wt) && a.K >= 192 && (a.M >= 4 || (a.M >= 2 && a.N >= 8192));
}

hipError_t gemv_regs(const GemvArgs &a, int wt, hipStream_t s) {
  if (!gemv_regs_ok(a, wt)) return hipErrorInvalidValue;
  return wt == WT_BF16 ? launch_wt<true>(a, s) : launch_wt<false>(a, s);
}

}  // namespace ec
