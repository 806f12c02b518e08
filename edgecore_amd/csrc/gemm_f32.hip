// Linears with 16-bit weights and fp32 activation rows (src/kernels.c:129-151)
// whose operands the vector kernels cannot read: rows of any length from 8
// elements, operands at any address.
//
//   C[m][n] = sum_k A[m][k] * B[n][k], fp32 FMAs
//
// The products run on the matrix cores' fp32 form (v_mfma_f32_16x16x4_f32),
// the weights converted to fp32 as they are staged.  So a product has all 24
// bits of its activation, whatever the rest of the row holds, and a value that
// is not finite reaches its own outputs as in a sequential fp32 sum.  The
// 16-bit parts of gemm_mfma.hip hold neither: two fp16 parts under one scale
// per row carry 22 bits of the largest values and fewer of the small ones (a
// row with one value 1e8 times the others, which meets a zero weight, came out
// 7e-5 off, 1e10 times 9e-3), three bf16 parts lose the last bits below 2^-110.
// It needs no workspace: a captured call names the caller's buffers alone.
//
// Two kernels:
//   gemm_f32_rows_kernel, up to 32 rows: a block of up to 16 waves per 16
//     columns, each lane loading its fragments straight from global memory (8
//     weights and 8 activations per row of its K step of 32), the K steps
//     dealt out to the waves, whose tiles meet in LDS;
//   gemm_f32_tile_kernel: 4 waves, 32 x 64 outputs, K in stages of 64 elements
//     through two LDS buffers, the next two stages in registers.
// Bound by the fp32 matrix rate (157 TFLOP/s nominal; 90 at 600 x 1001 x 9001)
// for large products, by the stages' latency for small ones, which give a CU one
// or two tiles.  Larger tiles measured no better: 64 x 64 and 64 x 128, us, at
// 600 x 1001 x 9001 117 to 131 and 126 (32 x 64: 120), at 333 x 1001 x 777 28
// and 48 (17.4).  One thread per output, which these shapes took before, took
// 963 us there.
// A fragment register holds k = 4 (l / 16) + i for lane l and instruction i of
// a 16-element slice, so that a lane reads its four values in one 16-byte load;
// any order of k does for a sum as long as both operands have the same.
#include "ec_device.h"
#include "ec_kernels.h"

namespace ec {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
// 16 bytes at any address (gfx950 loads them unaligned in one instruction)
typedef v4u v4u_u __attribute__((aligned(1)));
typedef v4f v4f_u __attribute__((aligned(1)));

// The 8 elements from c of a row of K, as loaded from min(c, K - 8): the first
// cut = c + 8 - K of them belong to the elements before c (all of them past the
// row) and count as zero.  Both operands' are loaded from the same place, so
// element j of one still meets element j of the other.
__device__ __forceinline__ int at8(int c, int K) { return min(c, K - 8); }

template <bool BF16>
__device__ __forceinline__ void to_f32(v4u h, float *f) {
  const uint32_t w[4] = {h.x, h.y, h.z, h.w};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    f[2 * i] = w2f<BF16>((uint16_t)(w[i] & 0xffffu));
    f[2 * i + 1] = w2f<BF16>((uint16_t)(w[i] >> 16));
  }
}

__device__ __forceinline__ v4f mma(float a, float b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// the value of output [m][n] from its sum v (SwiGLU: gate v and up u)
template <int EPI>
__device__ __forceinline__ void finish(const GemvArgs &a, int m, int n, float v, float u, const uint64_t *etab) {
  float *o = a.out + (size_t)m * a.ldo + n;
  if constexpr (EPI == EPI_SWIGLU) {
    v = silu(v, etab) * u;
  } else {
    if (a.bias) v = v + a.bias[n];
    if constexpr (EPI == EPI_RESID) v = *o + v;
    if constexpr (EPI == EPI_GELU) v = gelu_new(v);
  }
  *o = v;
}

constexpr int kRowWaves = 16;  // waves per block, at most

template <bool BF16, int TI, int EPI>
__global__ __launch_bounds__(64 * kRowWaves) void gemm_f32_rows_kernel(GemvArgs a) {
  constexpr bool SWI = EPI == EPI_SWIGLU;
  constexpr int NB = SWI ? 2 : 1;
  constexpr int U = TI * NB == 1 ? 4 : 2;  // K steps per wave in flight
  __shared__ v4f part[kRowWaves][TI][NB][64];
  __shared__ uint64_t etab[32];
  const int t = threadIdx.x, lane = t & 63, nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const int M = a.M, K = a.K, N = a.N, n0 = 16 * blockIdx.x, ns = (K + 31) / 32;
  if (SWI && t < 32) etab[t] = ec_exp2_32[t];

  const float *arow[TI];
  const uint16_t *brow[NB];
#pragma unroll
  for (int i = 0; i < TI; i++) arow[i] = (const float *)a.A + (size_t)min(16 * i + lr, M - 1) * a.lda;
#pragma unroll
  for (int j = 0; j < NB; j++)
    brow[j] = (const uint16_t *)(j ? a.W2 : a.W) + (size_t)min(n0 + lr, N - 1) * K;
  v4f acc[TI][NB];
#pragma unroll
  for (int i = 0; i < TI; i++)
#pragma unroll
    for (int j = 0; j < NB; j++) acc[i][j] = v4f{0, 0, 0, 0};

  for (int sb = wave; sb < ns; sb += nw * U) {
    v4f fa[U][TI][2];
    v4u fb[U][NB];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int st = sb + nw * u;  // uniform
      if (st < ns) {
        const int s = at8(32 * st + 8 * lq, K);
#pragma unroll
        for (int j = 0; j < NB; j++) fb[u][j] = *reinterpret_cast<const v4u_u *>(brow[j] + s);
#pragma unroll
        for (int i = 0; i < TI; i++) {
          fa[u][i][0] = *reinterpret_cast<const v4f_u *>(arow[i] + s);
          fa[u][i][1] = *reinterpret_cast<const v4f_u *>(arow[i] + s + 4);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int st = sb + nw * u;
      if (st < ns) {
        const int cut = 32 * st + 8 * lq + 8 - K;
        if (32 * st + 32 > K) {  // uniform: the row ends inside this step
#pragma unroll
          for (int i = 0; i < TI; i++)
#pragma unroll
            for (int e = 0; e < 8; e++) fa[u][i][e / 4][e % 4] = e >= cut ? fa[u][i][e / 4][e % 4] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < NB; j++) {
          float fw[8];
          to_f32<BF16>(fb[u][j], fw);
          if (32 * st + 32 > K) {  // a weight that is not finite would make NaN of a zero activation
#pragma unroll
            for (int e = 0; e < 8; e++) fw[e] = e >= cut ? fw[e] : 0.0f;
          }
          // the step's sums in two chains of 16 products
          v4f c[TI][2];
#pragma unroll
          for (int i = 0; i < TI; i++) c[i][0] = c[i][1] = v4f{0, 0, 0, 0};
#pragma unroll
          for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
              for (int h = 0; h < 2; h++) c[i][h] = mma(fa[u][i][h][e], fw[4 * h + e], c[i][h]);
#pragma unroll
          for (int i = 0; i < TI; i++) acc[i][j] = acc[i][j] + (c[i][0] + c[i][1]);
        }
      }
    }
  }

#pragma unroll
  for (int i = 0; i < TI; i++)
#pragma unroll
    for (int j = 0; j < NB; j++) part[wave][i][j][lane] = acc[i][j];
  __syncthreads();
  // output q: accumulator register r of lane q % 64 of fragment i
  for (int q = t; q < 256 * TI; q += blockDim.x) {
    const int i = q >> 8, r = (q >> 6) & 3, m = 16 * i + 4 * lq + r, n = n0 + lr;
    if (m >= M || n >= N) continue;
    float v[2] = {0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < NB; j++) {
      // the even and the odd waves' sums, each in order
      float w1 = 0.0f;
      for (int w = 0; w < nw; w += 2) {
        v[j] = v[j] + part[w][i][j][lane][r];
        if (w + 1 < nw) w1 = w1 + part[w + 1][i][j][lane][r];
      }
      v[j] = v[j] + w1;
    }
    finish<EPI>(a, m, n, v[0], v[1], etab);
  }
}

constexpr int kFBM = 32, kFBN = 64, kFBK = 64;  // a block's tile, elements of K per stage

// 2 x 2 waves of 16 rows and two 16-column tiles (SwiGLU: one of gate rows, one
// of up rows)
template <bool BF16, int EPI>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(GemvArgs a) {
  constexpr bool SWI = EPI == EPI_SWIGLU;
  constexpr int BM = kFBM, BN = kFBN, BK = kFBK, NOUT = SWI ? BN / 2 : BN, JO = SWI ? 1 : 2;
  constexpr int PITCH = BK + 4;             // floats per LDS row: 8 consecutive rows' 16-byte reads on distinct banks
  constexpr int CA = BK / 4, CB = BK / 8;   // 4-activation and 8-weight chunks per row
  constexpr int ACH = BM * CA / 256, BCH = BN * CB / 256;  // of them per thread
  constexpr int PF = 2;                                    // stages in registers
  __shared__ __attribute__((aligned(16))) float la[2][BM * PITCH], lb[2][BN * PITCH];
  __shared__ uint64_t etab[32];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wm = wave >> 1, wn = wave & 1;
  const int lr = lane & 15, lq = lane >> 4;
  const int M = a.M, K = a.K, N = a.N, ns = (K + BK - 1) / BK;
  // XCD-aware tile order: block b runs on XCD b % 8, which takes a contiguous
  // share of the weight rows with every row tile
  const int nM = (M + BM - 1) / BM, nN = (N + NOUT - 1) / NOUT, T = nM * nN, per = (T + 7) / 8;
  const int tl = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (tl >= T) return;
  const int m0 = (tl % nM) * BM, n0 = (tl / nM) * NOUT;
  if (SWI && t < 32) etab[t] = ec_exp2_32[t];

  const float *arow[ACH];
  const uint16_t *brow[BCH];
  const int ac = t % CA, bc = t % CB;  // this thread's chunk of a row
#pragma unroll
  for (int j = 0; j < ACH; j++)
    arow[j] = (const float *)a.A + (size_t)min(m0 + t / CA + 256 / CA * j, M - 1) * a.lda;
#pragma unroll
  for (int j = 0; j < BCH; j++) {
    const int r = t / CB + 256 / CB * j;
    const bool up = SWI && r >= BN / 2;
    brow[j] = (const uint16_t *)(up ? a.W2 : a.W) + (size_t)min(n0 + (up ? r - BN / 2 : r), N - 1) * K;
  }
  v4f ra[PF][ACH];
  v4u rb[PF][BCH];
  auto load = [&](int p, int k0) {
    int sa = k0 + 4 * ac, sb = k0 + 8 * bc;
    if (k0 + BK > K) {  // uniform: the row ends inside this stage
      sa = at8(k0 + 8 * (ac >> 1), K) + 4 * (ac & 1);
      sb = at8(sb, K);
    }
#pragma unroll
    for (int j = 0; j < ACH; j++) ra[p][j] = *reinterpret_cast<const v4f_u *>(arow[j] + sa);
#pragma unroll
    for (int j = 0; j < BCH; j++) rb[p][j] = *reinterpret_cast<const v4u_u *>(brow[j] + sb);
  };
  auto store = [&](int p, int k0, int buf) {
    float f[BCH][8];
#pragma unroll
    for (int j = 0; j < BCH; j++) to_f32<BF16>(rb[p][j], f[j]);
    if (k0 + BK > K) {
      const int cuta = k0 + 8 * (ac >> 1) + 8 - K - 4 * (ac & 1), cutb = k0 + 8 * bc + 8 - K;
#pragma unroll
      for (int j = 0; j < ACH; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) ra[p][j][e] = e >= cuta ? ra[p][j][e] : 0.0f;
#pragma unroll
      for (int j = 0; j < BCH; j++)
#pragma unroll
        for (int e = 0; e < 8; e++) f[j][e] = e >= cutb ? f[j][e] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < ACH; j++)
      *reinterpret_cast<v4f *>(&la[buf][(t / CA + 256 / CA * j) * PITCH + 4 * ac]) = ra[p][j];
#pragma unroll
    for (int j = 0; j < BCH; j++) {
      float *dst = &lb[buf][(t / CB + 256 / CB * j) * PITCH + 8 * bc];
      *reinterpret_cast<v4f *>(dst) = v4f{f[j][0], f[j][1], f[j][2], f[j][3]};
      *reinterpret_cast<v4f *>(dst + 4) = v4f{f[j][4], f[j][5], f[j][6], f[j][7]};
    }
  };
  // first LDS row of each of this wave's column tiles
  const int bt[2] = {SWI ? 16 * wn : 32 * wn, SWI ? BN / 2 + 16 * wn : 32 * wn + 16};
  v4f acc[2] = {};

#pragma unroll
  for (int p = 0; p < PF; p++) load(p, BK * min(p, ns - 1));
#pragma unroll 1
  for (int s0 = 0; s0 < ns; s0 += PF) {
#pragma unroll
    for (int p = 0; p < PF; p++) {
      const int s = s0 + p, buf = p & 1;
      if (s < ns) {  // uniform
        // written two stages ago: every wave has read it by the last barrier
        store(p, BK * s, buf);
        load(p, BK * min(s + PF, ns - 1));
        __syncthreads();
        const float *pa = la[buf] + (wm * 16 + lr) * PITCH + 4 * lq, *pb = lb[buf] + lr * PITCH + 4 * lq;
        // the stage's sums in two chains of 32 products, added to the total:
        // short chains round less than one over all of K, and the matrix
        // instructions of four chains follow one another without a wait
        v4f c[2][2] = {};
#pragma unroll
        for (int kk = 0; kk < BK; kk += 16) {
          const v4f fa = *reinterpret_cast<const v4f *>(pa + kk);
          v4f fb[2];
#pragma unroll
          for (int j = 0; j < 2; j++) fb[j] = *reinterpret_cast<const v4f *>(pb + bt[j] * PITCH + kk);
#pragma unroll
          for (int e = 0; e < 4; e++)
#pragma unroll
            for (int j = 0; j < 2; j++) c[e & 1][j] = mma(fa[e], fb[j][e], c[e & 1][j]);
        }
#pragma unroll
        for (int j = 0; j < 2; j++) acc[j] = acc[j] + (c[0][j] + c[1][j]);
      }
    }
  }

  const int row0 = m0 + 16 * wm + 4 * lq, col0 = n0 + (SWI ? 16 * wn : 32 * wn) + lr;
#pragma unroll
  for (int j = 0; j < JO; j++) {
    const int n = col0 + 16 * j;
    if (n >= N) continue;
#pragma unroll
    for (int r = 0; r < 4; r++)
      if (row0 + r < M) finish<EPI>(a, row0 + r, n, acc[j][r], SWI ? acc[1][r] : 0.0f, etab);
  }
}

template <bool BF16, int TI, int EPI>
hipError_t launch_rows(const GemvArgs &a, hipStream_t s) {
  // two or more K steps per wave
  const int ns = (a.K + 31) / 32, nw = max(4, min(kRowWaves, (ns + 1) / 2));
  klaunch((gemm_f32_rows_kernel<BF16, TI, EPI>), dim3((a.N + 15) / 16), dim3(64 * nw), 0, s, a);
  return hipGetLastError();
}

template <bool BF16, int EPI>
hipError_t launch_tile(const GemvArgs &a, hipStream_t s) {
  constexpr int NOUT = EPI == EPI_SWIGLU ? kFBN / 2 : kFBN;
  const int T = ((a.M + kFBM - 1) / kFBM) * ((a.N + NOUT - 1) / NOUT);
  klaunch((gemm_f32_tile_kernel<BF16, EPI>), dim3(8 * ((T + 7) / 8)), dim3(256), 0, s, a);
  return hipGetLastError();
}

// Up to 32 rows without stages, but for wide outputs, whose rows stream better
// through the stages: rows x K x N, us without and with: 8 x 1001 x 777 6.6 and
// 16.6, 4 x 1001 x 9001 13.5 and 18.1, 16 x 4001 x 12001 54 and 61; 8 x 897 x
// 17920 29.5 and 24.5, 3 x 1537 x 17001 44.5 and 37.8, 32 x 1501 x 16390 41.4
// and 36.9.
template <bool BF16, int EPI>
hipError_t launch_epi(const GemvArgs &a, hipStream_t s) {
  if (a.M > 32 || a.N >= 16384) return launch_tile<BF16, EPI>(a, s);
  return a.M <= 16 ? launch_rows<BF16, 1, EPI>(a, s) : launch_rows<BF16, 2, EPI>(a, s);
}

template <bool BF16>
hipError_t launch_wt(const GemvArgs &a, int epi, hipStream_t s) {
  switch (epi) {
    case EPI_STORE:
    case EPI_BIAS: return launch_epi<BF16, EPI_STORE>(a, s);
    case EPI_RESID:
    case EPI_BIAS_RESID: return launch_epi<BF16, EPI_RESID>(a, s);
    case EPI_GELU:
    case EPI_BIAS_GELU: return launch_epi<BF16, EPI_GELU>(a, s);
    case EPI_SWIGLU: return launch_epi<BF16, EPI_SWIGLU>(a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace

bool gemm_f32_ok(const GemvArgs &a, int wt, int epi) {
  return (wt == WT_F16 || wt == WT_BF16) && a.M >= 1 && a.N >= 1 && a.K >= 8 && a.lda >= a.K && a.A && a.W &&
         !a.cand && !a.ws && !a.ws2 && (epi != EPI_SWIGLU || a.W2) && epi >= EPI_STORE && epi <= EPI_BIAS_GELU;
}

hipError_t gemm_f32(const GemvArgs &a, int wt, int epi, hipStream_t s) {
  if (!gemm_f32_ok(a, wt, epi)) return hipErrorInvalidValue;
  GemvArgs q = a;
  // the 16-bit linears add a bias only in their BIAS epilogues
  if (epi != EPI_BIAS && epi != EPI_BIAS_RESID && epi != EPI_BIAS_GELU) q.bias = nullptr;
  return wt == WT_BF16 ? launch_wt<true>(q, epi, s) : launch_wt<false>(q, epi, s);
}

}  // namespace ec
