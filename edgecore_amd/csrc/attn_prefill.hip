// Causal attention of a prefill: M tokens of one slot at consecutive positions
// p0 .. p0+M-1, whose k / v rows are already in the fp16 cache (RoPE and the
// append ran first).  This is the reference's per-slot prefill loop
// (src/gpt2.c:527-557 GPT-2, 744-777 Qwen2 GQA) with its arithmetic order:
//
//   s_p   = (float)((double)(sequential fp32 sum over d of q_d * k_p[d]) * inv_hd)
//   e_p   = expf(s_p - max_p s_p)           (glibc-exact expf, ec_expf.h)
//   sum   = sum_p (double)e_p
//   pr_p  = (float)((double)e_p * (1 / sum))
//   out_d = sequential fp32 sum over p (ascending) of pr_p * v_p[d]
//
// Every product is rounded before its add, as in the reference's build.  The
// double sum runs in a tree order (lane-strided, then the wave); the
// reference's order differs from it by the last bits of a double, below what
// the float rounding of pr_p resolves except in rare ties.
//
// Two kernels: attn_prefill_mm_kernel (below), with the products on the matrix
// cores, for spans of up to 4096 positions, and attn_prefill_kernel for longer
// ones and for prompts that are few blocks (mm_takes).
//
// attn_prefill_kernel: one block takes one query head and NW consecutive
// tokens, one per wave (8, or 4 when the scores of 8 do not fit the LDS).  The
// keys of all of them are staged through LDS 64 positions at a time, converted
// to fp32 once for the block:
//   - scores: lane = position; each lane runs its position's sequential dot
//     off its K row (q in registers); K rows are head_dim + 4 floats apart, so
//     the 16-byte reads of 8 lanes hit distinct banks;
//   - softmax: per token, inside its wave, four of a lane's positions per
//     step (expf without branches);
//   - output: lane = element d; the wave adds pr_p * v_p[d] in position order
//     from V tiles staged transposed (a lane's positions contiguous, 16-byte
//     reads of four), the probabilities read by quad, the next quad's reads in
//     flight during the current quad's adds.
// The blocks with the longest key ranges start first; the grid is (head,
// token group), which spreads the blocks over all 8 XCDs.
#include <cfloat>
#include <type_traits>

#include "ec_device.h"
#include "ec_expf.h"
#include "ec_kernels.h"

namespace ec {

namespace {

constexpr int kPfTile = 64;  // positions per staged K / V tile

// V tiles are staged transposed: element d of the tile's position r at
// tile[pf_vrow(d) + r].  Rows are 68 floats apart plus 4 more every 8 rows,
// so that the 4-byte staging writes (32 lanes: 4 positions x 8 chunks of 8
// elements) and the 16-byte reads of 8 consecutive rows (served 8 lanes at a
// time) both hit distinct banks.
constexpr int pf_vrow(int d) { return d * (kPfTile + 4) + 4 * (d >> 3); }

// NW waves per block, each with one token (consecutive)
template <int HD, int NW>
__global__ __launch_bounds__(NW * 64) void attn_prefill_kernel(AttnArgs a, int ngroups, int nsc) {
  constexpr int NT = NW * 64;
  constexpr int KP = HD + 4;                   // floats per staged row
  constexpr int CPR = HD / 8;                  // 16-byte chunks (8 halves) per cache row
  constexpr int TCH = kPfTile * CPR;           // chunks per tile
  constexpr int NCH = (TCH + NT - 1) / NT;     // chunks per thread
  constexpr int DPL = HD > 64 ? HD / 64 : 1;   // output elements per lane
  constexpr int VJ = pf_vrow(64);              // transposed V: element d + 64 is VJ floats after d
  static_assert(pf_vrow(HD - 1) + kPfTile + 4 <= (kPfTile + 4) * KP, "transposed V tile fits the tile area");
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float *tile = lds;  // [kPfTile + 4][KP]: K rows (4 spare rows for look-ahead reads), then transposed V
  __shared__ uint64_t etab[32];

  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int h = blockIdx.x;
  const int kvh = h * a.KVH / a.H;
  const int m0 = (ngroups - 1 - (int)blockIdx.y) * NW;  // longest key ranges first
  const int slot = ld_uniform(a.slot + m0);
  const int pos_hi = ld_uniform(a.pos + min(m0 + NW - 1, a.M - 1));
  const int lo0 = a.window > 0 ? max(0, ld_uniform(a.pos + m0) - a.window + 1) : 0;
  // this wave's token (tail waves repeat the last token and store nothing)
  const bool act = m0 + w < a.M;
  const int mq = min(m0 + w, a.M - 1);
  const int pos = ld_uniform(a.pos + mq);
  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  float *sc = lds + (kPfTile + 4) * KP + w * nsc;  // its scores, then probabilities, at index p - lo0
  if (t < 32) etab[t] = ec_exp2_32[t];
  const size_t cbase = (size_t)slot * a.C * a.kv + (size_t)kvh * HD;
  const uint16_t *Kc = a.kc + cbase, *Vc = a.vc + cbase;

  // q rows of the block's tokens through the (still free) tile area into
  // each wave's registers
  for (int e = t; e < NW * HD / 4; e += NT) {
    const int r = e / (HD / 4), c4 = e - r * (HD / 4);
    const float *qrow = a.q + (size_t)min(m0 + r, a.M - 1) * a.ldq + (size_t)h * HD;
    *reinterpret_cast<float4 *>(tile + r * HD + 4 * c4) = *reinterpret_cast<const float4 *>(qrow + 4 * c4);
  }
  __syncthreads();
  float q[HD];
#pragma unroll
  for (int c4 = 0; c4 < HD / 4; c4++) {
    const float4 v = *reinterpret_cast<const float4 *>(tile + w * HD + 4 * c4);
    q[4 * c4] = v.x;
    q[4 * c4 + 1] = v.y;
    q[4 * c4 + 2] = v.z;
    q[4 * c4 + 3] = v.w;
  }

  // tile staging: the next tile's 16-byte chunks are loaded into registers
  // (gload) while the waves work on the current one, then converted to fp32
  // into LDS after the barrier, K row by row (lstore), V transposed
  // (lstore_v).  Rows past pos_hi are clamped to it.
  v4u pre[NCH];
  auto gload = [&](const uint16_t *src, int p0) {
#pragma unroll
    for (int j = 0; j < NCH; j++) {
      const int c = min(t + NT * j, TCH - 1), r = c / CPR, cc = c - r * CPR;
      pre[j] = *reinterpret_cast<const v4u *>(src + (size_t)min(p0 + r, pos_hi) * a.kv + 8 * cc);
    }
  };
  auto lstore = [&]() {
#pragma unroll
    for (int j = 0; j < NCH; j++) {
      const int c = t + NT * j;
      if (TCH % NT == 0 || c < TCH) {
        const int r = c / CPR, cc = c - r * CPR;
        const uint32_t hv[4] = {pre[j].x, pre[j].y, pre[j].z, pre[j].w};
        float f[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          f[2 * i] = h2f((uint16_t)(hv[i] & 0xffffu));
          f[2 * i + 1] = h2f((uint16_t)(hv[i] >> 16));
        }
        // the row's two halves in the opposite order for chunks 4-7: the 8
        // lanes of one row then write 8 distinct slots mod 8 per instruction
        // (16-byte accesses are served 8 lanes at a time)
        float *dst = tile + r * KP + 8 * cc;
        const bool sw = cc & 4;
        *reinterpret_cast<float4 *>(dst + (sw ? 4 : 0)) =
            sw ? make_float4(f[4], f[5], f[6], f[7]) : make_float4(f[0], f[1], f[2], f[3]);
        *reinterpret_cast<float4 *>(dst + (sw ? 0 : 4)) =
            sw ? make_float4(f[0], f[1], f[2], f[3]) : make_float4(f[4], f[5], f[6], f[7]);
      }
    }
  };
  auto lstore_v = [&]() {
#pragma unroll
    for (int j = 0; j < NCH; j++) {
      const int c = t + NT * j;
      if (TCH % NT == 0 || c < TCH) {
        const int r = c / CPR, cc = c - r * CPR;
        const uint32_t hv[4] = {pre[j].x, pre[j].y, pre[j].z, pre[j].w};
        // elements 8cc .. 8cc+7 share d >> 3: rows kPfTile + 4 floats apart
        float *dst = tile + pf_vrow(8 * cc) + r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          dst[(2 * i) * (kPfTile + 4)] = h2f((uint16_t)(hv[i] & 0xffffu));
          dst[(2 * i + 1) * (kPfTile + 4)] = h2f((uint16_t)(hv[i] >> 16));
        }
      }
    }
  };

  // ---- scores: lane = position, one sequential dot each ----
  float mx = -FLT_MAX;
  gload(Kc, lo0);
  for (int p0 = lo0; p0 <= pos_hi; p0 += kPfTile) {
    __syncthreads();  // the previous tile is consumed
    lstore();
    __syncthreads();
    // next K tile, or the first V tile after the last K tile
    if (p0 + kPfTile <= pos_hi) gload(Kc, p0 + kPfTile);
    else gload(Vc, lo0);
    const int p = p0 + lane;
    if (p >= lo && p <= pos) {
      const float *kr = tile + lane * KP;
      float s = 0.0f;
#pragma unroll
      for (int c = 0; c < HD / 4; c++) {
        const float4 k4 = *reinterpret_cast<const float4 *>(kr + 4 * c);
        const float kk[4] = {k4.x, k4.y, k4.z, k4.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float pr = q[4 * c + e] * kk[e];
          s = s + pr;
        }
      }
      const float si = (float)((double)s * a.inv_hd);
      sc[p - lo0] = si;
      mx = fmaxf(mx, si);
    }
  }

  // ---- softmax of the wave's token ----
  __syncthreads();
  {
    const float m = wave_max_dpp(mx);
    const int n = pos - lo + 1;
    float *sq = sc + (lo - lo0);
    // four of the lane's scores per step, k, k + 64, k + 128, k + 192 (the
    // lane's order of its part of the sum); past n a score of -inf adds
    // exp = 0 (reads clamped to the token's last slot)
    double sum = 0.0;
    for (int k = lane; k < n; k += 256) {
      float e[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const float v = sq[min(k + 64 * u, n - 1)];
        e[u] = k + 64 * u < n ? v - m : -__builtin_inff();
      }
#pragma unroll
      for (int u = 0; u < 4; u++) e[u] = ec_expf_tab(e[u], etab);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (k + 64 * u < n) sq[k + 64 * u] = e[u];
        sum += (double)e[u];
      }
    }
    sum = wave_sum_dpp(sum);
    const double isum = 1.0 / sum;
    for (int k = lane; k < n; k += 256) {
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) v[u] = sq[min(k + 64 * u, n - 1)];
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (k + 64 * u < n) sq[k + 64 * u] = (float)((double)v[u] * isum);
    }
  }

  // ---- output: lane = element d, the sum over positions in order ----
  float o[DPL];
#pragma unroll
  for (int j = 0; j < DPL; j++) o[j] = 0.0f;
  const int d0 = HD >= 64 ? lane : (lane & (HD - 1));
  // this lane's element of the tile's position p at vt[p - p0] (of element
  // d0 + 64 j at vt[p - p0 + VJ * j])
  const float *vt = tile + pf_vrow(d0);
  for (int p0 = lo0; p0 <= pos_hi; p0 += kPfTile) {
    __syncthreads();  // probabilities written / previous tile consumed
    lstore_v();
    __syncthreads();
    if (p0 + kPfTile <= pos_hi) gload(Vc, p0 + kPfTile);
    auto add1 = [&](int p) {
      const float pr = sc[p - lo0], *vr = vt + (p - p0);
#pragma unroll
      for (int j = 0; j < DPL; j++) {
        const float pv = pr * vr[VJ * j];
        o[j] = o[j] + pv;
      }
    };
    const int r0 = max(p0, lo), r1 = min(p0 + kPfTile - 1, pos);
    int p = r0;
    for (; p <= r1 && ((p - lo0) & 3); p++) add1(p);
    const int ng = p <= r1 ? (r1 - p + 1) >> 2 : 0;
    if (ng > 0) {
      // groups of 4 positions in two register sets (ping-pong): the
      // probabilities (one 16-byte read) and V elements of the next group are
      // read before the adds of the current one.  The look-ahead reads are
      // unconditional; past r1 they reach at most 4 positions further: the
      // tile's 4 spare rows, the next token's score slots or the 4 spare floats
      // after the last token's (values not used).
      float4 pa, pb;
      float va[4][DPL], vb[4][DPL];
      auto load4 = [&](int pp, float4 &pr, float (*vv)[DPL]) {
        pr = *reinterpret_cast<const float4 *>(sc + (pp - lo0));
        const float *vr = vt + (pp - p0);
#pragma unroll
        for (int j = 0; j < DPL; j++) {
          const float4 v4 = *reinterpret_cast<const float4 *>(vr + VJ * j);
          vv[0][j] = v4.x;
          vv[1][j] = v4.y;
          vv[2][j] = v4.z;
          vv[3][j] = v4.w;
        }
      };
      auto add4 = [&](const float4 &pr, float (*vv)[DPL]) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float pe = e == 0 ? pr.x : e == 1 ? pr.y : e == 2 ? pr.z : pr.w;
#pragma unroll
          for (int j = 0; j < DPL; j++) {
            const float pv = pe * vv[e][j];
            o[j] = o[j] + pv;
          }
        }
      };
      load4(p, pa, va);
      for (int g = 0;;) {
        load4(p + 4, pb, vb);
        __builtin_amdgcn_sched_barrier(0);
        add4(pa, va);
        __builtin_amdgcn_sched_barrier(0);
        p += 4;
        if (++g == ng) break;
        load4(p + 4, pa, va);
        __builtin_amdgcn_sched_barrier(0);
        add4(pb, vb);
        __builtin_amdgcn_sched_barrier(0);
        p += 4;
        if (++g == ng) break;
      }
    }
    for (; p <= r1; p++) add1(p);
  }
  if (act && (HD >= 64 || lane < HD)) {
    float *out = a.out + (size_t)mq * a.ldo + (size_t)h * HD + d0;
#pragma unroll
    for (int j = 0; j < DPL; j++) out[64 * j] = o[j];
  }
}

// ---------------------------------------------------------------------------
// Up to 4096 positions: the products on the matrix cores.
//
// v_mfma_f32_16x16x1_4b_f32 with a zero addend gives, per instruction, four
// 16 x 16 outer products whose elements are single rounded fp32 products (equal
// to v_mul_f32 bit for bit on 5 M random bit patterns, subnormals included), so
// such a product and a v_add_f32 keep the reference's order and rounding, and
// the instruction broadcasts its operands itself: no LDS broadcast reads, no
// DPP products.  What it does not do is run beside the adds (fp32 matrix
// instructions use the vector ALUs): 34 cycles for 1024 products, then 16 adds
// of 2.4 cycles, 4.4 cycles per product and add of 64 lanes with two or more
// waves per SIMD, against 6.4 for a DPP product and its add.  (The f16 forms do
// run beside the adds, but the sum of a factor's three 16-bit parts' products
// is not the rounded product: 19% of them off by a last bit.)
//
// One block takes 16 consecutive tokens of one query head, 8 waves.
//   - scores: tile t of 64 positions belongs to wave t % 8, which keeps its
//     16 x 64 scores in 16 registers per lane (up to NT tiles): scores never
//     reach LDS, so two blocks share a CU where 16 tokens' scores of 2048
//     positions (128 KB) left room for one.  NT 1 and 2 (spans to 1024) hold
//     them in registers; at NT 4, whose 64 are live beside 16 products twice
//     and a tile's K or V in 128, the compiler spills 105 (232 bytes of scratch
//     per lane; head_dim 128: 102 and 220), at NT 8 in 256 41 (104; 37 and 88).
//     B = the lane's position's k row,
//     A = four elements of the 16 tokens' q, one of them broadcast to the four
//     blocks per product.  Register 4 b + r of lane l: token 4 (l / 16) + r,
//     position 16 b + l % 16.
//   - softmax on those registers; maxima and double sums over the 16 lanes of
//     a DPP row, then over the waves.
//   - output: wave w < head_dim / 16 owns elements 16 w .. 16 w + 15 of the 16
//     tokens.  The probabilities of 8 tiles (written by their owners) are in
//     LDS in operand order, 64 floats per four positions, the values come
//     straight from the cache; the four blocks of a product are four
//     positions, whose products are added in order to the lane's four tokens.
// A masked product is replaced by -0 (x + -0 == x), so a value that is not
// finite outside a token's range does not reach it.
//
// 2048 tokens, 14 heads of 64: 363 us with the scores in LDS and DPP products,
// 251 (another card 266) here; 12 heads of 128: 667 and 317 us; 500 tokens, 14
// heads: 55 and 43 us.  The adds and products alone are about 125 us of that at
// 2.3 GHz, the exponentials 25 us; the rest is the output phase's one wave per
// SIMD and block (198 cycles per four positions where the SIMD could do 72) and
// the spilled scores' way to scratch and back, which that count includes.
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kMmTok = 16;  // tokens per block

template <int ABID>
__device__ __forceinline__ v16f mm_bcast(float a, float b) {  // block ABID of a to all four
  return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, v16f{0}, 2, ABID, 0);
}

// LDS accesses of the wave's other lanes before it come before those after it
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// the tile registers by a uniform index: a branch per tile (a move of 16
// registers in the taken one)
template <int NT>
__device__ __forceinline__ v16f mm_get(const v16f (&S)[NT], int k) {
  v16f v = S[0];
#pragma unroll
  for (int i = 1; i < NT; i++)
    if (k == i) {
      v = S[i];
      asm volatile("" : "+v"(v));
    }
  return v;
}
template <int NT>
__device__ __forceinline__ void mm_put(v16f (&S)[NT], int k, v16f v) {
#pragma unroll
  for (int i = 0; i < NT; i++)
    if (k == i) {
      S[i] = v;
      asm volatile("" : "+v"(S[i]));
    }
}

// LDS: q [HD][16] fp32, then per wave a K tile (up to 64 elements of 64 rows,
// fp16), later the probabilities of one of its tiles [64][16]
constexpr int kMmWaves = 8;
constexpr int kMmWaveLds = 8192;
static_assert(kPfTile * kMmTok * 4 <= kMmWaveLds, "a tile's probabilities");
template <int HD>
constexpr size_t mm_lds_bytes() {
  return (size_t)kMmTok * HD * 4 + kMmWaves * kMmWaveLds;
}

template <int HD, int NT>
__global__ __launch_bounds__(kMmWaves * 64, NT > 4 ? 2 : 4) void attn_prefill_mm_kernel(AttnArgs a, int ngroups) {
  constexpr int T = kMmTok, NW = kMmWaves, NTH = NW * 64;
  constexpr int DG = HD / 16;                       // groups of 16 output elements
  constexpr int KH = HD < 64 ? HD : 64;             // elements of a K row staged at a time
  constexpr int CPR = KH / 8, RPI = 64 / CPR;       // 16-byte chunks per staged row, rows per load instruction
  static_assert(NW >= DG, "a wave per 16 output elements");
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float *qt = lds;                                      // q as [HD][16]
  char *wbuf = reinterpret_cast<char *>(lds + T * HD);  // kMmWaveLds bytes per wave
  __shared__ uint64_t etab[32];
  __shared__ float s_max[NW][T];
  __shared__ double s_sum[NW][T];

  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, lq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int h = blockIdx.x, kvh = h * a.KVH / a.H;
  const int m0 = (ngroups - 1 - (int)blockIdx.y) * T;  // longest key ranges first
  const int slot = ld_uniform(a.slot + m0);
  const int pos_first = ld_uniform(a.pos + m0), pos_hi = ld_uniform(a.pos + min(m0 + T - 1, a.M - 1));
  const int lo0 = a.window > 0 ? max(0, pos_first - a.window + 1) : 0;
  const int lo_hi = a.window > 0 ? max(0, pos_hi - a.window + 1) : 0;
  const int ntile = (pos_hi - lo0) / kPfTile + 1;
  if (t < 32) etab[t] = ec_exp2_32[t];
  const size_t cbase = (size_t)slot * a.C * a.kv + (size_t)kvh * HD;
  const uint16_t *Kc = a.kc + cbase, *Vc = a.vc + cbase;

  for (int e = t; e < T * HD / 4; e += NTH) {
    const int r = e % T, c4 = e / T;
    const float4 v = *reinterpret_cast<const float4 *>(a.q + (size_t)min(m0 + r, a.M - 1) * a.ldq + (size_t)h * HD + 4 * c4);
    float *dst = qt + 4 * c4 * T + r;
    dst[0] = v.x;
    dst[T] = v.y;
    dst[2 * T] = v.z;
    dst[3 * T] = v.w;
  }
  __syncthreads();

  // whether every token takes every position of the tile that starts at p0
  auto whole = [&](int p0) { return p0 >= lo_hi && p0 + kPfTile - 1 <= pos_first; };
  // whether this lane's token r takes position p (tokens past the prompt, which
  // are not stored, take those of the last one)
  auto takes = [&](int p, int r) {
    const int tp = pos_first + min(4 * lq + r, pos_hi - pos_first);
    const int tl = a.window > 0 ? max(0, tp - a.window + 1) : 0;
    return (unsigned)(p - tl) <= (unsigned)(tp - tl);
  };

  // ---- scores ----
  v16f S[NT];
  float mx[4] = {-FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
  const int nk = w < ntile ? (ntile - 1 - w) / NW + 1 : 0;  // this wave's tiles
  // chunk c of row r of a staged tile is at chunk c ^ swz(r) of the row: 8
  // consecutive rows' 16-byte reads of one chunk fall on distinct banks
  auto swz = [](int r) { return CPR == 8 ? r & 7 : (r >> 1) & 3; };
  const int krow = lane / CPR, kchk = lane % CPR;
  const char *kld = wbuf + w * kMmWaveLds + lane * (2 * KH);
  const int ksw = 16 * swz(lane);
#pragma unroll 1
  for (int k = 0; k < nk; k++) {
    const int tile = k * NW + w, p0 = lo0 + kPfTile * tile;
    v16f acc = {0};
#pragma unroll 1
    for (int e0 = 0; e0 < HD; e0 += KH) {
      // the tile's rows, whole 128-byte lines per instruction, through this
      // wave's part of the LDS: a lane reads its position's row, which other
      // lanes wrote (no block barrier: one wave's LDS operations are in order;
      // wave_order keeps the compiler from moving them)
      wave_order();  // the previous rows are read
      {
        v4u kr[CPR];
#pragma unroll
        for (int i = 0; i < CPR; i++) {
          const int p = min(p0 + RPI * i + krow, pos_hi);
          kr[i] = *reinterpret_cast<const v4u *>(Kc + (size_t)p * a.kv + e0 + 8 * kchk);
        }
#pragma unroll
        for (int i = 0; i < CPR; i++) {
          const int r = RPI * i + krow;
          *reinterpret_cast<v4u *>(wbuf + w * kMmWaveLds + r * (2 * KH) + 16 * (kchk ^ swz(r))) = kr[i];
        }
      }
      wave_order();
      const float *qa = qt + e0 * T + lane;
      v4u kc = *reinterpret_cast<const v4u *>(kld + (0 ^ ksw));
      float aq = qa[0];
#pragma unroll
      for (int c = 0; c < CPR; c++) {
        const v4u kn = *reinterpret_cast<const v4u *>(kld + ((16 * (c + 1 < CPR ? c + 1 : c)) ^ ksw));
        const float a1 = qa[(2 * c + 1) * 64], a2 = qa[(2 * (c + 1 < CPR ? c + 1 : c)) * 64];
        const uint32_t hv[4] = {kc.x, kc.y, kc.z, kc.w};
        // the asm statements keep the compiler from forming all products first
#define MM_STEP(e, av, ab)                                                                             \
  {                                                                                                    \
    uint32_t hw = hv[(e) / 2];                                                                         \
    asm volatile("" : "+v"(acc), "+v"(hw));                                                            \
    acc += mm_bcast<ab>(av, h2f((uint16_t)((e) & 1 ? hw >> 16 : hw & 0xffffu)));                       \
  }
        MM_STEP(0, aq, 0)
        MM_STEP(1, aq, 1)
        MM_STEP(2, aq, 2)
        MM_STEP(3, aq, 3)
        MM_STEP(4, a1, 0)
        MM_STEP(5, a1, 1)
        MM_STEP(6, a1, 2)
        MM_STEP(7, a1, 3)
#undef MM_STEP
        aq = a2;
        kc = kn;
      }
    }
    const bool wh = whole(p0);
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float s = (float)((double)acc[4 * b + r] * a.inv_hd);
        if (wh || takes(p0 + 16 * b + lr, r)) mx[r] = fmaxf(mx[r], s);
        else s = -__builtin_inff();
        acc[4 * b + r] = s;
      }
    mm_put<NT>(S, k, acc);
  }

  // ---- softmax: maximum, exponentials and their sum ----
#pragma unroll
  for (int r = 0; r < 4; r++) {
    float v = mx[r];
    v = fmaxf(v, dpp_mov<0xB1>(v));
    v = fmaxf(v, dpp_mov<0x4E>(v));
    v = fmaxf(v, dpp_mov<0x141>(v));
    v = fmaxf(v, dpp_mov<0x140>(v));
    if (lr == 0) s_max[w][4 * lq + r] = v;
  }
  __syncthreads();
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int r = 0; r < 4; r++) {
    mx[r] = s_max[0][4 * lq + r];
#pragma unroll
    for (int i = 1; i < NW; i++) mx[r] = fmaxf(mx[r], s_max[i][4 * lq + r]);
  }
#pragma unroll 1
  for (int k = 0; k < nk; k++) {
    v16f v = mm_get<NT>(S, k);
    const int p0 = lo0 + kPfTile * (k * NW + w);
    const bool wh = whole(p0);
#pragma unroll
    for (int b = 0; b < 4; b++) {
      // four exponentials at a time (more exceed the registers): the table
      // reads of all four in flight together
      double er[4];
      uint64_t ki[4], et[4];
      float x[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        x[r] = v[4 * b + r] - mx[r];
        ki[r] = ec_expf_head(x[r], &er[r]);
        et[r] = etab[ki[r] % 32];
      }
      asm volatile("" : "+v"(v), "+v"(et[0]), "+v"(et[1]), "+v"(et[2]), "+v"(et[3]));
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float e = ec_expf_tail(x[r], er[r], ki[r], et[r]);
        if (!wh && !takes(p0 + 16 * b + lr, r)) e = 0.0f;
        v[4 * b + r] = e;
        sum[r] += (double)e;
      }
    }
    mm_put<NT>(S, k, v);
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    double v = sum[r];
    v = v + dpp_mov<0xB1>(v);
    v = v + dpp_mov<0x4E>(v);
    v = v + dpp_mov<0x141>(v);
    v = v + dpp_mov<0x140>(v);
    if (lr == 0) s_sum[w][4 * lq + r] = v;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; r++) {
    double v = s_sum[0][4 * lq + r];
#pragma unroll
    for (int i = 1; i < NW; i++) v += s_sum[i][4 * lq + r];
    sum[r] = 1.0 / v;
  }

  // ---- output ----
  // this lane's element of position p0 + 4 s + lane / 16, from the cache (two
  // bytes per lane, 32 of a row: the waves' loads of a row share its line);
  // rows past pos_hi read as zero (their products are masked)
  v4f o = {0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int NS = kPfTile / 8;  // steps of four positions per half tile
  uint16_t vr[NS], vn[NS];
  const uint64_t vbase = (uint64_t)(uintptr_t)(Vc + (size_t)lo0 * a.kv);
  const uint32_t vlo = __builtin_amdgcn_readfirstlane((uint32_t)vbase),
                 vhi = __builtin_amdgcn_readfirstlane((uint32_t)(vbase >> 32));
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(uintptr_t)(((uint64_t)vhi << 32) | vlo), 0, ((pos_hi - lo0) * a.kv + HD) * 2, 0x00020000);
  int voff = 2 * (lq * a.kv + 16 * (w < DG ? w : 0) + lr);  // the whole offset: the range check covers it
  auto vload = [&]() {
#pragma unroll
    for (int s = 0; s < NS; s++) {
      vn[s] = __builtin_amdgcn_raw_buffer_load_b16(vrs, voff, 0, 0);
      voff += 8 * a.kv;
    }
  };
  vload();
#pragma unroll 1
  for (int t0 = 0; t0 < ntile; t0 += NW) {
    __syncthreads();  // the previous NW tiles' probabilities are consumed
    if (t0 + w < ntile) {
      const v16f v = mm_get<NT>(S, t0 / NW);
      float *dst = reinterpret_cast<float *>(wbuf + w * kMmWaveLds) + lr * T + 4 * lq;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        float4 p;
        p.x = (float)((double)v[4 * b] * sum[0]);
        p.y = (float)((double)v[4 * b + 1] * sum[1]);
        p.z = (float)((double)v[4 * b + 2] * sum[2]);
        p.w = (float)((double)v[4 * b + 3] * sum[3]);
        *reinterpret_cast<float4 *>(dst + 16 * b * T) = p;
      }
    }
    __syncthreads();
    if (w >= DG) continue;
#pragma unroll 1
    for (int half = 0; half < 2 * min(NW, ntile - t0); half++) {
      const int p0 = lo0 + kPfTile * t0 + kPfTile / 2 * half;
      const float *pa = reinterpret_cast<const float *>(wbuf + (half >> 1) * kMmWaveLds) + (half & 1) * (64 * NS) + lane;
      // the next half tile's values are loaded while this one's are used
#pragma unroll
      for (int s = 0; s < NS; s++) vr[s] = vn[s];
      vload();
      // a step's probabilities are read four steps ahead, its products formed one ahead
      auto sums = [&](auto masked) {
        float fa[NS];
#pragma unroll
        for (int s = 0; s < 4; s++) fa[s] = pa[64 * s];
        v16f pn = __builtin_amdgcn_mfma_f32_16x16x1f32(fa[0], h2f(vr[0]), v16f{0}, 0, 0, 0);
#pragma unroll
        for (int s = 0; s < NS; s++) {
          v16f pc = pn;
          if (s + 4 < NS) fa[s + 4] = pa[64 * (s + 4)];
          if (s + 1 < NS) {
            asm volatile("" : "+v"(o), "+v"(fa[s + 1]));
            pn = __builtin_amdgcn_mfma_f32_16x16x1f32(fa[s + 1], h2f(vr[s + 1]), v16f{0}, 0, 0, 0);
          }
          if constexpr (masked.value) {
#pragma unroll
            for (int b = 0; b < 4; b++)
#pragma unroll
              for (int r = 0; r < 4; r++)
                if (!takes(p0 + 4 * s + b, r)) pc[4 * b + r] = -0.0f;
          }
#pragma unroll
          for (int b = 0; b < 4; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) o[r] = o[r] + pc[4 * b + r];
        }
      };
      if (p0 >= lo_hi && p0 + kPfTile / 2 - 1 <= pos_first) sums(std::false_type{});
      else if (p0 <= pos_hi) sums(std::true_type{});
    }
  }
  if (w < DG) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = m0 + 4 * lq + r;
      if (m < a.M) a.out[(size_t)m * a.ldo + (size_t)h * HD + 16 * w + lr] = o[r];
    }
  }
}

// positions that a block of qb consecutive tokens reads (any window up to
// INT_MAX: no sum with it before the comparison)
int pf_span(const AttnArgs &a, int qb) {
  return a.window > 0 && a.window < a.max_npos - (qb - 1) ? a.window + qb - 1 : a.max_npos;
}
int mm_span(const AttnArgs &a) { return pf_span(a, kMmTok); }
// the most positions whose scores the kernel's registers hold
constexpr int kMmMaxSpan = 8 * kMmWaves * kPfTile;

template <int HD, int NT>
void launch_mm(const AttnArgs &a, hipStream_t st) {
  const int ngroups = (a.M + kMmTok - 1) / kMmTok;
  klaunch((attn_prefill_mm_kernel<HD, NT>), dim3(a.H, ngroups), dim3(kMmWaves * 64), mm_lds_bytes<HD>(), st, a, ngroups);
}

// by the longest span: the fewest score registers that hold it (up to 2048
// positions two blocks share a CU, beyond that one).  The two-tile form spills
// none at head_dim 32 and 64 (16 registers at 128), the four-tile one 105 (102):
// 1024 tokens, us, with two and with four tiles: 16 heads of 32 72 and 95 (86
// with the scores in LDS), 14 heads of 64 83 and 96, 12 of 128 107 and 114.  A
// three-tile form spilled 214 and was slower than the four-tile one (1400
// tokens, 14 heads of 64: 159 and 145).
template <int HD>
void launch_mm_any(const AttnArgs &a, hipStream_t st) {
  const int n = mm_span(a);
  if (n <= kMmWaves * kPfTile) launch_mm<HD, 1>(a, st);
  else if (n <= 2 * kMmWaves * kPfTile) launch_mm<HD, 2>(a, st);
  else if (n <= 4 * kMmWaves * kPfTile) launch_mm<HD, 4>(a, st);
  else launch_mm<HD, 8>(a, st);
}

// score slots per token: the positions one block reads, window-bounded
int pf_nsc(const AttnArgs &a, int qb) { return (pf_span(a, qb) + 3) & ~3; }

// tile with 4 spare rows, the score slots of qb tokens and 4 spare floats,
// plus the static expf table (256 bytes)
size_t pf_lds_bytes(const AttnArgs &a, int qb) {
  return ((size_t)(kPfTile + 4) * (a.hd + 4) + (size_t)qb * pf_nsc(a, qb) + 4) * sizeof(float) + 256;
}

// waves (of one token) per block, largest first
constexpr int kPfShapes[2] = {8, 4};

int pf_pick(const AttnArgs &a, int max_lds) {
  for (int i = 0; i < 2; i++)
    if (pf_lds_bytes(a, kPfShapes[i]) <= (size_t)max_lds) return i;
  return -1;
}

// the 8-token blocks that the other kernel makes of a prompt
long pf_blocks8(const AttnArgs &a) { return (long)a.H * ((a.M + 7) / 8); }

// Whether the matrix-core kernel takes a prompt: its scores fit the registers,
// and the other kernel's blocks, twice as many and each with half the tokens,
// would be more than one per CU.  There and here, us: 14 heads of 64, 144 tokens
// (252 of its blocks) 24.7 and 29.2 after none, 54.8 and 71.2 after 1000, 131
// and 151 after 3500; 152 tokens (266) 25.0 and 29.5, 69.0 and 71.4, 237 and
// 152; 16 heads of 32, 128 tokens (256) after 3500 118 and 133, 136 (272) 212
// and 133.  At head_dim 128 from 192 of its own blocks: 12 heads, 128 tokens
// (96) 30.2 and 34.2, 256 tokens (192) 38.5 and 38.1; 64 tokens after 1500 (48)
// 99.6 and 111.5.
constexpr int kCus = 256;
bool mm_takes(const AttnArgs &a, int max_lds) {
  if (mm_span(a) > kMmMaxSpan) return false;
  if (a.hd == 128) return (long)a.H * ((a.M + kMmTok - 1) / kMmTok) >= 192;
  return pf_pick(a, max_lds) != 0 || pf_blocks8(a) > kCus;
}

// grid (head, token group): consecutive block ids, which the dispatcher deals
// out to the 8 XCDs in turn, spread every head over every XCD; one slot's K/V
// of all KV heads fits each XCD's L2 at the prefill lengths of the models
template <int HD, int NW>
void launch_pf(const AttnArgs &a, hipStream_t st) {
  const int ngroups = (a.M + NW - 1) / NW;
  const dim3 grid(a.H, ngroups);
  klaunch((attn_prefill_kernel<HD, NW>), grid, dim3(NW * 64), pf_lds_bytes(a, NW) - 256, st, a, ngroups,
          pf_nsc(a, NW));
}

template <int HD>
void launch_hd(const AttnArgs &a, int shape, hipStream_t st) {
  if (shape == 0) launch_pf<HD, 8>(a, st);
  else launch_pf<HD, 4>(a, st);
}

}  // namespace

bool attention_prefill_ok(const AttnArgs &a, int max_lds) {
  if (!(a.hd == 32 || a.hd == 64 || a.hd == 128) || !attn_vec(a.hd, a.kv) || a.fuse_kv || a.M < 1) return false;
  if (a.ldq % 4 || ((uintptr_t)a.q & 15u)) return false;  // q rows read as float4
  return mm_takes(a, max_lds) || pf_pick(a, max_lds) >= 0;
}

hipError_t attention_prefill(const AttnArgs &a, int max_lds, hipStream_t st) {
  if (!attention_prefill_ok(a, max_lds)) return hipErrorInvalidValue;
  if (mm_takes(a, max_lds)) {
    if (a.hd == 64) launch_mm_any<64>(a, st);
    else if (a.hd == 128) launch_mm_any<128>(a, st);
    else launch_mm_any<32>(a, st);
    return hipGetLastError();
  }
  const int shape = pf_pick(a, max_lds);
  if (a.hd == 64) launch_hd<64>(a, shape, st);
  else if (a.hd == 128) launch_hd<128>(a, shape, st);
  else launch_hd<32>(a, shape, st);
  return hipGetLastError();
}

}  // namespace ec
