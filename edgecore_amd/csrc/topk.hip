// Device top-k of logit rows for sampled decoding (the selection of
// sample_token, src/runtime_main.c:220-226, and what it reads): per row the
// top_k + 1 largest logits, value descending and index ascending among equal
// values, plus a status that tells whether they determine sample_token's
// choice (no NaN in the row, and the top_k-th and (top_k+1)-th values differ).
//
// Keys: an order-preserving 32-bit image of the float (sign bit flipped for
// positives, all bits for negatives) above the inverted index, so that one
// 64-bit comparison orders by value and then by smaller index.  -0 and +0
// get different keys; the status compares the boundary values as floats, so
// a -0/+0 pair at the boundary counts as a tie.
//
// Both launches select, they do not sort: a threshold that at least n = top_k +
// 1 keys reach (threshold_of, from one maximum per thread: every thread whose
// maximum reaches it holds a key that does), the keys that reach it into an LDS
// list, and each key's rank in that list by comparing it with the others, which
// is its place in the output.  The list holds a few more than n keys unless
// many are equal or one thread's share holds most of the largest; past
// kListCap keys the block sorts instead (sort_desc).
//
//   topk_chunk_kernel: a block of 512 threads takes a chunk of 4096 logits, its
//     top n keys and a NaN flag;
//   topk_merge_kernel: one block of 1024 threads per row takes the chunks'
//     candidates (at most 16384 keys), writes the row's top n and status.
//
// Bound by latency: the passes are a load, one wave's threshold search and the
// ranks.  16 rows of 151936, top 40: the chunks 145 us when every one was
// sorted (78 LDS passes and barriers), 7.5 now; the merge 32.6 -> 7.2 (both
// sort still, and cost what they did, where a row is one value).
#include "ec_device.h"
#include "ec_kernels.h"

namespace ec {

namespace {

constexpr int kChunk = 4096;
constexpr int kMergeMax = 16384;  // candidates of a row, at most (topk_ok)

__device__ __forceinline__ uint32_t fkey(float v) {
  const uint32_t u = __float_as_uint(v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float fkey_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);
}

// bitonic sort of S (a power of two) keys in LDS into descending order
template <int NT>
__device__ void sort_desc(unsigned long long *s, int S) {
  for (int k = 2; k <= S; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < S; i += NT) {
        const int l = i ^ j;
        if (l > i) {
          const unsigned long long a = s[i], b = s[l];
          const bool down = (i & k) == 0;  // this run descending
          if (down ? a < b : a > b) {
            s[i] = b;
            s[l] = a;
          }
        }
      }
      __syncthreads();
    }
  }
}

constexpr int kListCap = 512;

// A threshold that at least n of the NT per-thread maxima mx reach (0 when
// fewer than n are above it), built from the top bit down by one wave (NT / 64
// maxima per lane) and ended as soon as at most kSlack more than n reach it.
// Every thread of the block calls it; ends with a barrier.
constexpr int kSlack = 32;
template <int NT>
__device__ __forceinline__ uint32_t threshold_of(uint32_t mx, int n, uint32_t *s_mx, uint32_t *s_thr) {
  constexpr int PL = NT / 64;
  const int t = threadIdx.x;
  s_mx[t] = mx;
  __syncthreads();
  if (t < 64) {
    uint32_t v[PL];
#pragma unroll
    for (int j = 0; j < PL; j++) v[j] = s_mx[t + 64 * j];
    uint32_t thr = 0;
    for (int b = 31; b >= 0; b--) {
      const uint32_t c = thr | (1u << b);
      int cnt = 0;
#pragma unroll
      for (int j = 0; j < PL; j++) cnt += __popcll(__ballot(v[j] >= c));
      if (cnt >= n) {
        thr = c;
        if (cnt <= n + kSlack) break;
      }
    }
    if (t == 0) *s_thr = thr;
  }
  __syncthreads();
  return *s_thr;
}

// the number of the list's c keys above key (the list in LDS, read by every
// thread at the same place)
__device__ __forceinline__ int rank_of(unsigned long long key, const unsigned long long *list, int c) {
  int r = 0;
#pragma unroll 8
  for (int u = 0; u < c; u++) r += list[u] > key;
  return r;
}

__global__ __launch_bounds__(512) void topk_chunk_kernel(const float *L, int ld, int V, int n,
                                                         unsigned long long *cand, unsigned char *nan_flag) {
  constexpr int PT = kChunk / 512;  // logits per thread
  __shared__ unsigned long long s[kChunk];  // the list, or every key when the block sorts
  __shared__ uint32_t s_mx[512], s_thr;
  __shared__ int has_nan, count;
  const int row = blockIdx.y, c0 = blockIdx.x * kChunk, t = threadIdx.x;
  const float *l = L + (size_t)row * ld;
  if (t == 0) has_nan = count = 0;
  float x[PT];
#pragma unroll
  for (int j = 0; j < PT; j++) x[j] = l[min(c0 + t + 512 * j, V - 1)];
  uint32_t key[PT], mx = 0;
  bool nan_here = false;
#pragma unroll
  for (int j = 0; j < PT; j++) {
    const bool in = c0 + t + 512 * j < V;
    nan_here |= in && x[j] != x[j];
    key[j] = in ? fkey(x[j]) : 0u;
    mx = max(mx, key[j]);
  }
  const uint32_t thr = threshold_of<512>(mx, n, s_mx, &s_thr);
  if (nan_here) has_nan = 1;
  // 64-bit keys, 0 (below every key of a number) past the row
  auto key64 = [&](int j) -> unsigned long long {
    const int v = c0 + t + 512 * j;
    return v < V ? ((unsigned long long)key[j] << 32) | (0xFFFFFFFFu - (uint32_t)v) : 0ull;
  };
#pragma unroll
  for (int j = 0; j < PT; j++) {
    if (key[j] >= thr && c0 + t + 512 * j < V) {
      const int p = atomicAdd(&count, 1);
      if (p < kListCap) s[p] = key64(j);
    }
  }
  __syncthreads();
  const int c = count;
  unsigned long long *out = cand + ((size_t)row * gridDim.x + blockIdx.x) * n;
  if (c <= kListCap) {
    if (t < c) {
      const unsigned long long k = s[t];
      const int r = rank_of(k, s, c);
      if (r < n) out[r] = k;
    }
    if (t >= c && t < n) out[t] = 0ull;  // a last chunk of fewer than n logits
  } else {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PT; j++) s[t + 512 * j] = key64(j);
    __syncthreads();
    sort_desc<512>(s, kChunk);
    for (int i = t; i < n; i += 512) out[i] = s[i];
  }
  if (t == 0) nan_flag[(size_t)row * gridDim.x + blockIdx.x] = (unsigned char)has_nan;
}

// PT: candidates per thread
template <int PT>
__global__ __launch_bounds__(1024) void topk_merge_kernel(const unsigned long long *cand,
                                                          const unsigned char *nan_flag, int nb, int n,
                                                          int top_k, int S, float *vals, int *idx,
                                                          int *status) {
  extern __shared__ unsigned long long s[];  // S keys: every candidate when the block sorts
  __shared__ unsigned long long list[kListCap], top[kTopkMax + 1];
  __shared__ uint32_t s_mx[1024], s_thr;
  __shared__ int has_nan, count;
  const int row = blockIdx.x, tot = nb * n, t = threadIdx.x;
  const unsigned long long *cd = cand + (size_t)row * tot;
  if (t == 0) has_nan = count = 0;
  unsigned long long key[PT];
  uint32_t mx = 0;
#pragma unroll
  for (int j = 0; j < PT; j++) {
    const int i = t + 1024 * j;
    key[j] = cd[min(i, tot - 1)];
    if (i >= tot) key[j] = 0ull;
  }
#pragma unroll
  for (int j = 0; j < PT; j++) {
    mx = max(mx, (uint32_t)(key[j] >> 32));
  }
  const uint32_t thr = threshold_of<1024>(mx, n, s_mx, &s_thr);
  for (int b = t; b < nb; b += 1024)
    if (nan_flag[(size_t)row * nb + b]) has_nan = 1;
#pragma unroll
  for (int j = 0; j < PT; j++) {
    if (key[j] && (uint32_t)(key[j] >> 32) >= thr) {
      const int p = atomicAdd(&count, 1);
      if (p < kListCap) list[p] = key[j];
    }
  }
  __syncthreads();
  const int c = count;
  if (c <= kListCap) {
    if (t < c) {
      const unsigned long long k = list[t];
      const int r = rank_of(k, list, c);
      if (r < n) top[r] = k;
    }
    __syncthreads();
  } else {
#pragma unroll
    for (int j = 0; j < PT; j++)
      if (t + 1024 * j < S) s[t + 1024 * j] = key[j];
    __syncthreads();
    sort_desc<1024>(s, S);
    if (t < n) top[t] = s[t];
    __syncthreads();
  }
  if (t < n) {
    vals[(size_t)row * n + t] = fkey_value((uint32_t)(top[t] >> 32));
    idx[(size_t)row * n + t] = (int)(0xFFFFFFFFu - (uint32_t)top[t]);
  }
  if (t == 0) {
    const float a = fkey_value((uint32_t)(top[top_k - 1] >> 32)), b = fkey_value((uint32_t)(top[top_k] >> 32));
    status[row] = (has_nan || a == b) ? 1 : 0;
  }
}

int merge_size(int nb, int n) {
  int S = 1;
  while (S < nb * n) S <<= 1;
  return S;
}

}  // namespace

int topk_chunks(int V) { return (V + kChunk - 1) / kChunk; }

bool topk_ok(int V, int top_k) {
  return top_k > 0 && top_k < V && top_k <= kTopkMax && merge_size(topk_chunks(V), top_k + 1) <= kMergeMax;
}

hipError_t topk_select(const float *L, int rows, int V, int ld, int top_k, unsigned long long *cand,
                       unsigned char *nan_flag, hipStream_t st) {
  if (!topk_ok(V, top_k) || rows < 1) return hipErrorInvalidValue;
  klaunch(topk_chunk_kernel, dim3(topk_chunks(V), rows), dim3(512), 0, st, L, ld, V, top_k + 1, cand, nan_flag);
  return hipGetLastError();
}

hipError_t topk_merge(const unsigned long long *cand, const unsigned char *nan_flag, int rows, int V, int top_k,
                      float *vals, int *idx, int *status, hipStream_t st) {
  if (!topk_ok(V, top_k) || rows < 1) return hipErrorInvalidValue;
  const int nb = topk_chunks(V), n = top_k + 1, S = merge_size(nb, n), pt = (nb * n + 1023) / 1024;
  const uint32_t lds = (uint32_t)(S * sizeof(unsigned long long));
  auto go = [&](auto kernel) {
    klaunch(kernel, dim3(rows), dim3(1024), lds, st, cand, nan_flag, nb, n, top_k, S, vals, idx, status);
  };
  if (pt <= 1) go(topk_merge_kernel<1>);
  else if (pt <= 2) go(topk_merge_kernel<2>);
  else if (pt <= 4) go(topk_merge_kernel<4>);
  else if (pt <= 8) go(topk_merge_kernel<8>);
  else go(topk_merge_kernel<kMergeMax / 1024>);
  return hipGetLastError();
}

}  // namespace ec
