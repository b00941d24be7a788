// Selection of each pattern vertex's k most likely data vertices (ac_get_topk, ac_get_match) on the device.
//
// The order is the value, largest first, and the lower vertex on ties: one 64-bit key per entry, unique within a column.
//   k_sel_chunks: the largest value of each of S row chunks, per column (one coalesced read of MU);
//   k_sel_thresh: the k-th largest of a column's S chunk maxima.  The k chunks at or above it each hold an entry at
//                 least as large, so it bounds the column's k-th largest entry from below;
//   k_sel_filter: the keys of the entries at or above the bound (a second read of MU, k and a few more entries);
//   k_sel_rank:   the rank of each kept key among the others, and the first k written out in order.
// Bound by the two reads of MU and by four launches: k = 10 of 262,144 x 12 takes 25 us; selecting on the host took
// the copy of MU over PCIe and about 1 ns per entry, 3.6 ms there.
// A NaN has no place in that order, and a column may hold more ties than fit: both set a flag, and the caller then
// selects on the host.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "ac_select.hpp"

namespace ac {

namespace {

// Floats to unsigned, order-preserving (no NaN; -0.0 counts as +0.0).
__device__ __forceinline__ unsigned order_bits(float x) {
  const unsigned b = __float_as_uint(x + 0.f);
  return b & 0x80000000u ? ~b : b | 0x80000000u;
}

}  // namespace

__global__ __launch_bounds__(256) void k_sel_chunks(int64_t n, int P, int64_t rows, const float* __restrict__ X,
                                                    unsigned* __restrict__ cmax, int* __restrict__ flag,
                                                    int* __restrict__ count) {
  __shared__ unsigned red[256];
  __shared__ int nan;
  const int t = threadIdx.x, RP = 256 / P;
  if (t == 0) nan = 0;
  if (blockIdx.x == 0 && t < P) count[t] = 0;  // for k_sel_filter
  __syncthreads();
  const bool active = t < RP * P;
  const int p = active ? t % P : 0;
  const int64_t v0 = blockIdx.x * rows, v1 = std::min(n, v0 + rows);
  unsigned m = 0u;
  bool bad = false;
  if (active) {
    int64_t v = v0 + t / P;
    for (; v + 3 * RP < v1; v += 4 * RP) {
      const float a = X[v * P + p], b = X[(v + RP) * P + p], c = X[(v + 2 * RP) * P + p], d = X[(v + 3 * RP) * P + p];
      bad |= a != a || b != b || c != c || d != d;
      m = max(max(m, max(order_bits(a), order_bits(b))), max(order_bits(c), order_bits(d)));
    }
    for (; v < v1; v += RP) {
      const float a = X[v * P + p];
      bad |= a != a;
      m = max(m, order_bits(a));
    }
  }
  if (bad) nan = 1;
  red[t] = m;
  __syncthreads();
  if (t < P) {
    for (int r = 1; r < RP; ++r) m = max(m, red[r * P + t]);
    cmax[(int64_t)t * gridDim.x + blockIdx.x] = m;
  }
  if (t == 0 && nan) *flag = 1;
}

// One block per column: the k-th largest of S <= kSelChunks chunk maxima, bit by bit from the top (the largest T that k
// of them reach).  Ranking every one against all others took 153 us for 2,048 of them.
__global__ __launch_bounds__(256) void k_sel_thresh(int S, int k, const unsigned* __restrict__ cmax,
                                                    unsigned* __restrict__ thr) {
  __shared__ int part[2][4];
  const unsigned* c = cmax + (int64_t)blockIdx.x * S;
  unsigned x[kSelChunks / 256];
#pragma unroll
  for (int u = 0; u < kSelChunks / 256; ++u) {
    const int i = threadIdx.x + u * 256;
    x[u] = i < S ? c[i] : 0u;  // below every value
  }
  unsigned T = 0u;
  for (int bit = 31; bit >= 0; --bit) {
    const unsigned cand = T | (1u << bit);
    int m = 0;
#pragma unroll
    for (int u = 0; u < kSelChunks / 256; ++u) m += __popcll(__ballot(x[u] >= cand));
    int* p = part[bit & 1];  // two sets in turn: one barrier per bit
    if ((threadIdx.x & 63) == 0) p[threadIdx.x >> 6] = m;
    __syncthreads();
    if (p[0] + p[1] + p[2] + p[3] >= k) T = cand;
  }
  if (threadIdx.x == 0) thr[blockIdx.x] = T;
}

// A block counts its entries in LDS and reserves their places with one atomic per column: where most of a column ties
// (and the host selects after all), one per entry made 3.6 M of them follow each other on twelve counters (4.7 ms).
__global__ __launch_bounds__(256) void k_sel_filter(int64_t n, int P, const float* __restrict__ X,
                                                    const unsigned* __restrict__ thr, int* __restrict__ count,
                                                    unsigned long long* __restrict__ keys, int* __restrict__ flag) {
  constexpr int kRows = 8;  // a thread's, between barriers
  __shared__ int own[256], base[256];
  const int t = threadIdx.x, RP = 256 / P;
  const bool active = t < RP * P;
  const int p = active ? t % P : 0;
  const unsigned lo = thr[p];
  own[t] = 0;
  const int64_t step = (int64_t)gridDim.x * RP;
  for (int64_t v0 = (int64_t)blockIdx.x * RP; v0 < n; v0 += kRows * step) {
    unsigned b[kRows];
    int hits = 0;
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const int64_t v = v0 + u * step + t / P;
      const float x = X[(v < n ? v : n - 1) * P + p];
      b[u] = active && v < n ? order_bits(x) : 0u;  // below every value
      hits += b[u] >= lo && b[u] != 0u;
    }
    if (!__syncthreads_or(hits)) continue;
    int at = hits ? atomicAdd(own + p, hits) : 0;
    __syncthreads();
    if (t < P && own[t] > 0) {
      base[t] = atomicAdd(count + t, own[t]);
      if (base[t] + own[t] > kSelCap) *flag = 1;
      own[t] = 0;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kRows; ++u)
      if (b[u] >= lo && b[u] != 0u) {
        const int i = base[p] + at++;
        if (i < kSelCap)
          keys[(int64_t)p * kSelCap + i] =
              ((unsigned long long)b[u] << 32) | (0xFFFFFFFFu - (unsigned)(v0 + u * step + t / P));
      }
  }
}

__global__ __launch_bounds__(256) void k_sel_rank(int P, int k, const float* __restrict__ X,
                                                  const int* __restrict__ count,
                                                  const unsigned long long* __restrict__ keys,
                                                  const int* __restrict__ flag, int* __restrict__ idx,
                                                  float* __restrict__ val) {
  __shared__ unsigned long long x[kSelCap];
  if (*flag) return;  // (1.1 ms for a full column)
  const int p = blockIdx.x, m = min(count[p], kSelCap);
  for (int i = threadIdx.x; i < m; i += 256) x[i] = keys[(int64_t)p * kSelCap + i];
  __syncthreads();
  for (int i = threadIdx.x; i < m; i += 256) {
    const unsigned long long xi = x[i];
    int r = 0;
#pragma unroll 4
    for (int j = 0; j < m; ++j) r += x[j] > xi;
    if (r < k) {
      const int v = (int)(0xFFFFFFFFu - (unsigned)xi);
      idx[(int64_t)p * k + r] = v;
      val[(int64_t)p * k + r] = X[(int64_t)v * P + p];
    }
  }
}

SelShape sel_shape(int64_t n, int P, int k) {
  SelShape s;
  // Below 65,536 entries copying MU and selecting on the host (about 1 ns an entry) takes no longer than four launches.
  if (n * P < 65536 || P > 256 || k > kSelMaxK) return s;
  s.rows = (n + kSelChunks - 1) / kSelChunks;
  const int64_t chunks = (n + s.rows - 1) / s.rows;
  if (chunks < 2 * (int64_t)k) return s;  // the bound needs chunks to spare
  s.chunks = (int)chunks;
  return s;
}

void launch_select(int64_t n, int P, int k, const SelShape& s, const float* X, const SelBufs& b, hipStream_t st) {
  hipLaunchKernelGGL(k_sel_chunks, dim3(s.chunks), dim3(256), 0, st, n, P, s.rows, X, b.cmax, b.flag, b.count);
  hipLaunchKernelGGL(k_sel_thresh, dim3(P), dim3(256), 0, st, s.chunks, k, b.cmax, b.thr);
  const int RP = 256 / P;
  const int blocks = (int)std::max<int64_t>(1, std::min<int64_t>((n + 4 * RP - 1) / (4 * RP), 2048));
  hipLaunchKernelGGL(k_sel_filter, dim3(blocks), dim3(256), 0, st, n, P, X, b.thr, b.count, b.keys, b.flag);
  hipLaunchKernelGGL(k_sel_rank, dim3(P), dim3(256), 0, st, P, k, X, b.count, b.keys, b.flag, b.idx, b.val);
}

}  // namespace ac
