// The reference's operator library (src/ac.hxx) as stand-alone stage operators on caller-owned device buffers,
// FP32 values and int32 ids, same argument meaning and pattern-major layouts.  They are not used by the fused
// matcher; they exist so each reference operator can be dropped in (and checked) on its own.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>

#include "../../include/ac_mi355x.h"
#include "ac_host.hpp"
#include "ac_lse.hpp"

namespace {

hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

int launch_status(const char* who) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    ac::set_global_error(std::string(who) + ": " + hipGetErrorString(e));
    return AC_ERR_HIP;
  }
  return AC_OK;
}

int bad(const char* msg) {
  ac::set_global_error(msg);
  return AC_ERR_ARG;
}

unsigned grid_for(int64_t total, int block) {
  int64_t g = (total + block - 1) / block;
  return (unsigned)(g < 1 ? 1 : (g > (1 << 20) ? (1 << 20) : g));
}

// ---- cdist (src/ac.hxx:33-56) -------------------------------------------------------------------------------------
// out[j][i] = ||a_j - b_i||: the squared differences summed in FP64 in ascending feature order (one fma chain per
// pair), the root rounded once to FP32.  Both kernels below evaluate exactly that sequence, so they agree bit for bit.

// A thread per output.  Its b row is read element by element (lanes 4 * dim bytes apart) and again for every a row, and
// every pair converts its own operands: 4.99 ms for 16 x 1,000,003 outputs of 64 features.  Kept for short b and small
// calls of few features (ac_cdist), where a thread per b row would leave lanes or most of the chip idle.
__global__ void k_stage_cdist(int64_t n_a, int64_t n_b, int64_t dim, const float* __restrict__ a,
                              const float* __restrict__ b, float* __restrict__ out) {
  const int64_t total = n_a * n_b;
  for (int64_t o = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; o < total; o += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = o / n_b, i = o - j * n_b;
    const float* x = a + j * dim;
    const float* y = b + i * dim;
    double acc = 0.0;
    for (int64_t k = 0; k < dim; ++k) {
      const double d = (double)x[k] - (double)y[k];
      acc = fma(d, d, acc);
    }
    out[o] = (float)sqrt(acc);
  }
}

// R b rows per thread against JP rows of a, tiles of NT * R b rows staged in LDS kCdChunk features at a time by
// coalesced loads.  The a rows are wave-uniform: scalar loads, converted once per wave for R rows of every lane.
// Bound by the vector unit: 16 x 1,000,003 outputs of 64 features issue 48 M wave instructions (32 M of them the FP64
// subtractions and fmas), 91 us of issue on 1,024 SIMDs at 2.06 GHz, against 67 us for moving the 320 MB at a copy's
// 4.75 TB/s.  Measured there: 157 us (a thread per output: 4.99 ms); 4 x 4,000,000 of 13 features, bound by its bytes
// (57 us): 68 us.  R = 4 is no faster (152 us) and slower for narrow rows (87 us); chunks of 32 features halve the
// resident waves and gain nothing.
// Read-only inputs through the constant address space: loads at wave-uniform addresses become scalar loads.
typedef const __attribute__((address_space(4))) float cfloat_t;
constexpr int kCdChunk = 16;

// Elements t, t + NT, ... of the T x nc block at src (rows ld elements apart, rows past nr read as the last one), handed
// to put(row, column, value): T / NT * nc of them for every thread, U loads in flight at a time; (row, column) steps
// without a division.
template <int NT, int T, int U, typename V, typename Put>
__device__ __forceinline__ void stage_rows(const V* __restrict__ src, int64_t ld, int nr, int nc, int t, Put put) {
  const int dr = NT / nc, dc = NT % nc, total = T / NT * nc;
  int r = t / nc, c = t % nc, done = 0;
  auto step = [&] {
    r += dr, c += dc;
    if (c >= nc) c -= nc, ++r;
  };
  for (; done + U <= total; done += U) {
    V v[U];
    int r1 = r, c1 = c;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      v[u] = src[(r < nr ? r : nr - 1) * ld + c];
      step();
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      put(r1, c1, v[u]);
      r1 += dr, c1 += dc;
      if (c1 >= nc) c1 -= nc, ++r1;
    }
  }
  for (; done < total; ++done) {
    put(r, c, src[(r < nr ? r : nr - 1) * ld + c]);
    step();
  }
}

template <int JP, int R, int NT>
__global__ __launch_bounds__(NT) void k_stage_cdist_tile(int64_t n_a, int64_t n_b, int64_t dim,
                                                         const float* __restrict__ a, const float* __restrict__ b,
                                                         float* __restrict__ out, int64_t ntiles, int64_t ngroups) {
  constexpr int T = NT * R;
  __shared__ float xs[T][kCdChunk + 1];  // odd stride: a lane per row reads without bank conflicts
  const int t = threadIdx.x;
  const bool vec = (dim & 3) == 0 && (reinterpret_cast<uintptr_t>(b) & 15) == 0;
  for (int64_t w = blockIdx.x; w < ntiles * ngroups; w += gridDim.x) {
    const int64_t tile = w / ngroups, i0 = tile * T, j0 = (w - tile * ngroups) * JP;
    const int nt = (int)std::min<int64_t>(T, n_b - i0);
    double acc[JP][R];
#pragma unroll
    for (int j = 0; j < JP; ++j)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[j][r] = 0.0;
    cfloat_t* ar[JP];  // rows past n_a repeat the last one and are not stored
#pragma unroll
    for (int j = 0; j < JP; ++j) ar[j] = (cfloat_t*)(a + std::min(j0 + j, n_a - 1) * dim);
    for (int64_t k0 = 0; k0 < dim; k0 += kCdChunk) {
      const int cw = (int)std::min<int64_t>(kCdChunk, dim - k0);
      const float* src = b + i0 * dim + k0;
      __syncthreads();  // the previous chunk is consumed
      if (vec)
        stage_rows<NT, T, 4>(reinterpret_cast<const float4*>(src), dim / 4, nt, cw / 4, t, [&](int r, int c, float4 v) {
          xs[r][4 * c] = v.x, xs[r][4 * c + 1] = v.y, xs[r][4 * c + 2] = v.z, xs[r][4 * c + 3] = v.w;
        });
      else
        stage_rows<NT, T, 8>(src, dim, nt, cw, t, [&](int r, int c, float v) { xs[r][c] = v; });
      __syncthreads();
#pragma unroll 4
      for (int k = 0; k < cw; ++k) {
        double x[R];
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = (double)xs[t + r * NT][k];
#pragma unroll
        for (int j = 0; j < JP; ++j) {
          const double p = (double)ar[j][k0 + k];
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const double d = p - x[r];
            acc[j][r] = fma(d, d, acc[j][r]);
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < JP; ++j)
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (j0 + j < n_a && t + r * NT < nt) out[(j0 + j) * n_b + i0 + t + r * NT] = (float)sqrt(acc[j][r]);
  }
}

// ---- row log-softmax (src/ac.hxx:77-113) --------------------------------------------------------------------------
// Max-stabilised: x <- (x - m) - log1p(t), m the row maximum and t the sum of exp(x - m) over the row with one maximal
// element left out, so that log-probabilities near 0 keep relative accuracy.  One launch for rows that a block holds
// (k_lsm_row), else three, HBM-bound (one read for the partials, one read and one write to apply):
//   k_lsm_parts : block (row, chunk) accumulates (m, t) over its chunk of the row into parts[row * nchunk + chunk];
//   k_lsm_rows  : one block per row merges the row's partials in a fixed order into fin[row] = (m, log1p(t));
//   k_lsm_apply : block (row, chunk) writes its chunk normalised.
// The chunking depends only on (n_row, n_col), so the merge order, and with it every result, is the same from call to
// call and for the allocating and the static-scratch entry points.

constexpr int kLsmBlock = 256;
constexpr int64_t kLsmChunkMin = 8192;  // elements per chunk, at least (32 per thread)
// Scratch of one call, in ac::Lse entries: n_row * nchunk partials, then n_row finals.  The static scratch of
// ac_row_log_softmax_static holds this many (1 MiB), and both entry points size their chunking to fit it.
constexpr int64_t kLsmScratch = 1 << 16;

int64_t lsm_chunks(int64_t n_row, int64_t n_col) {
  const int64_t want = (n_col + kLsmChunkMin - 1) / kLsmChunkMin;
  const int64_t room = kLsmScratch / n_row - 1;
  return std::max<int64_t>(1, std::min(want, room));
}

__device__ __forceinline__ ac::Lse block_lse(ac::Lse s, ac::Lse* red) {
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = kLsmBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] = ac::lse_merge(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  const ac::Lse r = red[0];
  __syncthreads();
  return r;
}

__device__ __forceinline__ void chunk_range(int64_t n_col, int64_t nchunk, int64_t chunk, int64_t& c0, int64_t& c1) {
  const int64_t csize = (n_col + nchunk - 1) / nchunk;
  c0 = std::min(n_col, chunk * csize);
  c1 = std::min(n_col, c0 + csize);
}

// The elements [c0, c1) of x over a block of NT threads: four(c, x[c .. c + 3]) for the 16-byte aligned quadruples, four
// of them loaded together per thread, and one(c, x[c]) for the elements before and after them.
template <int NT, typename Four, typename One>
__device__ __forceinline__ void stream_chunk(const float* __restrict__ x, int64_t c0, int64_t c1, Four four, One one) {
  const int t = threadIdx.x;
  const int64_t head = std::min<int64_t>(c1 - c0, (4 - ((reinterpret_cast<uintptr_t>(x + c0) >> 2) & 3)) & 3);
  const int64_t b0 = c0 + head, n4 = (c1 - b0) / 4;
  if (t < head) one(c0 + t, x[c0 + t]);
  const float4* x4 = reinterpret_cast<const float4*>(x + b0);
  int64_t i = t;
  for (; i + 3 * NT < n4; i += 4 * NT) {
    const float4 v0 = x4[i], v1 = x4[i + NT], v2 = x4[i + 2 * NT], v3 = x4[i + 3 * NT];
    four(b0 + 4 * i, v0);
    four(b0 + 4 * (i + NT), v1);
    four(b0 + 4 * (i + 2 * NT), v2);
    four(b0 + 4 * (i + 3 * NT), v3);
  }
  for (; i < n4; i += NT) four(b0 + 4 * i, x4[i]);
  for (int64_t c = b0 + 4 * n4 + t; c < c1; c += NT) one(c, x[c]);
}

// Running log-sum-exp of floats, taken a few at a time: the maximum in FP32 (exact), the sum of exp(x - max) over all
// but one maximal element in FP64, its terms FP32 exponentials of the differences.  As lse_add, -inf adds nothing, a NaN
// makes the sum NaN, and so does a second +inf (inf - inf).
struct LseRun {
  float m = -INFINITY;
  double t = 0.0;
  template <int N>
  __device__ __forceinline__ void add(const float (&x)[N]) {
    float M = m;
#pragma unroll
    for (int u = 0; u < N; ++u) M = fmaxf(M, x[u]);
    int at = 0;  // maximal elements among x that count: all, or all but one where the maximum is new
    if (M > m) {
      t = (1.0 + t) * (double)__expf(m - M);
      at = -1;
    }
    double d = 0.0;
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const bool eq = x[u] == M;
      at += eq && M != -INFINITY;
      d += eq ? 0.0 : (double)__expf(x[u] - M);
    }
    t += d + (double)at;
    m = M;
  }
  __device__ __forceinline__ ac::Lse get() const {
    return ac::Lse{(double)m, m == INFINITY && t >= 1.0 ? (double)NAN : t};
  }
};

__global__ __launch_bounds__(kLsmBlock) void k_lsm_parts(int64_t n_col, int64_t nchunk, const float* __restrict__ x,
                                                         ac::Lse* __restrict__ parts) {
  __shared__ ac::Lse red[kLsmBlock];
  const int64_t row = blockIdx.x / nchunk, chunk = blockIdx.x - row * nchunk;
  int64_t c0, c1;
  chunk_range(n_col, nchunk, chunk, c0, c1);
  LseRun r;
  stream_chunk<kLsmBlock>(x + row * n_col, c0, c1, [&](int64_t, float4 v) {
    const float q[4] = {v.x, v.y, v.z, v.w};
    r.add(q);
  }, [&](int64_t, float v) {
    const float q[1] = {v};
    r.add(q);
  });
  ac::Lse s = r.get();
  s = block_lse(s, red);
  if (threadIdx.x == 0) parts[blockIdx.x] = s;
}

__global__ __launch_bounds__(kLsmBlock) void k_lsm_rows(int64_t nchunk, const ac::Lse* __restrict__ parts,
                                                        ac::Lse2* __restrict__ fin) {
  __shared__ ac::Lse red[kLsmBlock];
  const int64_t row = blockIdx.x;
  ac::Lse s = ac::lse_empty();
  for (int64_t k = threadIdx.x; k < nchunk; k += kLsmBlock) s = ac::lse_merge(s, parts[row * nchunk + k]);
  s = block_lse(s, red);
  if (threadIdx.x == 0) fin[row] = ac::Lse2{s.m, log1p(s.t)};
}

__global__ __launch_bounds__(kLsmBlock) void k_lsm_apply(int64_t n_col, int64_t nchunk, float* __restrict__ x,
                                                         const ac::Lse2* __restrict__ fin) {
  const int64_t row = blockIdx.x / nchunk, chunk = blockIdx.x - row * nchunk;
  int64_t c0, c1;
  chunk_range(n_col, nchunk, chunk, c0, c1);
  const ac::Lse2 f = fin[row];
  float* xr = x + row * n_col;
  auto one = [&](float v) { return (float)(((double)v - f.m) - f.l); };
  stream_chunk<kLsmBlock>(xr, c0, c1, [&](int64_t c, float4 v) {
    *reinterpret_cast<float4*>(xr + c) = make_float4(one(v.x), one(v.y), one(v.z), one(v.w));
  }, [&](int64_t c, float v) { xr[c] = one(v); });
}

// Rows of up to 32 * 1024 elements in one launch, a block of NT threads per row, the row in registers.  Bound by one
// block's latency (12 x 20,000: 11.0 us), which costs less than three launches and a stream-ordered allocation: distance,
// log-softmax and row maximum of that size take 21 us in place of 35.  A thread's elements, which a NaN's reach depends
// on when the row is shorter than the block, are those of k_lsm_parts.
constexpr int kRowRegs = 32;
constexpr int64_t kRowMax = (int64_t)kRowRegs * 1024;
template <int NT>
__global__ __launch_bounds__(NT) void k_lsm_row(int64_t n_col, float* __restrict__ x) {
  __shared__ ac::Lse red[NT / 64];
  float* xr = x + (int64_t)blockIdx.x * n_col;
  const int t = threadIdx.x, lane = t & 63, n = (int)n_col;
  float v[kRowRegs];
#pragma unroll
  for (int u = 0; u < kRowRegs; ++u) {
    v[u] = -INFINITY;  // adds nothing
    if (u * NT < n && t + u * NT < n) v[u] = xr[t + u * NT];
  }
  LseRun r;
#pragma unroll
  for (int u = 0; u < kRowRegs; u += 4)
    if (u * NT < n) {
      const float q[4] = {v[u], v[u + 1], v[u + 2], v[u + 3]};
      r.add(q);
    }
  ac::Lse s = ac::lanes_lse_merge(r.get(), 64);
  if (lane == 0) red[t >> 6] = s;
  __syncthreads();
  s = ac::lanes_lse_merge(lane < NT / 64 ? red[lane] : ac::lse_empty(), 64);
  if (s.m == (double)INFINITY && s.t >= 1.0) s.t = NAN;  // +inf in more than one lane
  const double l = log1p(s.t);
#pragma unroll
  for (int u = 0; u < kRowRegs; ++u)
    if (u * NT < n && t + u * NT < n) xr[t + u * NT] = (float)(((double)v[u] - s.m) - l);
}

// The three launches on `scratch`, which holds lsm_entries(n_row, n_col) entries.
int64_t lsm_entries(int64_t n_row, int64_t n_col) { return n_row * (lsm_chunks(n_row, n_col) + 1); }

// Launches over n_row rows with a block of nt threads for each of a row's `per` parts, in slices of rows whose grids
// stay at 2^31 threads (a grid takes fewer than 2^32): go(first row, rows).
template <typename Go>
void for_row_slices(int64_t n_row, int64_t per, int nt, Go go) {
  const int64_t slice = std::max<int64_t>(1, (int64_t(1) << 31) / (nt * per));
  for (int64_t r0 = 0; r0 < n_row; r0 += slice) go(r0, (unsigned)std::min(slice, n_row - r0));
}

// The whole operator in one launch where the rows fit: every entry point takes this path first.
bool lsm_fused(int64_t n_col) { return n_col <= kRowMax; }

int enqueue_row_lsm(int64_t n_row, int64_t n_col, float* x, ac::Lse* scratch, hipStream_t st, const char* who) {
  if (lsm_fused(n_col)) {
    // The smallest block that holds a row where there are more rows than CUs (256), so that a CU works on several at once:
    // 4,096 x 4,097 in 31 us with blocks of 256, 82 with 1,024 (three launches: 51); 4,096 x 12,000 69 with 512, 108 with
    // 1,024 (114).  Few rows take the largest, whose threads have the fewest elements: 256 x 4,097 in 7.6 us.
    const bool many = n_row > 256;
    const int nt = n_col <= 16 * kLsmBlock || (many && n_col <= kRowRegs * kLsmBlock) ? kLsmBlock
                   : many && n_col <= kRowRegs * 512                                  ? 512
                                                                                      : 1024;
    const auto kernel = nt == kLsmBlock ? k_lsm_row<kLsmBlock> : nt == 512 ? k_lsm_row<512> : k_lsm_row<1024>;
    for_row_slices(n_row, 1, nt, [&](int64_t r0, unsigned rows) {
      hipLaunchKernelGGL(kernel, dim3(rows), dim3(nt), 0, st, n_col, x + r0 * n_col);
    });
    return launch_status(who);
  }
  // (Rows this long are below 2^24 blocks in any memory.)
  const int64_t nchunk = lsm_chunks(n_row, n_col);
  const int64_t nblk = n_row * nchunk;
  ac::Lse2* fin = reinterpret_cast<ac::Lse2*>(scratch + nblk);
  hipLaunchKernelGGL(k_lsm_parts, dim3((unsigned)nblk), dim3(kLsmBlock), 0, st, n_col, nchunk, x, scratch);
  hipLaunchKernelGGL(k_lsm_rows, dim3((unsigned)n_row), dim3(kLsmBlock), 0, st, nchunk, scratch, fin);
  hipLaunchKernelGGL(k_lsm_apply, dim3((unsigned)nblk), dim3(kLsmBlock), 0, st, n_col, nchunk, x, fin);
  return launch_status(who);
}

// Scratch of ac_row_log_softmax_static: one copy per GPU, held until the process ends.  Host code reaches it only
// through the address hipGetSymbolAddress returns on each device; the array's name itself is a host-side stand-in.
static __device__ __align__(256) ac::Lse scratch[kLsmScratch];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
ac::Lse* g_scratch_ptr[kMaxDevices] = {};

// The scratch's address on the current device, looked up on the first call there (with that device current).
int static_scratch(ac::Lse** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    ac::set_global_error(std::string("ac_row_log_softmax_static: hipGetDevice: ") + hipGetErrorString(e));
    return AC_ERR_HIP;
  }
  if (dev < 0 || dev >= kMaxDevices) return bad("ac_row_log_softmax_static: device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      ac::set_global_error(std::string("ac_row_log_softmax_static: hipGetSymbolAddress: ") + hipGetErrorString(e));
      return AC_ERR_HIP;
    }
    g_scratch_ptr[dev] = static_cast<ac::Lse*>(p);
  }
  *out = g_scratch_ptr[dev];
  return AC_OK;
}

// Float max as integer atomics: non-negative floats order like signed ints, negative floats order inversely to
// their unsigned bit patterns, so the result is exact and independent of the order of the updates.
__device__ __forceinline__ void atomic_max_float(float* addr, float v) {
  if (!(v < 0.f) && !signbit(v))
    atomicMax(reinterpret_cast<int*>(addr), __float_as_int(v));
  else
    atomicMin(reinterpret_cast<unsigned int*>(addr), __float_as_uint(v));
}

// ---- row max (src/ac.hxx:58-75) -----------------------------------------------------------------------------------
// out[r] starts at -inf (k_stage_fill_rows without fill values), then block (row, chunk) reduces its chunk with wave
// shuffles and folds the result in with one atomic; rows of one chunk need neither.  Max is exact and order-free, so no
// scratch is needed.  Bound by the one read and by the atomics, which follow each other on the few cache lines of out:
// as many chunks as fill the chip once with blocks of 1024 threads, and no more (16 x 1,000,003: 37 us with 1968 blocks,
// 12.5 with 256; 12 x 262,144: 9.9 and 7.3).
constexpr int kMaxBlock = 256;
constexpr int64_t kRowMaxBlocks = 256;

template <int NT>
__global__ __launch_bounds__(NT) void k_stage_row_max(int64_t n_col, int64_t nchunk, const float* __restrict__ in,
                                                      float* __restrict__ out) {
  __shared__ float red[NT / 64];
  const int64_t row = blockIdx.x / nchunk, chunk = blockIdx.x - row * nchunk;
  int64_t c0, c1;
  chunk_range(n_col, nchunk, chunk, c0, c1);
  float m = -INFINITY;
  stream_chunk<NT>(in + row * n_col, c0, c1, [&](int64_t, float4 v) {
    m = fmaxf(m, fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)));
  }, [&](int64_t, float v) { m = fmaxf(m, v); });
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < NT / 64; ++w) m = fmaxf(m, red[w]);
    if (nchunk == 1)
      out[row] = m;
    else
      atomic_max_float(out + row, m);
  }
}

// ac::EdgeMaxReduce2_t (src/ac.hxx:115-149): fill, then scatter-max.  The fill of long rows: a block per (row, chunk),
// 16-byte stores and no division per element (16 x 262,144: 5.9 us; 6.4 a thread per element, as short rows have it).
__global__ __launch_bounds__(kMaxBlock) void k_stage_fill_long(int64_t n_col, int64_t nchunk,
                                                               const float* __restrict__ vymax,
                                                               float* __restrict__ xmax) {
  const int64_t row = blockIdx.x / nchunk, chunk = blockIdx.x - row * nchunk;
  int64_t c0, c1;
  chunk_range(n_col, nchunk, chunk, c0, c1);
  const float v = vymax[row];
  float* x = xmax + row * n_col;
  const int64_t head = std::min<int64_t>(c1 - c0, (4 - ((reinterpret_cast<uintptr_t>(x + c0) >> 2) & 3)) & 3);
  const int64_t b0 = c0 + head, n4 = (c1 - b0) / 4;
  if ((int)threadIdx.x < head) x[c0 + threadIdx.x] = v;
  for (int64_t i = threadIdx.x; i < n4; i += kMaxBlock) reinterpret_cast<float4*>(x + b0)[i] = make_float4(v, v, v, v);
  for (int64_t c = b0 + 4 * n4 + threadIdx.x; c < c1; c += kMaxBlock) x[c] = v;
}
__global__ void k_stage_fill_rows(int64_t n_row, int64_t n_col, const float* __restrict__ vymax,
                                  float* __restrict__ xmax) {
  const int64_t total = n_row * n_col;
  for (int64_t o = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; o < total; o += (int64_t)gridDim.x * blockDim.x)
    xmax[o] = vymax ? vymax[o / n_col] : -INFINITY;
}
// v can raise the entry x (bitwise: +0.0 raises -0.0, as in the atomic's order).
__device__ __forceinline__ bool above(float v, float x) { return !(v < x) && __float_as_uint(v) != __float_as_uint(x); }

// Bound by the one read of xe.  A value at or below its row's fill can change nothing, so only the others look at
// their node, and of those only the ones above its present value (read without an atomic: the entries only rise, so a
// stale value is a low one) issue the atomic.  R-MAT 18's 16 x 3.94 M values into 16 x 262,144, with the fill pass, by the
// share of them above their fill: none 43 us (5.9 TB/s), 0.1 % 55 by source and 59 by destination, 12 % 237 and 478, all 741
// and 1,473 us; an atomic per value took 8.8-9.2 and 5.6-5.8 ms.  In the iterations of a matcher the share is 0 to 2 % by
// source and 0 by destination (1,000 vertices, 10/12 pattern), 0 to 12 % and 0 to 0.14 % (R-MAT 14, 24/36), 0 to 0.2 % and
// 0 (R-MAT 15, 12/16).  NaNs pass both comparisons and reach the atomic.
__global__ __launch_bounds__(kMaxBlock) void k_stage_scatter_max(int64_t n_col_in, int64_t n_col_out, int64_t nchunk,
                                                                 const float* __restrict__ vymax,
                                                                 const float* __restrict__ xe,
                                                                 float* __restrict__ xmax,
                                                                 const int* __restrict__ nodes) {
  const int64_t row = blockIdx.x / nchunk, chunk = blockIdx.x - row * nchunk;
  int64_t c0, c1;
  chunk_range(n_col_in, nchunk, chunk, c0, c1);
  const float fill = vymax[row];
  float* out = xmax + row * n_col_out;
  stream_chunk<kMaxBlock>(xe + row * n_col_in, c0, c1, [&](int64_t c, float4 v) {
    if (!(above(v.x, fill) || above(v.y, fill) || above(v.z, fill) || above(v.w, fill))) return;
    const float vv[4] = {v.x, v.y, v.z, v.w};
    // One after the other: neighbours often share a node (edges sorted by source), and each then sees the last one's.
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (above(vv[u], fill)) {
        float* e = out + nodes[c + u];
        if (above(vv[u], __hip_atomic_load(e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))) atomic_max_float(e, vv[u]);
      }
  }, [&](int64_t c, float v) {
    if (above(v, fill)) atomic_max_float(out + nodes[c], v);
  });
}

// Rows shorter than a block and small calls: a thread per value, whatever its row.
__global__ __launch_bounds__(kMaxBlock) void k_stage_scatter_short(int64_t n_row, int64_t n_col_in, int64_t n_col_out,
                                                                   const float* __restrict__ vymax,
                                                                   const float* __restrict__ xe,
                                                                   float* __restrict__ xmax,
                                                                   const int* __restrict__ nodes) {
  const int64_t total = n_row * n_col_in;
  for (int64_t o = blockIdx.x * (int64_t)kMaxBlock + threadIdx.x; o < total; o += (int64_t)gridDim.x * kMaxBlock) {
    const int64_t row = o / n_col_in;
    const float v = xe[o];
    if (above(v, vymax[row])) atomic_max_float(xmax + row * n_col_out + nodes[o - row * n_col_in], v);
  }
}

// ac::ComputeMU2_t (src/ac.hxx:151-186), summed per data vertex in ascending q, FP64, rounded once.  Block (v tile,
// p): the incident pattern edges are the same for the whole block and are listed first; their values are then read
// kMuBatch rows at a time and added in order.  kV elements of a row per thread (4: 16-byte accesses, where every row
// starts on that grid).  Bound by the read of both matrices, each once per endpoint: 12 x 16, 262,144 columns in 13.7 us
// (31 with scalar loads issued one edge after another).  More incident edges than a list holds are listed and added
// part by part (read one by one as they were met, 2,000 edges on 2 vertices, 5,000 columns: 731 us, now 235).
constexpr int kMuList = 512, kMuBatch = 4;
template <int kV>
__global__ __launch_bounds__(256) void k_stage_compute_mu(int64_t n_col_in, int64_t n_row_in, int64_t n_col_out,
                                                          int64_t n_row_out, const float* __restrict__ cv,
                                                          const float* __restrict__ fmax,
                                                          const float* __restrict__ rmax,
                                                          const int* __restrict__ srcs, const int* __restrict__ dsts,
                                                          float* __restrict__ mu) {
  typedef float vec __attribute__((ext_vector_type(kV)));
  __shared__ const float* list[kMuList];  // rows to add, in ascending q, the fmax term before the rmax term
  __shared__ int len;
  __shared__ int64_t next;  // the first q that is not listed yet
  for (int64_t p = blockIdx.y; p < n_row_out; p += gridDim.y) {
    for (int64_t v0 = blockIdx.x * (int64_t)256 * kV; v0 < n_col_out; v0 += (int64_t)gridDim.x * 256 * kV) {
      const int64_t v = v0 + threadIdx.x * kV, o = p * n_col_out + v;
      const bool in = v < n_col_out;
      vec c = 0.f;
      if (in) c = *reinterpret_cast<const vec*>(cv + o);
      double acc[kV];
#pragma unroll
      for (int e = 0; e < kV; ++e) acc[e] = -(double)c[e];
      for (int64_t q1 = 0; q1 < n_row_in; q1 = next) {  // listed piece by piece where one list does not hold them
        __syncthreads();
        if (threadIdx.x < 64) {  // one wave lists them: a ballot gives each its place
          int at = 0;
          int64_t q0 = q1;
          for (; q0 < n_row_in && at + 128 <= kMuList; q0 += 64) {
            const int64_t q = q0 + threadIdx.x;
            const bool f = q < n_row_in && dsts[q] == p, r = q < n_row_in && srcs[q] == p;
            const unsigned long long below = (1ull << threadIdx.x) - 1ull, bf = __ballot(f), br = __ballot(r);
            const int i = at + __popcll(bf & below) + __popcll(br & below);
            if (f) list[i] = fmax + q * n_col_in;
            if (r) list[i + (f ? 1 : 0)] = rmax + q * n_col_in;
            at += __popcll(bf) + __popcll(br);
          }
          if (threadIdx.x == 0) len = at, next = q0;
        }
        __syncthreads();
        const int n = len;
        if (v < n_col_in && in) {
          int k = 0;
          for (; k + kMuBatch <= n; k += kMuBatch) {
            vec x[kMuBatch];
#pragma unroll
            for (int u = 0; u < kMuBatch; ++u) x[u] = *reinterpret_cast<const vec*>(list[k + u] + v);
#pragma unroll
            for (int u = 0; u < kMuBatch; ++u)
#pragma unroll
              for (int e = 0; e < kV; ++e) acc[e] += (double)x[u][e];
          }
          for (; k < n; ++k) {
            const vec x = *reinterpret_cast<const vec*>(list[k] + v);
#pragma unroll
            for (int e = 0; e < kV; ++e) acc[e] += (double)x[e];
          }
        }
      }
      if (!in) continue;
      vec out;
#pragma unroll
      for (int e = 0; e < kV; ++e) out[e] = (float)acc[e];
      *reinterpret_cast<vec*>(mu + o) = out;
    }
  }
}

// ac::transpose (src/ac.hxx:17-31).  (One side is a pattern's few columns: tiles through LDS took as long.)
__global__ void k_stage_transpose(const float* __restrict__ in, float* __restrict__ out, int64_t n_rows,
                                  int64_t n_cols) {
  const int64_t total = n_rows * n_cols;
  for (int64_t o = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; o < total; o += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = o / n_rows, r = o - c * n_rows;
    out[o] = in[r * n_cols + c];
  }
}

}  // namespace

extern "C" int ac_cdist(int64_t n_a, int64_t n_b, int64_t dim, const float* feats_a, const float* feats_b, float* out,
                        void* stream) {
  if (n_a < 0 || n_b < 0 || dim < 0 || (n_a * n_b > 0 && (!out || (dim > 0 && (!feats_a || !feats_b)))))
    return bad("ac_cdist: bad arguments");
  if (n_a * n_b == 0) return AC_OK;
  hipStream_t st = as_stream(stream);
  // A thread per output where a wave of b rows would leave lanes idle and the reads cost little: b shorter than a wave,
  // or small enough as a whole to stay in the cache (50,001 x 65 of 5 features 16.0 against 18.7 us; 50,001 x 80 of 8: 62
  // against 18.8), and for small calls of few features, a launch's latency (12 x 1,000 of 13: 3.6 against 4.5 us; 24 x
  // 3,000 of 16: 5.5 against 4.4).
  if (n_b < 64 || n_b * dim < 384 || (dim <= 24 && n_a * n_b < 1'500'000 / std::max<int64_t>(1, dim))) {
    hipLaunchKernelGGL(k_stage_cdist, dim3(grid_for(n_a * n_b, 256)), dim3(256), 0, st, n_a, n_b, dim, feats_a,
                       feats_b, out);
    return launch_status("ac_cdist");
  }
  // The a rows in ngroups groups of equal size, at most 16 (a multiple of 4): 24 rows as 2 x 12 rather than 16 + 8.  Groups
  // of four where those of 16 would be fewer than two waves for each of the 256 CUs, since a wave takes its rows one after
  // the other: 16 x 1,000 of 64 features 15.0 -> 6.6 us (a thread per output: 10.0), 16 x 16,000 15.3 -> 7.8 us.
  const bool few = (n_b + 63) / 64 * ((n_a + 15) / 16) < 512;
  const int64_t ngroups = few ? (n_a + 3) / 4 : (n_a + 15) / 16;
  const int jp = (int)((n_a + ngroups - 1) / ngroups + 3) / 4 * 4;
  // Short b takes one wave and one row per thread, so that the tiles reach more of the chip and fewer rows are idle in
  // the last one (100,000 x 100 of 13 features 65 -> 41 us).
  const bool small = few || n_b <= 192 || n_b * ngroups < (int64_t)256 * 2048;
  const int64_t ntiles = (n_b + (small ? 63 : 255)) / (small ? 64 : 256);
  const unsigned blocks = (unsigned)std::min<int64_t>(ntiles * ngroups, 1 << 20);
#define AC_STAGE_CD(JP)                                                                                             \
  case JP:                                                                                                          \
    if (small)                                                                                                      \
      hipLaunchKernelGGL((k_stage_cdist_tile<JP, 1, 64>), dim3(blocks), dim3(64), 0, st, n_a, n_b, dim, feats_a,    \
                         feats_b, out, ntiles, ngroups);                                                            \
    else                                                                                                            \
      hipLaunchKernelGGL((k_stage_cdist_tile<JP, 2, 128>), dim3(blocks), dim3(128), 0, st, n_a, n_b, dim, feats_a,  \
                         feats_b, out, ntiles, ngroups);                                                            \
    break;
  switch (jp) {
    AC_STAGE_CD(4)
    AC_STAGE_CD(8)
    AC_STAGE_CD(12)
    AC_STAGE_CD(16)
  }
#undef AC_STAGE_CD
  return launch_status("ac_cdist");
}

extern "C" int ac_row_log_softmax(int64_t n_row, int64_t n_col, float* x, void* stream) {
  if (n_row < 0 || n_col < 0 || n_row > INT32_MAX || (n_row * n_col > 0 && !x)) return bad("ac_row_log_softmax: bad arguments");
  if (n_row * n_col == 0) return AC_OK;
  hipStream_t st = as_stream(stream);
  if (lsm_fused(n_col)) return enqueue_row_lsm(n_row, n_col, x, nullptr, st, "ac_row_log_softmax");
  // Stream-ordered temporary (the reference's RowSoftmax2 allocates its own too, src/ac.hxx:108-113).
  ac::Lse* tmp = nullptr;
  hipError_t e = hipMallocAsync((void**)&tmp, (size_t)lsm_entries(n_row, n_col) * sizeof(ac::Lse), st);
  if (e != hipSuccess) {
    ac::set_global_error(std::string("ac_row_log_softmax: hipMallocAsync: ") + hipGetErrorString(e));
    return e == hipErrorOutOfMemory ? AC_ERR_OOM : AC_ERR_HIP;
  }
  const int rc = enqueue_row_lsm(n_row, n_col, x, tmp, st, "ac_row_log_softmax");
  e = hipFreeAsync(tmp, st);
  if (rc != AC_OK) return rc;
  if (e != hipSuccess) {
    ac::set_global_error(std::string("ac_row_log_softmax: hipFreeAsync: ") + hipGetErrorString(e));
    return AC_ERR_HIP;
  }
  return AC_OK;
}

extern "C" int ac_row_log_softmax_static(int64_t n_row, int64_t n_col, float* x, void* stream) {
  if (n_row < 0 || n_col < 0 || (n_row * n_col > 0 && !x)) return bad("ac_row_log_softmax_static: bad arguments");
  if (n_row > kLsmScratch / 2)
    return bad("ac_row_log_softmax_static: more than 32768 rows (its fixed scratch holds 65536 partials)");
  if (n_row * n_col == 0) return AC_OK;
  ac::Lse* scr = nullptr;
  const int rc = static_scratch(&scr);
  if (rc != AC_OK) return rc;
  return enqueue_row_lsm(n_row, n_col, x, scr, as_stream(stream), "ac_row_log_softmax_static");
}

extern "C" int ac_row_max(int64_t n_row, int64_t n_col, const float* in, float* out, void* stream) {
  if (n_row < 0 || n_col < 0 || n_row > INT32_MAX || (n_row > 0 && (!out || (n_col > 0 && !in))))
    return bad("ac_row_max: bad arguments");
  if (n_row == 0) return AC_OK;
  hipStream_t st = as_stream(stream);
  const int64_t nchunk = n_col <= kRowMax ? 1 : std::min<int64_t>((n_col + kLsmChunkMin - 1) / kLsmChunkMin,
                                                                  std::max<int64_t>(1, kRowMaxBlocks / n_row));
  if (n_col == 0 || nchunk > 1)
    hipLaunchKernelGGL(k_stage_fill_rows, dim3(grid_for(n_row, 256)), dim3(256), 0, st, n_row, (int64_t)1,
                       (const float*)nullptr, out);
  // The larger block where a row has work for it; short rows a wave each (1,000,000 x 4 223 us, 810 with blocks of 256;
  // 30,000 x 1,000 22.4 and 28.7 us).
  const int nt = n_col <= 1024 ? 64 : n_col <= kLsmChunkMin ? kMaxBlock : 1024;
  const auto kernel = nt == 64 ? k_stage_row_max<64> : nt == kMaxBlock ? k_stage_row_max<kMaxBlock> : k_stage_row_max<1024>;
  if (n_col > 0)
    for_row_slices(n_row, nchunk, nt, [&](int64_t r0, unsigned rows) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)(rows * nchunk)), dim3(nt), 0, st, n_col, nchunk, in + r0 * n_col, out + r0);
    });
  return launch_status("ac_row_max");
}

extern "C" int ac_edge_max_reduce(int64_t n_col_in, int64_t n_col_out, int64_t n_row, const float* vymax,
                                  const float* xe, float* xmax, const int32_t* nodes, void* stream) {
  if (n_col_in < 0 || n_col_out < 0 || n_row < 0 || (n_row * n_col_out > 0 && (!vymax || !xmax)) ||
      (n_row * n_col_in > 0 && (!xe || !nodes)))
    return bad("ac_edge_max_reduce: bad arguments");
  hipStream_t st = as_stream(stream);
  const int64_t fchunk = (n_col_out + 4095) / 4096;
  if (n_col_out >= 4096 && n_row > 0 && n_row <= (1 << 23) / fchunk)  // (below 2^32 threads)
    hipLaunchKernelGGL(k_stage_fill_long, dim3((unsigned)(n_row * fchunk)), dim3(kMaxBlock), 0, st, n_col_out, fchunk,
                       vymax, xmax);
  else if (n_row * n_col_out > 0)
    hipLaunchKernelGGL(k_stage_fill_rows, dim3(grid_for(n_row * n_col_out, 256)), dim3(256), 0, st, n_row,
                       n_col_out, vymax, xmax);
  // Small calls take a thread per value too, whose reads do not follow each other (16 x 4,000 values above their fill 7.8 us,
  // 9.3 in chunks; 60,000 of one row 7.8 and 16.7): up to 2^17 values, or 2^18 of rows shorter than a chunk.
  const bool few = n_row * n_col_in <= (n_col_in < 1024 ? 1 << 18 : 1 << 17);
  if ((few || n_col_in < kMaxBlock) && n_row * n_col_in > 0) {
    hipLaunchKernelGGL(k_stage_scatter_short, dim3(grid_for(n_row * n_col_in, kMaxBlock)), dim3(kMaxBlock), 0, st, n_row,
                       n_col_in, n_col_out, vymax, xe, xmax, nodes);
  } else if (n_row * n_col_in > 0) {
    // Chunks of 8192 values (32 a thread), shorter ones down to 1024 where fewer than 2048 blocks would result (a
    // block of low-fill values is a chain of dependent reads and atomics: 39 us for 16 x 20,000 values in chunks of
    // 8192, 15 us in chunks of 1024).
    const int64_t csize = std::min<int64_t>(8192, std::max<int64_t>(1024, (n_col_in / 2048) * std::min<int64_t>(n_row, 8192)));
    const int64_t nchunk = std::max<int64_t>(1, std::min<int64_t>((n_col_in + csize - 1) / csize, 1 << 23));
    for_row_slices(n_row, nchunk, kMaxBlock, [&](int64_t r0, unsigned rows) {
      hipLaunchKernelGGL(k_stage_scatter_max, dim3((unsigned)(rows * nchunk)), dim3(kMaxBlock), 0, st, n_col_in, n_col_out,
                         nchunk, vymax + r0, xe + r0 * n_col_in, xmax + r0 * n_col_out, nodes);
    });
  }
  return launch_status("ac_edge_max_reduce");
}

extern "C" int ac_compute_mu(int64_t n_col_in, int64_t n_row_in, int64_t n_col_out, int64_t n_row_out,
                             const float* cv, const float* fmax, const float* rmax, const int32_t* srcs,
                             const int32_t* dsts, float* mu, void* stream) {
  if (n_col_in < 0 || n_row_in < 0 || n_col_out < 0 || n_row_out < 0 ||
      (n_row_out * n_col_out > 0 && (!cv || !mu)) || (n_row_in > 0 && (!fmax || !rmax || !srcs || !dsts)))
    return bad("ac_compute_mu: bad arguments");
  if (n_row_out * n_col_out == 0) return AC_OK;
  // Four elements a thread where both widths are multiples of four and every matrix starts on a 16-byte boundary.
  const uintptr_t bits = reinterpret_cast<uintptr_t>(cv) | reinterpret_cast<uintptr_t>(mu) |
                         (n_row_in > 0 ? reinterpret_cast<uintptr_t>(fmax) | reinterpret_cast<uintptr_t>(rmax) : 0);
  const bool vec = (n_col_in & 3) == 0 && (n_col_out & 3) == 0 && (bits & 15) == 0;
  const int64_t per = vec ? 1024 : 256;
  const dim3 grid((unsigned)std::min<int64_t>((n_col_out + per - 1) / per, 1 << 16),
                  (unsigned)std::min<int64_t>(n_row_out, 4096));
  hipLaunchKernelGGL(vec ? k_stage_compute_mu<4> : k_stage_compute_mu<1>, grid, dim3(256), 0, as_stream(stream), n_col_in,
                     n_row_in, n_col_out, n_row_out, cv, fmax, rmax, srcs, dsts, mu);
  return launch_status("ac_compute_mu");
}

extern "C" int ac_transpose(const float* in, float* out, int64_t n_rows, int64_t n_cols, void* stream) {
  if (n_rows < 0 || n_cols < 0 || (n_rows * n_cols > 0 && (!in || !out))) return bad("ac_transpose: bad arguments");
  if (n_rows * n_cols == 0) return AC_OK;
  hipLaunchKernelGGL(k_stage_transpose, dim3(grid_for(n_rows * n_cols, 256)), dim3(256), 0, as_stream(stream), in,
                     out, n_rows, n_cols);
  return launch_status("ac_transpose");
}
