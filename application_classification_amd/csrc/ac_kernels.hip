// Matcher kernels for gfx950 (CDNA4, wave64).
//
// Dataflow of one iteration (src/main.cu:160-245), reorganised so that no pattern-edge x data-edge matrix other than
// the edge costs CE is ever stored, and so that every stored value is normalised (small in magnitude near the
// matches that decide the output), with all arithmetic in FP64 registers:
//   vertex pass A  : MU = LSM(-CV + sum FMax + sum RMax) (recomputed, never stored), VF = MU[pd] - FMax,
//                    VR = MU[ps] - RMax; stores VR and VFm = VF - minCEo; column maxima and the two edge
//                    log-sum-exps, using  sum_e exp(X[src e] - CE_e) = sum_v exp(X[v] - minCEo[v] + lsO[v]).
//   edge walk B    : FMaxN[v] = max over in-edges of (VR[src] - CE) - LSE_FE   (CSC order; the pieces of a vertex with a
//                    long in-edge list raise its row by atomic maxima)
//   vertex pass C  : column log-sum-exp of MU for the next iteration's normalisation.
// RMax needs no edge pass: max over out-edges of (VF[v] - CE_e) = VF[v] - min over out-edges of CE_e, exactly.
// The log-softmax of CE and CV in the reference's prep (src/main.cu:116,118) shift each row by a constant, which
// every later log-softmax removes again, so the raw costs are used.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <type_traits>

#include "ac_internal.hpp"
#include "ac_lse.hpp"
#include "ac_sqrt_rn.hpp"

namespace ac {

namespace {

constexpr double kInf = __builtin_huge_val();

// Edge costs are row-major [rows][Qs].
__device__ __forceinline__ int64_t ce_index(int64_t k, int q, int Qs) { return k * Qs + q; }

// Native 4-wide vector (register-resident across loop iterations, unlike the HIP float4 wrapper struct).
typedef float f4v __attribute__((ext_vector_type(4)));

// Streaming loads (__builtin_nontemporal_load): data read once per pass (edge costs, edge ids) is loaded
// non-temporally so that it does not evict the gathered rows that are reused from L2.

// Packed costs: four 24-bit codes in three dwords, c0 | c1 << 24, c1 >> 8 | c2 << 16, c2 >> 16 | c3 << 8.  A code
// is the cost's bit pattern minus the bundle's base (a biased exponent << 23, so one bundle spans two binades);
// code 0 stands for +inf (padding rows and columns past Q).
struct U3 {
  unsigned x, y, z;
};
__device__ __forceinline__ U3 nt_load_u3(const unsigned* p) {
  return U3{__builtin_nontemporal_load(p), __builtin_nontemporal_load(p + 1), __builtin_nontemporal_load(p + 2)};
}
__device__ __forceinline__ float decode_cost(unsigned c, unsigned base) {
  return c ? __uint_as_float(base + c) : INFINITY;
}
__device__ __forceinline__ f4v decode_costs(U3 w, unsigned base) {
  const unsigned c0 = w.x & 0xFFFFFFu;
  const unsigned c1 = __builtin_amdgcn_alignbit(w.y, w.x, 24) & 0xFFFFFFu;
  const unsigned c2 = __builtin_amdgcn_alignbit(w.z, w.y, 16) & 0xFFFFFFu;
  const unsigned c3 = w.z >> 8;
  return f4v{decode_cost(c0, base), decode_cost(c1, base), decode_cost(c2, base), decode_cost(c3, base)};
}

// max with the position of the maximum: the larger value wins, equal values keep the lower vertex (-1 = none).
__device__ __forceinline__ void argmax_merge(double& m, int& a, double x, int b) {
  if (x > m || (x == m && b >= 0 && (a < 0 || b < a))) {
    m = x;
    a = b;
  }
}

}  // namespace

// ---------------------------------------------------------------------------------------------------------------
// cdist (src/ac.hxx:33-56): out[r][c] = || feats[row r] - pat_c ||, FP64 accumulation of (a - b)^2 rounded once to
// FP32.  Pattern features are [Kp / 8][dim][8] doubles (Kp = K rounded up to 8, zero padded: each group of eight
// patterns is one contiguous block, eight values per feature); row r of the output reads
// feature row idx[r] (idx == nullptr: row r).  Columns K <= c < Kstore of the output are written as 0, and rows with
// idx[r] < 0 (padding of the bundle layout) as +inf.  With w != nullptr the distance is weighted per dimension,
// sqrt(sum_k w_k (a_k - b_k)^2) (the learnable feature metric of the adjoint).

constexpr int kCdTile = 128;

// A tile of kCdTile feature rows is staged in LDS with row-contiguous (coalesced) loads; each thread then computes
// one row's distances to eight patterns at a time, the pattern values being wave-uniform (scalar loads).
template <bool kW>
__global__ __launch_bounds__(kCdTile) void k_cdist_rows(int64_t nrows, const int* __restrict__ idx,
                                                        const float* __restrict__ feats, int dim,
                                                        const double* __restrict__ pat, int K, int Kp, int Kstore,
                                                        float* __restrict__ out, int out_stride, int tile,
                                                        const double* __restrict__ w) {
  extern __shared__ float rows[];  // [tile][dim + 1], tile <= kCdTile
  const int ld = dim + 1;
  for (int64_t base = blockIdx.x * (int64_t)tile; base < nrows; base += (int64_t)gridDim.x * tile) {
    const int nt = (int)((nrows - base) < tile ? (nrows - base) : tile);
    __syncthreads();
    for (int e = threadIdx.x; e < nt * dim; e += kCdTile) {
      const int r = e / dim, c = e - r * dim;
      const int64_t src = idx ? (int64_t)idx[base + r] : base + r;
      rows[r * ld + c] = src >= 0 ? feats[src * dim + c] : 0.f;
    }
    __syncthreads();
    if ((int)threadIdx.x < nt) {
      const float* x = rows + threadIdx.x * ld;
      const int64_t row = base + threadIdx.x;
      const bool pad = idx && idx[row] < 0;
      float* o = out + row * out_stride;
      for (int k0 = 0; k0 < Kstore; k0 += 8) {
        double a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
        for (int i = 0; i < dim; ++i) {
          const double xi = (double)x[i];
          const double* pv = pat + ((int64_t)(k0 / 8) * dim + i) * 8;
          const double wi = kW ? w[i] : 1.0;
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            const double d = xi - pv[c];
            a[c] = fma(kW ? wi * d : d, d, a[c]);
          }
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const int k = k0 + c;
          if (k < Kstore) o[k] = pad ? INFINITY : k < K ? (float)sqrt(a[c]) : 0.f;
        }
      }
    }
  }
}

// FP64 matrix cores (v_mfma_f64_16x16x4f64), GEMM form: d^2 = |x|^2 + |p|^2 - 2 x.p with the weights folded in
// (x.p -> sum w x p, |x|^2 -> sum w x^2, |p|^2 -> sum w p^2).  One wave takes 16 feature rows at a time and forms
// D = C + A B with the patterns as A (16 pattern columns by 4 features per instruction, scaled by -2) and the rows as
// B (4 features by 16 rows), accumulating from C = |x|^2 + |p|^2, so D is d^2 itself.  The operand k index is
// permuted so that each lane's B fragment is one contiguous chunk of its row: lane l = j + 16 kk holds row j's
// features [kk D4, (kk + 1) D4), and step s of the product takes feature kk D4 + s from both operands (the sum over k
// is order-free in exact arithmetic and the accumulation is FP64).  Register r of lane l holds D[4 r + l / 16][l % 16]:
// A row m = 4 r + g is staged as pattern column 4 g + r of its tile, so lane j + 16 g ends with four consecutive
// columns 4 g .. 4 g + 3 of its own row j.  Its |x|^2, row id and output address are then its own (no lane
// exchange), and the four distances leave as one 16-byte store.  Pairs with d^2 below 2^-10 (|x|^2 + |p|^2) (with
// the largest |p|^2 of the lane's four columns, a superset) lose digits to cancellation and are recomputed directly
// as sum w (x - p)^2 in FP64, so the result keeps the direct form's accuracy (relative error of d^2 below 1e-11
// elsewhere).
typedef double d4v __attribute__((ext_vector_type(4)));

// Pattern column of MFMA row m within a tile (and the reverse: the map is its own inverse).
__device__ __forceinline__ int mfma_col(int m) { return 4 * (m & 3) + (m >> 2); }

// LDS position of pattern operand e = c * 4 D4 + d (pattern column c = 16 pt + mfma_col(m), feature d = D4 kk + s2):
// the layout [pt][s2][kk][m], so that product step s2 of tile pt reads 64 consecutive doubles across the wave (lane
// 16 kk + m), one conflict-free LDS access.  In the natural [column][feature] layout the 64 lanes' operands lie 128 or 512
// bytes apart, all in one bank pair, and each access is serialised.
__device__ __forceinline__ int lds_operand(int e, int D4) {
  const int c = e / (4 * D4), d = e - c * (4 * D4);
  const int pt = c >> 4, m = mfma_col(c & 15), kk = d / D4, s2 = d - kk * D4;
  return ((pt * D4 + s2) * 4 + kk) * 16 + m;
}

// Correctly rounded square root of x >= 0 in FP32 (x >= 2^-104): the hardware root corrected by sqrt_rn_fix, eight
// VALU instructions against the library's general sequence.
__device__ __forceinline__ float sqrt_rn(float x) { return sqrt_rn_fix(x, __builtin_amdgcn_sqrtf(x)); }

// Up to 64 features the kernel fits three waves per SIMD (at most 168 registers), which keeps the matrix core busy
// while other waves run their epilogues and loads; wider rows keep the whole register file.  kW: weighted metric (a
// template parameter, so the unweighted loop carries no per-feature select).  kVec: the row width is exactly 4 D4
// (e.g. 32 or 64 features), so each lane's 16-float chunk loads as float4s with no feature past dim; otherwise each
// feature loads on its own at a clamped index (a separate instantiation, whose per-lane offsets would otherwise
// occupy registers in the float4 loop too).
template <int D4, bool kIdx, bool kW, bool kVec>
__global__ __launch_bounds__(256, D4 <= 16 ? 3 : 1) void k_cdist_mfma(int64_t nrows, const int* __restrict__ idx,
                                                    const float* __restrict__ feats, int dim,
                                                    const double* __restrict__ w, const double* __restrict__ pat,
                                                    int K, int Kstore, float* __restrict__ out, int out_stride) {
  // LDS: npt * 16 * 4 D4 pattern operands -2 w_d p_c[d] (zero past dim and past K, laid out by lds_operand; the factor is
  // exact), [4 D4] weights, [npt * 16] pattern norms sum_d w_d p_c[d]^2.  Every block forms them from the pattern's
  // features: a kernel of their own took 5-25 us before each distance launch.
  extern __shared__ double bsh[];
  const int lane = threadIdx.x & 63, i = lane & 15, kk = lane >> 4;
  const int64_t nw = (int64_t)gridDim.x * 4, step = nw * 16;
  const int npt = (Kstore + 15) / 16;
  double* wsh = bsh + npt * 16 * 4 * D4;
  double* psh = wsh + 4 * D4;
  const int K8 = (K + 7) / 8 * 8;  // columns of pat
  if (dim < 4 * D4 || K8 < npt * 16) {
    for (int e = threadIdx.x; e < npt * 16 * 4 * D4; e += 256) bsh[e] = 0.0;
    __syncthreads();
  }
  for (int e = threadIdx.x; e < K8 * dim; e += 256) {  // in the order of pat
    const int cd = e >> 3, cg = cd / dim, d = cd - cg * dim, c = 8 * cg + (e & 7);
    const double pv = pat[e];
    bsh[lds_operand(c * 4 * D4 + d, D4)] = -2.0 * (kW ? w[d] * pv : pv);
  }
  if (kW)
    for (int d = threadIdx.x; d < 4 * D4; d += 256) wsh[d] = d < dim ? w[d] : 0.0;
  // Norms: a wave per 16 columns, four lanes to a column.
  for (int pt = threadIdx.x >> 6; pt < npt; pt += 4) {
    const int c = 16 * pt + i;
    double s = 0.0;
    if (c < K)
      for (int d = kk; d < dim; d += 4) {
        const double pv = pat[((int64_t)(c >> 3) * dim + d) * 8 + (c & 7)];
        s = fma(kW ? w[d] * pv : pv, pv, s);
      }
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if (kk == 0) psh[c] = s;
  }
  __syncthreads();
  // Without kVec the features past dim are zeroed at conversion (lim of this lane's chunk exist).  Rows that do not
  // exist are not zeroed: their loads read row 0 and their outputs are +inf regardless.
  static_assert(D4 % 4 == 0, "chunks of whole float4s");
  constexpr bool vec = kVec;
  const int lim = dim - kk * D4;
  // Four columns leave as one 16-byte store when every group of four starts a 16-byte aligned address.
  const bool vst = (Kstore & 3) == 0 && (out_stride & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  // Feature row of lane row i in the tile at r (-1: past the end or a padding row), in two steps so that the id load
  // stays in flight: row_raw loads idx at a valid (clamped) row, row_of interprets the loaded value later.
  auto row_raw = [&](int64_t r) -> int {
    const int64_t row = r + i;
    return kIdx ? idx[row < nrows ? row : nrows - 1] : 0;
  };
  auto row_of = [&](int64_t r, int raw) -> int64_t {
    const int64_t row = r + i;
    return row < nrows ? (kIdx ? (int64_t)raw : row) : -1;
  };
  // This lane's chunk [kk D4, (kk + 1) D4) of row src as raw floats.  Every load has a valid address (row 0 for
  // src < 0, the last feature past dim) and no lane's register is written twice, so the loads stay in flight until
  // the values are converted.
  auto load_x = [&](int64_t src, float* x) {
    const float* xs = feats + (src >= 0 ? src : 0) * dim;
    if constexpr (vec) {
      const f4v* x4 = reinterpret_cast<const f4v*>(xs + kk * D4);
#pragma unroll
      for (int u = 0; u < D4 / 4; ++u) {
        const f4v v = x4[u];
#pragma unroll
        for (int c = 0; c < 4; ++c) x[4 * u + c] = v[c];
      }
    } else {
#pragma unroll
      for (int s2 = 0; s2 < D4; ++s2) {
        const int d = kk * D4 + s2;
        x[s2] = xs[d < dim ? d : dim - 1];
      }
    }
  };
  auto convert = [&](const float* x, double* a) {
    if constexpr (vec) {
#pragma unroll
      for (int s2 = 0; s2 < D4; ++s2) a[s2] = (double)x[s2];
    } else {
#pragma unroll
      for (int s2 = 0; s2 < D4; ++s2) a[s2] = s2 < lim ? (double)x[s2] : 0.0;
    }
  };
  // d^2 of feature row src against pattern column c, directly in FP64 (the cancellation fallback).
  auto direct = [&](int64_t src, int c) -> double {
    const float* xs = feats + src * dim;
    double d2 = 0.0;
    for (int d = 0; d < dim; ++d) {
      const double e = (double)xs[d] - pat[((int64_t)(c / 8) * dim + d) * 8 + c % 8];
      d2 = fma(kW ? w[d] * e : e, e, d2);
    }
    return d2;
  };
  // The next tile's features are in flight (raw floats) during this tile's products and are converted at the end of
  // the iteration; its row ids are loaded a tile earlier still, so that its gather issues at once.
  float xr[D4];
  double a[D4];
  int64_t r0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
  int64_t src = -1, srcn = -1;
  if (r0 < nrows) {
    src = row_of(r0, row_raw(r0));
    srcn = row_of(r0 + step, row_raw(r0 + step));
    load_x(src, xr);
    convert(xr, a);
  }
  for (; r0 < nrows; r0 += step) {
    const bool more = r0 + step < nrows;
    if (more) load_x(srcn, xr);
    const int rawnn = row_raw(r0 + 2 * step);
    double xx = 0.0;
#pragma unroll
    for (int s2 = 0; s2 < D4; ++s2) xx = fma(kW ? wsh[kk * D4 + s2] * a[s2] : a[s2], a[s2], xx);
    xx += __shfl_xor(xx, 16, 64);
    xx += __shfl_xor(xx, 32, 64);  // every lane: |x|^2 of its row i
    const bool live = src >= 0, rok = r0 + i < nrows;
    float* orow = out + (rok ? r0 + i : 0) * out_stride;
    // C = |x|^2 + |p|^2 of this lane's four columns 16 t + 4 kk + r of tile t, and the largest |p|^2 among them.
    auto init = [&](int t, d4v& acc, double& pm) {
      const double* pc = psh + t * 16 + 4 * kk;
      pm = fmax(fmax(pc[0], pc[1]), fmax(pc[2], pc[3]));
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = xx + pc[r];
    };
    // Epilogue of tile t, branch-free but for the rare cancellation: the square root in FP32 (sqrt_rn of the rounded
    // d^2, within 0.75 ulp of the distance, since FP64 VALU work here competes with the products for the same FP64
    // rate), +inf for rows that do not exist, 0 in the padding columns [K, Kstore).
    auto emit = [&](int t, const d4v& acc, double pm) {
      const int cb = t * 16 + 4 * kk;
      const double thr = 0x1p-10 * (xx + pm);
      double d2[4];
      bool fix = false;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        d2[r] = acc[r];
        fix |= live && cb + r < K && d2[r] < thr;
      }
      if (__any(fix)) {  // cancellation: recompute those pairs directly
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (live && cb + r < K && d2[r] < thr) d2[r] = direct(src, cb + r);
      }
      // The root is taken unconditionally (of 0 in the padding columns and rows that do not exist), so no lane
      // branches around it.
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float s = sqrt_rn(live && cb + r < K ? (float)d2[r] : 0.f);
        v[r] = live ? s : INFINITY;
      }
      if (vst) {
        if (rok && cb < Kstore) *reinterpret_cast<f4v*>(orow + cb) = f4v{v[0], v[1], v[2], v[3]};
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (rok && cb + r < Kstore) orow[cb + r] = v[r];
      }
    };
    // Pattern tiles in pairs: two independent accumulator chains interleave on the matrix core.
    for (int pt = 0; pt < npt; pt += 2) {
      const double* bp0 = bsh + (pt * D4 * 4 + kk) * 16 + i;
      d4v acc0, acc1;
      double pm0, pm1;
      init(pt, acc0, pm0);
      if (pt + 1 < npt) {
        const double* bp1 = bp0 + D4 * 64;
        init(pt + 1, acc1, pm1);
#pragma unroll
        for (int s2 = 0; s2 < D4; ++s2) {
          acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(bp0[s2 * 64], a[s2], acc0, 0, 0, 0);
          acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(bp1[s2 * 64], a[s2], acc1, 0, 0, 0);
        }
        emit(pt, acc0, pm0);
        emit(pt + 1, acc1, pm1);
      } else {
#pragma unroll
        for (int s2 = 0; s2 < D4; ++s2) acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(bp0[s2 * 64], a[s2], acc0, 0, 0, 0);
        emit(pt, acc0, pm0);
      }
    }
    if (more) convert(xr, a);
    // An empty register barrier: the loaded id is first read here, so its load stays in flight until now.
    int raw = rawnn;
    if (kIdx) asm volatile("" : "+v"(raw));
    src = srcn;
    srcn = row_of(r0 + 2 * step, raw);
  }
}

int cdist_mfma_d4(int dim) {
  if (dim <= 16) return 4;
  if (dim <= 32) return 8;
  if (dim <= 64) return 16;
  if (dim <= 128) return 32;
  return 0;
}

// Fallback for feature widths too large to stage: one thread per output element, rows read from global memory.
__global__ void k_cdist_direct(int64_t nrows, const int* __restrict__ idx, const float* __restrict__ feats, int dim,
                               const double* __restrict__ pat, int K, int Kp, int Kstore, float* __restrict__ out,
                               int out_stride, const double* __restrict__ w) {
  const int64_t total = nrows * Kstore;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = e / Kstore;
    const int k = (int)(e - r * Kstore);
    const int64_t src = idx ? (int64_t)idx[r] : r;
    const float* x = feats + src * dim;
    double a = 0.0;
    if (k < K && src >= 0)
      for (int i = 0; i < dim; ++i) {
        const double d = (double)x[i] - pat[((int64_t)(k / 8) * dim + i) * 8 + k % 8];
        a = fma(w ? w[i] * d : d, d, a);
      }
    out[r * out_stride + k] = src < 0 ? INFINITY : k < K ? (float)sqrt(a) : 0.f;
  }
}

void launch_cdist(int64_t nrows, const int* idx, const float* feats, int dim, const double* pat, int K, int Kp,
                  int Kstore, float* out, int out_stride, const double* w, bool mfma, hipStream_t st) {
  if (nrows == 0 || Kstore == 0) return;
  const int D4 = cdist_mfma_d4(dim);
  // The pattern operands, weights and norms are staged in LDS: up to 64 KB.
  if (mfma && D4 && dim > 0 &&
      ((size_t)((Kstore + 15) / 16 * 16 + 1) * 4 * D4 + (Kstore + 15) / 16 * 16) * sizeof(double) <= 65536) {
    const int Kp16 = (Kstore + 15) / 16 * 16;
    // Three blocks a CU, resident at once, so that the operands are formed once per CU slot (the prep of R-MAT 20 with 24
    // columns of 64 features, and of R-MAT 16 slabs with 128 columns: 3.62 ms and 819 us at 8192 blocks, 3.75 / 767 at
    // 3072, 3.59 / 761 at 1024, 3.48 / 786 at 768).
    const int blocks = (int)std::min<int64_t>((nrows + 63) / 64, 768);
    const size_t lds = ((size_t)(Kp16 + 1) * 4 * D4 + Kp16) * sizeof(double);  // operands, weights, norms
#define AC_CD_MFMA_V(N, V)                                                                                        \
  if (idx && w)                                                                                                   \
    hipLaunchKernelGGL((k_cdist_mfma<N, true, true, V>), dim3(blocks), dim3(256), lds, st, nrows, idx, feats, dim, \
                       w, pat, K, Kstore, out, out_stride);                                             \
  else if (idx)                                                                                                   \
    hipLaunchKernelGGL((k_cdist_mfma<N, true, false, V>), dim3(blocks), dim3(256), lds, st, nrows, idx, feats,     \
                       dim, w, pat, K, Kstore, out, out_stride);                                        \
  else if (w)                                                                                                     \
    hipLaunchKernelGGL((k_cdist_mfma<N, false, true, V>), dim3(blocks), dim3(256), lds, st, nrows, idx, feats,     \
                       dim, w, pat, K, Kstore, out, out_stride);                                        \
  else                                                                                                            \
    hipLaunchKernelGGL((k_cdist_mfma<N, false, false, V>), dim3(blocks), dim3(256), lds, st, nrows, idx, feats,    \
                       dim, w, pat, K, Kstore, out, out_stride);
#define AC_CD_MFMA(N)                \
  case N:                            \
    if (dim == 4 * N) {              \
      AC_CD_MFMA_V(N, true)          \
    } else {                         \
      AC_CD_MFMA_V(N, false)         \
    }                                \
    return;
    switch (D4) {
      AC_CD_MFMA(4)
      AC_CD_MFMA(8)
      AC_CD_MFMA(16)
      AC_CD_MFMA(32)
      default:
        break;
    }
#undef AC_CD_MFMA
#undef AC_CD_MFMA_V
  }
  if (dim <= 255) {
    // At most 64 KB of LDS: 128 rows up to 127 features, fewer rows beyond.
    const int tile = std::min(kCdTile, 16384 / (dim + 1));
    const size_t lds = (size_t)tile * (dim + 1) * sizeof(float);
    const int blocks = (int)std::min<int64_t>((nrows + tile - 1) / tile, 1 << 16);
    if (w)
      hipLaunchKernelGGL(k_cdist_rows<true>, dim3(blocks), dim3(kCdTile), lds, st, nrows, idx, feats, dim, pat, K,
                         Kp, Kstore, out, out_stride, tile, w);
    else
      hipLaunchKernelGGL(k_cdist_rows<false>, dim3(blocks), dim3(kCdTile), lds, st, nrows, idx, feats, dim, pat, K,
                         Kp, Kstore, out, out_stride, tile, w);
  } else {
    const int blocks = (int)std::min<int64_t>((nrows * Kstore + 255) / 256, 1 << 16);
    hipLaunchKernelGGL(k_cdist_direct, dim3(blocks), dim3(256), 0, st, nrows, idx, feats, dim, pat, K, Kp, Kstore,
                       out, out_stride, w);
  }
}

// Merge of a block's per-thread accumulators by column: thread t holds s of column t % C, C <= NT, threads
// t >= rows * C none.  Thread c < C gets column c's, its rows summed in order.  sh: (rows + 1) * C doubles.
__device__ __forceinline__ Lse block_columns_lse(const Lse& s, int C, int rows, double* sh) {
  const int t = threadIdx.x;
  const bool active = t < rows * C;
  if (active) sh[t] = s.m;
  __syncthreads();
  Lse acc = lse_empty();
  if (t < C) {
    for (int r = 0; r < rows; ++r) acc.m = fmax(acc.m, sh[r * C + t]);
    sh[rows * C + t] = acc.m;
  }
  __syncthreads();
  const double x = active ? lse_rescaled(s, sh[rows * C + t % C]) : 0.0;
  if (active) sh[t] = x;
  __syncthreads();
  if (t < C) {
    bool seen = false;
    for (int r = 0; r < rows; ++r) lse_sum_step(acc.t, seen, sh[r * C + t]);
  }
  return acc;
}

// ---------------------------------------------------------------------------------------------------------------
// Column log-sum-exp of -X over the n rows of X[n][P] (the prep's LSM(-CV) normaliser, src/main.cu:117).

__global__ __launch_bounds__(256) void k_col_lse_neg(int64_t n, int P, const float* __restrict__ X,
                                                     Lse* __restrict__ part) {
  __shared__ double red[512];
  const int t = threadIdx.x;
  const int RP = 256 / P;
  const bool active = t < RP * P;
  const int p = active ? t % P : 0;
  Lse acc = lse_empty();
  if (active)
    for (int64_t v = (int64_t)blockIdx.x * RP + t / P; v < n; v += (int64_t)gridDim.x * RP)
      lse_add(acc, -(double)X[v * P + p]);
  const Lse s = block_columns_lse(acc, P, RP, red);
  if (t < P) part[(int64_t)t * gridDim.x + blockIdx.x] = s;
}

void launch_col_lse_neg(int64_t n, int P, const float* X, Lse* part, int nblocks, hipStream_t st) {
  hipLaunchKernelGGL(k_col_lse_neg, dim3(nblocks), dim3(256), 0, st, n, P, X, part);
}

// Partials a thread of a fixed-order reduction holds in registers, all loaded at once: kRed* x 256 partials take one
// memory round trip and one exponential each.  Further ones are merged into them one by one.  Slots past the last
// partial load the last partial (an in-bounds address) and then hold the empty one.
constexpr int kRedLse = 8, kRedQ = 5;

// Reduce per-block partials [ncol][nparts] column by column in a fixed order (deterministic).  (A column's partials lie
// together: by block, [nparts][ncol], every partial of a column was a line of its own.)
__global__ __launch_bounds__(256) void k_reduce_lse(int nparts, const Lse* __restrict__ part, Lse2* __restrict__ out,
                                                    Lse2* __restrict__ out2) {
  __shared__ double red[8];
  const int c = blockIdx.x, t = threadIdx.x;
  Lse v[kRedLse];
#pragma unroll
  for (int u = 0; u < kRedLse; ++u) {
    v[u] = lse_empty();
    if (u * 256 >= nparts) continue;  // (the same for the whole block)
    const int b = t + u * 256;
    const Lse x = part[(int64_t)c * nparts + (b < nparts ? b : nparts - 1)];
    if (b < nparts) v[u] = x;
  }
  for (int b0 = 256 * kRedLse + t; b0 < nparts; b0 += 256 * kRedLse) {
    Lse w[kRedLse];
#pragma unroll
    for (int u = 0; u < kRedLse; ++u) {
      const int b = b0 + u * 256;
      w[u] = part[(int64_t)c * nparts + (b < nparts ? b : nparts - 1)];
    }
#pragma unroll
    for (int u = 0; u < kRedLse; ++u)
      if (b0 + u * 256 < nparts) v[u] = lse_merge(v[u], w[u]);
  }
  double m = v[0].m;
#pragma unroll
  for (int u = 1; u < kRedLse; ++u) m = fmax(m, v[u].m);
  const double M = block_max<256>(m, red);
  double sum = 0.0;
  bool seen = false;
#pragma unroll
  for (int u = 0; u < kRedLse; ++u)
    if (u * 256 < nparts) lse_sum_step(sum, seen, lse_rescaled(v[u], M));
  sum = block_lse_sum<256>(sum, seen, red);
  if (t == 0) {
    out[c] = Lse2{M, log1p(sum)};
    if (out2) out2[c] = Lse2{M, log1p(sum)};
  }
}

void launch_reduce_lse(int nparts, int ncol, const Lse* part, Lse2* out, hipStream_t st, Lse2* out2) {
  if (ncol == 0) return;
  hipLaunchKernelGGL(k_reduce_lse, dim3(ncol), dim3(256), 0, st, nparts, part, out, out2);
}

// FMaxN rows of the split vertices to -inf, over nblocks blocks: the walk's pieces of a split vertex then raise its row
// with atomic maxima.
__device__ __forceinline__ void reset_split_rows(int block, int nblocks, int nsplit, const Split* __restrict__ splits,
                                                 int Qs, float* __restrict__ FMaxN) {
  const int L4 = Qs / 4;
  const int64_t total = (int64_t)nsplit * L4;
  for (int64_t i = (int64_t)block * blockDim.x + threadIdx.x; i < total; i += (int64_t)nblocks * blockDim.x) {
    const int s = (int)(i / L4), j = (int)(i - (int64_t)s * L4);
    reinterpret_cast<f4v*>(FMaxN)[(int64_t)splits[s].v * L4 + j] = f4v{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  }
}

// Blocks that reset nsplit rows: four 16-byte stores a thread, at most 256 blocks.
static int reset_blocks(int nsplit, int Qs) {
  return (int)std::min<int64_t>(256, ((int64_t)nsplit * (Qs / 4) + 1023) / 1024);
}

// cnull != nullptr: the iteration's fills are lowered by the PNNL Cnull term, fillF = max VR - cnull[q] and
// fillR = max VF - cnull[q] (test.py:148-149; cnull <= 0, so the fills rise and the pruning bound below, which assumes
// the unraised fill, stays valid).
// Four groups of 256 threads, one for each of RE's log-sum-exp, FE's, max VF and max VR, side by side (one group taking
// them in turn, partials of a column a line each: 7.4-12 us; now 5.2-7.3 us).
__global__ __launch_bounds__(1024) void k_reduce_q(int nparts, int Q, const QPart* __restrict__ part,
                                                   const double* __restrict__ cnull, QStat* __restrict__ out,
                                                   SplitRows rows) {
  if ((int)blockIdx.x >= Q) {  // the blocks after the Q reducing ones
    reset_split_rows(blockIdx.x - Q, gridDim.x - Q, rows.nsplit, rows.splits, rows.Qs, rows.FMaxN);
    return;
  }
  __shared__ double sm[4][4], ss[4][4];
  __shared__ int sa[4][4];
  const int q = blockIdx.x, t = threadIdx.x & 255, lane = t & 63, w = t >> 6;
  const int job = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  double m = -kInf, sum = 0.0;
  int arg = -1;
  bool seen = false;
  const QPart* pq = part + (int64_t)q * nparts;
  if (job < 2) {
    Lse v[kRedQ];
#pragma unroll
    for (int u = 0; u < kRedQ; ++u) {
      v[u] = lse_empty();
      if (u * 256 >= nparts) continue;  // (the same for the whole block)
      const int b = t + u * 256;
      const QPart* p = pq + (b < nparts ? b : nparts - 1);
      const Lse x = job == 0 ? p->re : p->fe;
      if (b < nparts) v[u] = x;
    }
    for (int b0 = 256 * kRedQ + t; b0 < nparts; b0 += 256 * kRedQ)
#pragma unroll
      for (int u = 0; u < kRedQ; ++u) {
        const int b = b0 + u * 256;
        if (b < nparts) v[u] = lse_merge(v[u], job == 0 ? pq[b].re : pq[b].fe);
      }
#pragma unroll
    for (int u = 0; u < kRedQ; ++u) m = fmax(m, v[u].m);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if (lane == 0) sm[job][w] = m;
    __syncthreads();
    m = fmax(fmax(sm[job][0], sm[job][1]), fmax(sm[job][2], sm[job][3]));
#pragma unroll
    for (int u = 0; u < kRedQ; ++u)
      if (u * 256 < nparts) lse_sum_step(sum, seen, lse_rescaled(v[u], m));
    const unsigned long long holders = __ballot(seen);
    if (seen && lane != __ffsll((long long)holders) - 1) sum += 1.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if (lane == 0) {
      ss[job][w] = sum;
      sa[job][w] = holders != 0;
    }
  } else {
    for (int b0 = t; b0 < nparts; b0 += 256 * kRedQ) {
      double x[kRedQ];
      int a[kRedQ];
#pragma unroll
      for (int u = 0; u < kRedQ; ++u) {
        const int b = b0 + u * 256;
        const QPart* p = pq + (b < nparts ? b : nparts - 1);  // (past the end: the last one again)
        x[u] = job == 2 ? p->vfmax : p->vrmax;
        a[u] = job == 2 ? p->avf : p->avr;
      }
#pragma unroll
      for (int u = 0; u < kRedQ; ++u) argmax_merge(m, arg, x[u], a[u]);
    }
    // Ties: the lowest vertex, in any order.
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) argmax_merge(m, arg, __shfl_xor(m, o, 64), __shfl_xor(arg, o, 64));
    if (lane == 0) {
      sm[job][w] = m;
      sa[job][w] = arg;
    }
    __syncthreads();
  }
  __syncthreads();
  if (t == 0) {
    if (job < 2) {
      sum = ss[job][0];
      bool any = sa[job][0] != 0;
      for (int i = 1; i < 4; ++i) {
        sum += ss[job][i];
        if (sa[job][i]) {
          if (any) sum += 1.0;
          any = true;
        }
      }
      ss[job][0] = sum;
      sm[job][1] = log1p(sum);
    } else {
      for (int i = 1; i < 4; ++i) argmax_merge(m, arg, sm[job][i], sa[job][i]);
      sa[job][0] = arg;
    }
    sm[job][0] = m;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const double vfmax = sm[2][0], vrmax = sm[3][0];
    // Edge pruning bound.  An edge term is (VR[src] - CE) - LSE_FE with VR[src] <= fillF (rounded to FP32 once),
    // so it cannot exceed fillF when CE + LSE_FE >= 2^-22 (|fillF| + |CE| + |LSE_FE|); cthr = -LSE_FE plus four
    // times that margin (a cost near the bound has |CE| ~ |LSE_FE|; a larger one clears it by itself).
    const double fF = vrmax, sl = sm[1][0] + sm[1][1];
    double cthr = kInf;
    if (fF > -kInf && fF < kInf && sl > -kInf && sl < kInf)
      cthr = -sl + 0x1p-20 * (fabs(fF) + 2.0 * fabs(sl) + 1.0);
    const double fillF = cnull ? vrmax - cnull[q] : vrmax, fillR = cnull ? vfmax - cnull[q] : vfmax;
    out[q] = QStat{fillF, fillR, sm[0][0], sm[0][1], sm[1][0], sm[1][1], sa[3][0], sa[2][0], cthr};
  }
}

void launch_reduce_q(int nparts, int Q, const QPart* part, QStat* out, hipStream_t st, const double* cnull,
                     const SplitRows& rows) {
  if (Q == 0) return;
  hipLaunchKernelGGL(k_reduce_q, dim3(Q + reset_blocks(rows.nsplit, rows.Qs)), dim3(1024), 0, st, nparts, Q, part, cnull,
                     out, rows);
}

// Isolated-vertex columns: one pass over X[n][P] giving per-block partials of LSE(-X) and of (min X, lowest row).
__global__ __launch_bounds__(256) void k_iso_cols(int64_t n, int P, const float* __restrict__ X, Lse* __restrict__ lpart,
                                                  float* __restrict__ pv, int* __restrict__ pi) {
  __shared__ double red[512];
  __shared__ float rv[256];
  __shared__ int ri[256];
  const int t = threadIdx.x, RP = 256 / P;
  const bool active = t < RP * P;
  const int p = active ? t % P : 0;
  Lse acc = lse_empty();
  float best = INFINITY;
  int bi = INT_MAX;
  if (active)
    for (int64_t v = (int64_t)blockIdx.x * RP + t / P; v < n; v += (int64_t)gridDim.x * RP) {
      const float x = X[v * P + p];
      lse_add(acc, -(double)x);
      if (x < best) {  // rows ascend within a thread
        best = x;
        bi = (int)v;
      }
    }
  rv[t] = best;
  ri[t] = bi;
  const Lse s = block_columns_lse(acc, P, RP, red);
  if (t < P) {
    for (int r = 0; r < RP; ++r) {
      const float x = rv[r * P + t];
      const int xi = ri[r * P + t];
      if (x < best || (x == best && xi < bi)) {
        best = x;
        bi = xi;
      }
    }
    lpart[(int64_t)blockIdx.x * P + t] = s;
    pv[(int64_t)blockIdx.x * P + t] = best;
    pi[(int64_t)blockIdx.x * P + t] = bi;
  }
}

// One block per column: partials merged by a fixed tree (the minimum's lowest row wins ties in any order).
__global__ __launch_bounds__(256) void k_iso_final(int nparts, int P, int base, const Lse* __restrict__ lpart,
                                                   const float* __restrict__ pv, const int* __restrict__ pi,
                                                   IsoCol* __restrict__ out) {
  __shared__ double rs[8];
  __shared__ float rv[256];
  __shared__ int ri[256];
  const int p = blockIdx.x, t = threadIdx.x;
  Lse s = lse_empty();
  float best = INFINITY;
  int bi = INT_MAX;
  for (int b = t; b < nparts; b += 256) {
    s = lse_merge(s, lpart[(int64_t)b * P + p]);
    const float x = pv[(int64_t)b * P + p];
    const int xi = pi[(int64_t)b * P + p];
    if (x < best || (x == best && xi < bi)) {
      best = x;
      bi = xi;
    }
  }
  rv[t] = best;
  ri[t] = bi;
  const double M = block_max<256>(s.m, rs);
  double sum = 0.0;
  bool seen = false;
  lse_sum_step(sum, seen, lse_rescaled(s, M));
  sum = block_lse_sum<256>(sum, seen, rs);
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w) {
      if (rv[t + w] < rv[t] || (rv[t + w] == rv[t] && ri[t + w] < ri[t])) {
        rv[t] = rv[t + w];
        ri[t] = ri[t + w];
      }
    }
    __syncthreads();
  }
  // A column whose isolated costs are all +inf has no finite share: treat it as empty.
  if (t == 0)
    out[p] = ri[0] == INT_MAX ? IsoCol{-kInf, 0.0, INFINITY, -1} : IsoCol{M, sum, rv[0], base + ri[0]};
}

void launch_iso_cols(int64_t n, int P, const float* X, int base, Lse* lpart, float* pv, int* pi, int nparts,
                     IsoCol* out, hipStream_t st) {
  if (P == 0) return;
  hipLaunchKernelGGL(k_iso_cols, dim3(nparts), dim3(256), 0, st, n, P, X, lpart, pv, pi);
  hipLaunchKernelGGL(k_iso_final, dim3(P), dim3(256), 0, st, nparts, P, base, lpart, pv, pi, out);
}

// Scalars of the prep state (src/main.cu:116-146): MU0 = LSM(-CV), RE0 = FE0 = LSM(-CE).  The column maximum of
// MU0 sits at the minimum cost, where (x - m) = 0, so max_v MU0[v][p] = -log1p(t_p).
__global__ void k_prep_scalars(int Q, const int* __restrict__ ps, const int* __restrict__ pd,
                               const Lse2* __restrict__ cv, const Lse2* __restrict__ ce, QStat* __restrict__ qs,
                               SplitRows rows) {
  if (blockIdx.x > 0) {
    reset_split_rows(blockIdx.x - 1, gridDim.x - 1, rows.nsplit, rows.splits, rows.Qs, rows.FMaxN);
    return;
  }
  const int q = threadIdx.x;  // Q <= 256
  if (q >= Q) return;
  qs[q] = QStat{-cv[ps[q]].l, -cv[pd[q]].l, ce[q].m, ce[q].l, ce[q].m, ce[q].l, -1, -1, kInf};
}

void launch_prep_scalars(int P, int Q, const int* ps, const int* pd, const Lse2* cv, const Lse2* ce, QStat* qs,
                         hipStream_t st, const SplitRows& rows) {
  (void)P;
  if (Q == 0) return;
  hipLaunchKernelGGL(k_prep_scalars, dim3(1 + reset_blocks(rows.nsplit, rows.Qs)), dim3(256), 0, st, Q, ps, pd, cv, ce,
                     qs, rows);
}

// The constant rows of the per-vertex arrays [n][w], in one launch: rows [a0, a1) and [b0, n) of minC (+inf), ls (0) and
// vfm (-inf), rows [f0, n) of fmaxn (-inf).
__global__ void k_fill_const(int64_t n, int w, int64_t a0, int64_t a1, int64_t b0, int64_t f0, float* __restrict__ minC,
                             float* __restrict__ ls, float* __restrict__ vfm, float* __restrict__ fmaxn) {
  const int64_t la = (a1 - a0) * w, lo = la + (n - b0) * w, total = lo + (n - f0) * w;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    if (i < lo) {
      const int64_t o = i < la ? a0 * w + i : b0 * w + (i - la);
      minC[o] = INFINITY;
      ls[o] = 0.f;
      vfm[o] = -INFINITY;
    } else {
      fmaxn[f0 * w + (i - lo)] = -INFINITY;
    }
  }
}

void launch_fill_const(int64_t n, int w, int64_t a0, int64_t a1, int64_t b0, int64_t f0, float* minC, float* ls,
                       float* vfm, float* fmaxn, hipStream_t st) {
  const int64_t total = ((a1 - a0) + (n - b0) + (n - f0)) * w;
  if (total == 0) return;
  const int blocks = (int)std::min<int64_t>((total + 1023) / 1024, 1 << 14);
  hipLaunchKernelGGL(k_fill_const, dim3(blocks), dim3(256), 0, st, n, w, a0, a1, b0, f0, minC, ls, vfm, fmaxn);
}

// -inf into three ranges of each of nslots slots (stride `stride`): [a0, a0 + al) of A, and [b0, b0 + bl) and [c0, c0 + cl)
// of B, in units of four floats.  One launch for every slot; bound by the stores (13 slots at R-MAT 18 with 16 pattern
// edges: 47 us a float at a time, 27 now).
__global__ __launch_bounds__(256) void k_fill_slots(f4v* __restrict__ A, f4v* __restrict__ B, int64_t stride, int64_t a0,
                                                    int64_t al, int64_t b0, int64_t bl, int64_t c0, int64_t cl) {
  const f4v x = f4v{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  const int64_t per = al + bl + cl, s = blockIdx.y;
  for (int64_t r = blockIdx.x * (int64_t)256 + threadIdx.x; r < per; r += (int64_t)gridDim.x * 256)
    if (r < al)
      A[s * stride + a0 + r] = x;
    else if (r < al + bl)
      B[s * stride + b0 + (r - al)] = x;
    else
      B[s * stride + c0 + (r - al - bl)] = x;
}

void launch_fill_slots(float* A, float* B, int nslots, int w, int64_t stride, int64_t a0, int64_t al, int64_t b0, int64_t bl,
                       int64_t c0, int64_t cl, hipStream_t st) {
  const int64_t w4 = w / 4, per = (al + bl + cl) * w4;
  if (per == 0 || nslots == 0) return;
  for (int s0 = 0; s0 < nslots; s0 += 32768) {  // (the grid's second dimension)
    const dim3 grid((unsigned)std::min<int64_t>((per + 1023) / 1024, 4096), (unsigned)std::min(nslots - s0, 32768));
    hipLaunchKernelGGL(k_fill_slots, grid, dim3(256), 0, st, reinterpret_cast<f4v*>(A) + s0 * stride * w4,
                       reinterpret_cast<f4v*>(B) + s0 * stride * w4, stride * w4, a0 * w4, al * w4, b0 * w4, bl * w4,
                       c0 * w4, cl * w4);
  }
}

// Zeros into several buffers at once (16-byte aligned, whole 4-byte words): a row of blocks per buffer.  The eight buffers
// of a step back at R-MAT 18 take 56 us, at 1,000 vertices 2.9 (a fill each: 77 and 18).
__global__ __launch_bounds__(256) void k_zero(ZeroList z) {
  unsigned* p = z.p[blockIdx.y];
  const int64_t n = z.words[blockIdx.y], n4 = n / 4;
  const int64_t i0 = blockIdx.x * (int64_t)256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  for (int64_t i = i0; i < n4; i += step) reinterpret_cast<uint4*>(p)[i] = make_uint4(0u, 0u, 0u, 0u);
  if (i0 < n - 4 * n4) p[4 * n4 + i0] = 0u;
}

void launch_zero(const ZeroList& z, hipStream_t st) {
  int64_t most = 0;
  for (int i = 0; i < z.count; ++i) most = std::max(most, z.words[i]);
  if (most == 0) return;
  hipLaunchKernelGGL(k_zero, dim3((unsigned)std::min<int64_t>((most + 4095) / 4096, 8192), (unsigned)z.count), dim3(256), 0,
                     st, z);
}

// ---------------------------------------------------------------------------------------------------------------
// Edge walks.  A group of Qs/4 lanes walks one run of consecutive edges; lane j owns pattern edges 4j..4j+3 and
// reads them as one float4 of the edge's cost row (and of the gathered VR row).  Runs cover whole vertices except
// the pieces of long edge lists: the source statistics' and the taped walks' partial results go to carry slots and are
// combined by a fixup kernel, a plain walk's raise the vertex's row by atomic maxima.

int walk_blocks(int64_t nruns, int Qs) {
  const int L4 = Qs / 4;
  const int G = 64 / L4;
  const int64_t per_block = (int64_t)(kWalkBlock / 64) * G;
  return (int)((nruns + per_block - 1) / per_block);
}

// Source-side statistics of the edge costs (CSR walk): for every vertex v with out-edges and every q,
//   minCEo[v][q] = min_e CE[e][q],  lsO[v][q] = log1p(sum_{other e} exp(minCEo - CE)),  VFm[v][q] = -minCEo
// (VFm of the prep state: RE0 = -CE up to a per-q constant), and per-block partials of log sum_e exp(-CE[e][q]).
// kArg: also the row of the least-cost out-edge of every (v, q), the lowest one on ties, into AO (pieces: into carg).
template <bool kArg>
__global__ __launch_bounds__(kWalkBlock) void k_walk_src(int64_t nruns, const Run* __restrict__ runs,
                                                         const int2* __restrict__ ks, const float* __restrict__ CE,
                                                         int Q, int Qs, float* __restrict__ minCEo,
                                                         float* __restrict__ lsO, float* __restrict__ VFm,
                                                         double* __restrict__ carry, Lse* __restrict__ gpart,
                                                         int* __restrict__ AO, int* __restrict__ carg) {
  __shared__ double red[kWalkBlock * 4 + 256];
  const int L4 = Qs / 4, G = 64 / L4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane / L4, j = lane - g * L4;
  const int64_t r = ((int64_t)blockIdx.x * (kWalkBlock / 64) + wave) * G + g;
  Lse glob[4] = {lse_empty(), lse_empty(), lse_empty(), lse_empty()};
  if (g < G && r < nruns) {
    const Run R = runs[r];
    // The open vertex's least cost and the sum of exp(least - cost) over its other edges.  The difference of two floats
    // rounded to FP32 is the argument of the FP32 exponential whether it is formed in FP32 or in FP64; the sum is FP64.
    float mn[4] = {INFINITY, INFINITY, INFINITY, INFINITY};
    double tt[4] = {0.0, 0.0, 0.0, 0.0};
    int ar[4] = {INT_MAX, INT_MAX, INT_MAX, INT_MAX};
    auto add = [&](int c, float x, int row) {
      if (kArg && (x < mn[c] || (x == mn[c] && row < ar[c]))) ar[c] = row;
      const float d = mn[c] - x;  // > 0: a new least cost, the old ones rescaled to it
      float e = __expf(-fabsf(d));
      e = x == INFINITY ? 0.f : e;  // (and exp(-inf) = 0 where x is the first finite cost)
      tt[c] = d > 0.f ? fma(tt[c], (double)e, (double)e) : tt[c] + (double)e;
      mn[c] = fminf(mn[c], x);
    };
    int cur = ks[R.kb].y;
    // A finished source vertex.  It runs at vertex changes, which differ between the wave's runs, so each costs the
    // whole wave: its log1p and the merge into the block partial take FP32 transcendentals (lsO is stored in FP32;
    // the merge's exponential has the precision of the sum's terms).
    auto emit = [&](int v) {
      float4 ls;
      ls.x = log1pf((float)tt[0]), ls.y = log1pf((float)tt[1]), ls.z = log1pf((float)tt[2]);
      ls.w = log1pf((float)tt[3]);
      reinterpret_cast<float4*>(minCEo)[(int64_t)v * L4 + j] = make_float4(mn[0], mn[1], mn[2], mn[3]);
      reinterpret_cast<float4*>(lsO)[(int64_t)v * L4 + j] = ls;
      reinterpret_cast<float4*>(VFm)[(int64_t)v * L4 + j] = make_float4(-mn[0], -mn[1], -mn[2], -mn[3]);
      if (kArg) reinterpret_cast<int4*>(AO)[(int64_t)v * L4 + j] = make_int4(ar[0], ar[1], ar[2], ar[3]);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        ar[c] = INT_MAX;
        glob[c] = lse_merge_fast(glob[c], Lse{-(double)mn[c], tt[c]});
        mn[c] = INFINITY;
        tt[c] = 0.0;
      }
    };
    // Steps in batches of kSrcBatch: the batch's (row, vertex) pairs, then its cost rows, are loaded together (two
    // memory round trips per batch rather than per step); the steps are then taken in order.  Slots past the run's
    // end load its last pair (a valid address) and are not taken.
    constexpr int kSrcBatch = 8;
    for (int k0 = R.kb; k0 < R.ke; k0 += kSrcBatch) {
      int2 e[kSrcBatch];
      float4 c[kSrcBatch];
#pragma unroll
      for (int u = 0; u < kSrcBatch; ++u) e[u] = ks[k0 + u < R.ke ? k0 + u : R.ke - 1];
#pragma unroll
      for (int u = 0; u < kSrcBatch; ++u) c[u] = reinterpret_cast<const float4*>(CE + ce_index(e[u].x, 4 * j, Qs))[0];
#pragma unroll
      for (int u = 0; u < kSrcBatch; ++u) {
        if (k0 + u >= R.ke) break;
        if (e[u].y != cur) {
          emit(cur);
          cur = e[u].y;
        }
        add(0, c[u].x, e[u].x);
        add(1, c[u].y, e[u].x);
        add(2, c[u].z, e[u].x);
        add(3, c[u].w, e[u].x);
      }
    }
    if (R.slot >= 0) {
      if (kArg) reinterpret_cast<int4*>(carg)[(int64_t)R.slot * L4 + j] = make_int4(ar[0], ar[1], ar[2], ar[3]);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const Lse s{-(double)mn[c], tt[c]};
        carry[((int64_t)R.slot * Qs + 4 * j + c) * 2 + 0] = s.m;
        carry[((int64_t)R.slot * Qs + 4 * j + c) * 2 + 1] = s.t;
        glob[c] = lse_merge_fast(glob[c], s);
      }
    } else {
      emit(cur);
    }
  }
  // Block partial of the global log-sum-exp, per pattern edge in a fixed (wave, group) order: the groups' maxima, then
  // every group's share of the largest, then their sum.
  const int slots = (kWalkBlock / 64) * G, sl = wave * G + g;  // [slots][Qs], then the maxima [Qs]
  if (g < G)
#pragma unroll
    for (int c = 0; c < 4; ++c) red[sl * Qs + 4 * j + c] = glob[c].m;
  __syncthreads();
  double* mx = red + kWalkBlock * 4;
  for (int q = threadIdx.x; q < Qs; q += kWalkBlock) {
    double m = -kInf;
    for (int i = 0; i < slots; ++i) m = fmax(m, red[i * Qs + q]);
    mx[q] = m;
  }
  __syncthreads();
  if (g < G)
#pragma unroll
    for (int c = 0; c < 4; ++c) red[sl * Qs + 4 * j + c] = lse_rescaled(glob[c], mx[4 * j + c]);
  __syncthreads();
  for (int q = threadIdx.x; q < Q; q += kWalkBlock) {
    Lse acc{mx[q], 0.0};
    bool seen = false;
    for (int i = 0; i < slots; ++i) lse_sum_step(acc.t, seen, red[i * Qs + q]);
    gpart[(int64_t)q * gridDim.x + blockIdx.x] = acc;
  }
}

void launch_walk_src(int64_t nruns, const Run* runs, const int2* ks, const float* CE, int Q, int Qs, float* minCEo,
                     float* lsO, float* VFm, double* carry, Lse* gpart, int nblocks, hipStream_t st, int* AO,
                     int* carg) {
  if (AO)
    hipLaunchKernelGGL(k_walk_src<true>, dim3(nblocks), dim3(kWalkBlock), 0, st, nruns, runs, ks, CE, Q, Qs, minCEo, lsO,
                       VFm, carry, gpart, AO, carg);
  else
    hipLaunchKernelGGL(k_walk_src<false>, dim3(nblocks), dim3(kWalkBlock), 0, st, nruns, runs, ks, CE, Q, Qs, minCEo, lsO,
                       VFm, carry, gpart, AO, carg);
}

// The split vertices' pieces combined: groups of Qs/4 lanes take a vertex's pieces round-robin (lane j owns pattern edges
// 4j..4j+3), and their results are combined through LDS in a fixed order.  Bound by latency, a few dependent reads per
// vertex, and by the hubs' chains, so the vertices of a list (hubs first, those of few pieces last) are taken in three
// ways: a hub by all kFixWaves waves of a block, one of at most kFewPieces pieces by a thread per pattern edge, its pieces
// all in flight (where a wave has as many groups, so that the pieces' order is that of the groups), the others by a wave.  A
// wave for every vertex, before: R-MAT 18, 12/16 pattern, 48 us for the source side's sums and 15 us for the taped maxima;
// now 26 and 10 us; 50,001 vertices, 40/70: 48 and 20 us for the sums.
constexpr int kFixWaves = 8;
struct FixTask {
  Split S;
  int g, j, w, W;  // the lane's group and place in it; the wave's place among the W that share the vertex
  bool active, few;
};
__device__ __forceinline__ FixTask fix_task(const SplitList& L, int Qs) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, L4 = Qs / 4, G = 64 / L4;
  const int nfew = G >= kFewPieces ? L.nfew : 0, nmid = L.n - L.nhub - nfew;
  const int bmid = L.nhub + (nmid + kFixWaves - 1) / kFixWaves, b = blockIdx.x;
  FixTask f;
  f.g = lane / L4;
  f.j = lane - f.g * L4;
  f.W = b < L.nhub ? kFixWaves : 1;
  f.w = b < L.nhub ? wave : 0;
  f.few = b >= bmid;
  int i = b < L.nhub ? b : L.nhub + (b - L.nhub) * kFixWaves + wave, end = L.n - nfew;
  f.active = f.g < G;
  if (f.few) {  // g: unused; j: the thread's pattern edge
    const int64_t e0 = (int64_t)(b - bmid) * (64 * kFixWaves), v0 = e0 / Qs;  // (the same for the block)
    const int e = (int)(e0 - v0 * Qs) + threadIdx.x;
    i = L.n - nfew + (int)v0 + e / Qs;
    end = L.n;
    f.j = e - e / Qs * Qs;
    f.active = true;
  }
  f.active = f.active && i < end;
  f.S = f.active ? L.splits[i] : Split{0, 0, 0, 0};
  return f;
}
static unsigned fix_blocks(const SplitList& L, int Qs) {
  const int G = 64 / (Qs / 4), nfew = G >= kFewPieces ? L.nfew : 0, nmid = L.n - L.nhub - nfew;
  return L.nhub + (nmid + kFixWaves - 1) / kFixWaves +
         (int)(((int64_t)nfew * Qs + 64 * kFixWaves - 1) / (64 * kFixWaves));
}

// The largest maximum first, then the pieces' shares of it, whose exponentials do not wait for each other.
__global__ __launch_bounds__(64 * kFixWaves) void k_walk_src_fixup(SplitList L,
                                                                   const double* __restrict__ carry, int Q, int Qs,
                                                                   float* __restrict__ minCEo, float* __restrict__ lsO,
                                                                   float* __restrict__ VFm, const int* __restrict__ carg,
                                                                   int* __restrict__ AO) {
  __shared__ double red[kFixWaves][64][4];
  __shared__ int rarg[kFixWaves][64][4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, L4 = Qs / 4, G = 64 / L4;
  const FixTask f = fix_task(L, Qs);
  const int c0 = f.w * G + f.g, step = f.W * G, row = wave - f.w, j = f.j;  // row of red: the vertex's combined results
  if (f.few) {
    if (!f.active) return;
    const double2* o = reinterpret_cast<const double2*>(carry) + (int64_t)f.S.first * Qs + j;
    double2 x[kFewPieces];
#pragma unroll
    for (int c = 0; c < kFewPieces; ++c) x[c] = o[(int64_t)min(c, f.S.count - 1) * Qs];
    double M = x[0].x, sum = 0.0;
    bool any = false;
    int a = INT_MAX;
#pragma unroll
    for (int c = 1; c < kFewPieces; ++c) M = fmax(M, x[c].x);  // (past the last piece: that piece again)
#pragma unroll
    for (int c = 0; c < kFewPieces; ++c)
      if (c < f.S.count) {
        if (AO && x[c].x == M) a = min(a, carg[(int64_t)(f.S.first + c) * Qs + j]);
        lse_sum_step(sum, any, lse_rescaled(Lse{x[c].x, x[c].y}, M));
      }
    const int64_t at = (int64_t)f.S.v * Qs + j;
    minCEo[at] = j < Q ? (float)(-M) : 0.f;
    lsO[at] = j < Q ? (float)log1p(sum) : 0.f;
    VFm[at] = j < Q ? (float)M : 0.f;
    if (AO) AO[at] = a;
    return;
  }
  const double* base = carry + ((int64_t)f.S.first * Qs + 4 * j) * 2;
  double M[4] = {-kInf, -kInf, -kInf, -kInf}, sum[4] = {0.0, 0.0, 0.0, 0.0};
  bool seen[4] = {false, false, false, false};
  if (f.active)
#pragma unroll 4
    for (int c = c0; c < f.S.count; c += step)
#pragma unroll
      for (int u = 0; u < 4; ++u) M[u] = fmax(M[u], base[(int64_t)c * Qs * 2 + 2 * u]);
#pragma unroll
  for (int u = 0; u < 4; ++u) red[wave][lane][u] = M[u];
  __syncthreads();
  const int used = min(G, f.S.count);  // groups that have a piece
  if (f.W > 1) {
    if (t < 256)
      for (int w = 1; w < kFixWaves; ++w) red[0][t >> 2][t & 3] = fmax(red[0][t >> 2][t & 3], red[w][t >> 2][t & 3]);
    __syncthreads();
  }
  if (f.active)
    for (int gg = 0; gg < used; ++gg)
#pragma unroll
      for (int u = 0; u < 4; ++u) M[u] = fmax(M[u], red[row][gg * L4 + j][u]);
  int ar[4] = {INT_MAX, INT_MAX, INT_MAX, INT_MAX};  // with AO: the lowest row of the pieces that hold the least cost
  if (f.active)
#pragma unroll 4
    for (int c = c0; c < f.S.count; c += step)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double* o = base + (int64_t)c * Qs * 2 + 2 * u;
        if (AO && o[0] == M[u]) ar[u] = min(ar[u], carg[(int64_t)(f.S.first + c) * Qs + 4 * j + u]);
        lse_sum_step(sum[u], seen[u], lse_rescaled(Lse{o[0], o[1]}, M[u]));
      }
  __syncthreads();  // the maxima are read
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    red[wave][lane][u] = seen[u] ? -sum[u] : sum[u];  // a share of the group (lse_sum_step)
    rarg[wave][lane][u] = ar[u];
  }
  __syncthreads();
  if (f.W > 1) {
    if (t < 256) {
      double x = 0.0;
      bool any = false;
      int a = INT_MAX;
      for (int w = 0; w < kFixWaves; ++w) {
        lse_sum_step(x, any, red[w][t >> 2][t & 3]);
        a = min(a, rarg[w][t >> 2][t & 3]);
      }
      red[0][t >> 2][t & 3] = any ? -x : x;
      rarg[0][t >> 2][t & 3] = a;
    }
    __syncthreads();
  }
  if (f.active && f.w == 0 && f.g == 0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      double x = 0.0;
      bool any = false;
      for (int gg = 0; gg < used; ++gg) lse_sum_step(x, any, red[row][gg * L4 + j][u]);
      const int q = 4 * j + u;
      const int64_t o = (int64_t)f.S.v * Qs + q;
      minCEo[o] = q < Q ? (float)(-M[u]) : 0.f;
      lsO[o] = q < Q ? (float)log1p(x) : 0.f;
      VFm[o] = q < Q ? (float)M[u] : 0.f;
      if (AO) {
        int a = INT_MAX;
        for (int gg = 0; gg < used; ++gg) a = min(a, rarg[row][gg * L4 + j][u]);
        AO[o] = a;
      }
    }
  }
}

void launch_walk_src_fixup(const SplitList& L, const double* carry, int Q, int Qs, float* minCEo,
                           float* lsO, float* VFm, hipStream_t st, const int* carg, int* AO) {
  if (L.n == 0) return;
  hipLaunchKernelGGL(k_walk_src_fixup, dim3(fix_blocks(L, Qs)), dim3(64 * kFixWaves), 0, st, L, carry, Q, Qs, minCEo, lsO, VFm, carg, AO);
}

// ---------------------------------------------------------------------------------------------------------------
// Destination maxima (CSC walk), src/main.cu:220-224 with the log-softmax of src/main.cu:218 folded in:
//   FMaxN[v][q] = max over in-edges e of v of (VR[src e][q] - CE[e][q])  -  log sum_e exp(FE[q][e])
// computed exactly in FP64 (a difference of two floats is exact in double) and rounded once.  With VR == nullptr
// it is the prep's max over in-edges of -CE (src/main.cu:143-146).
//
// One wave walks one bundle of G runs, group g (Qs/4 lanes) walking run g, lane j owning pattern edges 4j..4j+3.
// Step s of the bundle reads rows base + s*G + g of CE (one contiguous block of G*Qs floats for the wave), of bsrc
// and of bdst, and gathers row bsrc of VR.  The steps go in batches of B, software-pipelined two batches deep with
// two register sets used in turn (no register copies, so no wait for loads in flight at a loop back-edge): while
// batch t is reduced, the costs, destinations and gathered rows of batch t + 1 and the sources of batches t + 2 and
// t + 3 are in flight.  Loads past the bundle's last batch are clamped to it and never used.

int walk_groups(int Qs) { return 64 / (Qs / 4); }

int walk_batch() {
  if (const char* e = std::getenv("AC_WALK_BATCH")) {  // tuning override: 1, 2 or 4
    const int b = std::atoi(e);
    if (b == 1 || b == 2 || b == 4) return b;
  }
  return 4;  // measured at R-MAT 22 with packed costs and runs of 128 edges
}

// Float maximum by integer atomics, exact and independent of order: floats of positive sign order like signed ints,
// those of negative sign inversely to their unsigned bit patterns.  A NaN wins whatever its sign.
__device__ __forceinline__ void atomic_raise(float* addr, float v) {
  if (v != v) v = __uint_as_float(0x7FC00000u);
  if (signbit(v))
    atomicMin(reinterpret_cast<unsigned*>(addr), __float_as_uint(v));
  else
    atomicMax(reinterpret_cast<int*>(addr), __float_as_int(v));
}

// kArg: also records, per (v, q), the row of the in-edge attaining the maximum (the first one in walk order on
// ties; -1 if none) into FA[v][Qs], and per carry slot into carg, for the adjoint's max-subgradient routing.
// kPrune (bmin != nullptr): exact pruning, per bundle and per lane (below).
template <bool kWithVR, int B, bool kArg, bool kPrune>
__global__ __launch_bounds__(kWalkBlock) void k_walk_max(int64_t nbundles, const Bundle* __restrict__ bundles,
                                                         const int* __restrict__ gslot, const int* __restrict__ bsrc,
                                                         const int* __restrict__ bdst, const float* __restrict__ CE,
                                                         const float* __restrict__ VR, int VRs, int Q, int Qs,
                                                         const QStat* __restrict__ qs, float* __restrict__ FMaxN,
                                                         double* __restrict__ carry, int* __restrict__ FA,
                                                         int* __restrict__ carg, const float* __restrict__ bmin,
                                                         const unsigned* __restrict__ CEp,
                                                         const unsigned* __restrict__ bpack,
                                                         unsigned* __restrict__ CEpo, int* __restrict__ bstate) {
  const int L4 = Qs / 4, G = 64 / L4, VR4s = VRs / 4;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane / L4, j = lane - g * L4;
  const int64_t b = (int64_t)blockIdx.x * (kWalkBlock / 64) + wave;  // wave-uniform: the bundle header is scalar
  if (g >= G || b >= nbundles) return;
  const Bundle Bd = bundles[b];
  const int gs = gslot[b * G + g], slot = gs < 0 ? gs : gs & ~kCrowded;
  // bstate (nullable): whether the bundle's FMaxN rows may hold anything but -inf.
  const int written = kPrune && bstate ? bstate[b] : 1;
  // Exact pruning: an edge whose cost is at or above its pattern edge's bound cannot raise FMax above the fill, so a
  // term that is -inf instead gives the same FMax (the fill wins, as it would have).  A wave with no live lane skips
  // its bundle and writes -inf rows; a dead lane (none of its four pattern edges has a cost below the bound in this
  // bundle) skips its cost loads and VR gathers, and its maxima stay -inf.
  bool live = true;
  if (kPrune) {
    live = false;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = 4 * j + u;
      if (q < Q && (double)bmin[b * Qs + q] < qs[q].cthr) live = true;
    }
    if (!__any(live)) {
      if (slot >= 0 && kArg) {
        double* o = carry + (int64_t)slot * Qs + 4 * j;
        o[0] = o[1] = o[2] = o[3] = -kInf;
      } else if (slot < 0 && written) {  // (a piece leaves its split vertex's row, reset to -inf, alone)
        const int v0 = bdst[Bd.base + g], v1 = bdst[Bd.base + (int64_t)(Bd.len - 1) * G + g];
        const float4 ninf = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
        if (v0 >= 0)
          for (int v = v0; v <= v1; ++v) reinterpret_cast<float4*>(FMaxN)[(int64_t)v * L4 + j] = ninf;
      }
      if (bstate && written && lane == 0) bstate[b] = 0;
      return;
    }
  }
  if (bstate && lane == 0 && (!kPrune || !written)) bstate[b] = 1;
  // log sum_e exp(FE[q][e]) as one FP64 value (its FP64 rounding is far below the FP32 rounding of the result).
  double sl[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int q = 4 * j + c;
    sl[c] = q < Q ? qs[q].mFE + qs[q].lFE : 0.0;
  }
  double mx0 = -kInf, mx1 = -kInf, mx2 = -kInf, mx3 = -kInf;
  int a0 = -1, a1 = -1, a2 = -1, a3 = -1;
  int cur = -1;
  // Finished vertex v: its row of maxima, normalised (a macro rather than a lambda, so that the walk's loop-carried
  // state is not captured by reference twice over and stays in registers).
#define AC_WK_EMIT(V)                                                                           \
  {                                                                                             \
    const f4v o_ = f4v{(float)(mx0 - sl[0]), (float)(mx1 - sl[1]), (float)(mx2 - sl[2]),         \
                       (float)(mx3 - sl[3])};                                                   \
    reinterpret_cast<f4v*>(FMaxN)[(int64_t)(V) * L4 + j] = o_;                                  \
    if (kArg) {                                                                                 \
      reinterpret_cast<int4*>(FA)[(int64_t)(V) * L4 + j] = make_int4(a0, a1, a2, a3);           \
      a0 = a1 = a2 = a3 = -1;                                                                   \
    }                                                                                           \
    mx0 = mx1 = mx2 = mx3 = -kInf;                                                              \
  }
  const int GL4 = G * L4;
  // Streams: a wave-uniform bundle base plus small per-lane offsets (32-bit address arithmetic).
  const int* srcb = bsrc + Bd.base;
  const f4v* ceb = reinterpret_cast<const f4v*>(CE) + Bd.base * L4;
  const unsigned so = (unsigned)g, co = (unsigned)(g * L4 + j);
  // Plain walk (kWithVR, !kArg): destinations come from the sources' new-vertex flags (a run's vertices are
  // consecutive), so only the run's first destination is read.
  constexpr bool kFlags = kWithVR && !kArg;
  if (kFlags) cur = bdst[Bd.base + g];
  const int* dstp = bdst + Bd.base + g;
  const f4v* VRv = reinterpret_cast<const f4v*>(VR);
  const int last = Bd.len / B - 1;
  // Packed costs (CEp != nullptr): the bundle's base, 0 when it keeps its FP32 rows.  Decoding is exact, so maxima
  // and recorded argmax rows are those of the FP32 walk.
  const unsigned pbase = CEp ? bpack[b] : 0u;
  const unsigned* cpb = CEp ? CEp + Bd.base * L4 * 3 : nullptr;
  // Packing on the way (the prep walk, CEpo != nullptr, no pruning): every row is reduced exactly once from its FP32
  // costs, and is also written out as 24-bit codes when the bundle's base is nonzero (pack_base: each cost of a column
  // q < Q other than +inf codes as its bit pattern minus the base, +inf and columns q >= Q as 0).
  const unsigned obase = CEpo && !kPrune ? bpack[b] : 0u;
  unsigned* const cpo = obase ? CEpo + Bd.base * L4 * 3 : nullptr;
#define AC_WK_SRC(S, T)                                                          \
  if (kWithVR) {                                                                 \
    const int t_ = (T) < last ? (T) : last;                                      \
    _Pragma("unroll") for (int u = 0; u < B; ++u) S[u] =                         \
        __builtin_nontemporal_load(srcb + (so + (unsigned)((t_ * B + u) * G)));  \
  }
#define AC_WK_BATCH(C, D, W, S, T)                                                                       \
  {                                                                                                      \
    const int t_ = (T) < last ? (T) : last;                                                              \
    _Pragma("unroll") for (int u = 0; u < B; ++u) {                                                      \
      if constexpr (kP)                                                                                  \
        C[u] = (!kPrune || live) ? nt_load_u3(cpb + 3 * (co + (unsigned)((t_ * B + u) * GL4)))           \
                                 : U3{0u, 0u, 0u};                                                       \
      else                                                                                               \
        C[u] = (!kPrune || live) ? __builtin_nontemporal_load(ceb + (co + (unsigned)((t_ * B + u) * GL4))) \
                                 : f4v{INFINITY, INFINITY, INFINITY, INFINITY};                          \
    }                                                                                                    \
    _Pragma("unroll") for (int u = 0; u < B; ++u) D[u] =                                                 \
        kFlags ? (S[u] & kNewVertex) : __builtin_nontemporal_load(dstp + (t_ * B + u) * G);              \
    _Pragma("unroll") for (int u = 0; u < B; ++u) W[u] =                                                 \
        (kWithVR && (!kPrune || live)) ? VRv[(int64_t)(S[u] & ~kNewVertex) * VR4s + j]                   \
                                       : f4v{0.f, 0.f, 0.f, 0.f};                                        \
  }
#define AC_WK_REDUCE(C, D, W, T)                                                    \
  _Pragma("unroll") for (int u = 0; u < B; ++u) {                                   \
    if (kFlags) {                                                                   \
      if (D[u]) {                                                                   \
        AC_WK_EMIT(cur);                                                            \
        ++cur;                                                                      \
      }                                                                             \
    } else if (D[u] != cur) {                                                       \
      if (cur >= 0) AC_WK_EMIT(cur);                                                \
      cur = D[u];                                                                   \
    }                                                                               \
    f4v c_;                                                                         \
    if constexpr (kP)                                                               \
      c_ = decode_costs(C[u], pbase);                                               \
    else                                                                            \
      c_ = C[u];                                                                    \
    if (!kP && cpo) {                                                               \
      unsigned k_[4];                                                               \
      _Pragma("unroll") for (int w_ = 0; w_ < 4; ++w_) {                            \
        const unsigned x_ = __float_as_uint(c_[w_]);                                \
        k_[w_] = (4 * j + w_ < Q && x_ != 0x7F800000u) ? x_ - obase : 0u;           \
      }                                                                             \
      unsigned* o_ = cpo + 3 * (co + (unsigned)(((T) * B + u) * GL4));             \
      o_[0] = k_[0] | (k_[1] << 24);                                                \
      o_[1] = (k_[1] >> 8) | (k_[2] << 16);                                         \
      o_[2] = (k_[2] >> 16) | (k_[3] << 8);                                         \
    }                                                                               \
    const double d0 = (double)W[u].x - (double)c_.x;                                \
    const double d1 = (double)W[u].y - (double)c_.y;                                \
    const double d2 = (double)W[u].z - (double)c_.z;                                \
    const double d3 = (double)W[u].w - (double)c_.w;                                \
    if (kArg) {                                                                     \
      const int row_ = (int)(Bd.base + g) + ((T) * B + u) * G;                       \
      if (d0 > mx0) mx0 = d0, a0 = row_;                                            \
      if (d1 > mx1) mx1 = d1, a1 = row_;                                            \
      if (d2 > mx2) mx2 = d2, a2 = row_;                                            \
      if (d3 > mx3) mx3 = d3, a3 = row_;                                            \
    } else {                                                                        \
      mx0 = fmax(mx0, d0);                                                          \
      mx1 = fmax(mx1, d1);                                                          \
      mx2 = fmax(mx2, d2);                                                          \
      mx3 = fmax(mx3, d3);                                                          \
    }                                                                               \
  }
  // The pipelined walk over the bundle, for FP32 cost rows (kP false) or packed ones (decoded when reduced, so the
  // loads stay in flight as raw dwords).  kP is written in terms of the template parameters so that it is
  // value-dependent: the discarded `if constexpr` branches are then not instantiated.
#define AC_WK_PIPELINE(KP)                                                   \
  {                                                                          \
    constexpr bool kP = (KP);                                                \
    typedef typename std::conditional<kP, U3, f4v>::type CostRow;            \
    int SA[B], SB[B], DA[B], DB[B];                                          \
    CostRow CA[B], CB[B];                                                    \
    f4v WA[B], WB[B];                                                        \
    _Pragma("unroll") for (int u = 0; u < B; ++u) SA[u] = SB[u] = 0;         \
    AC_WK_SRC(SA, 0);                                                        \
    AC_WK_SRC(SB, 1);                                                        \
    AC_WK_BATCH(CA, DA, WA, SA, 0);                                          \
    AC_WK_SRC(SA, 2);                                                        \
    for (int t = 0;; t += 2) {                                               \
      AC_WK_BATCH(CB, DB, WB, SB, t + 1);                                    \
      AC_WK_SRC(SB, t + 3);                                                  \
      AC_WK_REDUCE(CA, DA, WA, t);                                           \
      if (t + 1 > last) break;                                               \
      AC_WK_BATCH(CA, DA, WA, SA, t + 2);                                    \
      AC_WK_SRC(SA, t + 4);                                                  \
      AC_WK_REDUCE(CB, DB, WB, t + 1);                                       \
      if (t + 2 > last) break;                                               \
    }                                                                        \
  }
  if (pbase)
    AC_WK_PIPELINE(kWithVR || B > 0)
  else
    AC_WK_PIPELINE(false && kWithVR)
#undef AC_WK_PIPELINE
#undef AC_WK_SRC
#undef AC_WK_BATCH
#undef AC_WK_REDUCE
  if (slot >= 0 && kArg) {
    double* o = carry + (int64_t)slot * Qs + 4 * j;
    o[0] = mx0;
    o[1] = mx1;
    o[2] = mx2;
    o[3] = mx3;
    reinterpret_cast<int4*>(carg)[(int64_t)slot * L4 + j] = make_int4(a0, a1, a2, a3);
  } else if (slot >= 0) {
    // A piece of a split vertex: its maximum, normalised and rounded like a finished row, raises the row.  Rounding
    // is monotone, so the maximum over the pieces of the rounded values is the rounded maximum (exact, in any order).
    const float o[4] = {(float)(mx0 - sl[0]), (float)(mx1 - sl[1]), (float)(mx2 - sl[2]), (float)(mx3 - sl[3])};
    float* row = FMaxN + (int64_t)cur * Qs + 4 * j;
    if (!__any(gs & kCrowded)) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (4 * j + u < Q && o[u] != -INFINITY) atomic_raise(row + u, o[u]);
      return;
    }
    // Pieces of a vertex of very many: a wave whose pieces are all one vertex's sends their maximum only, and a value not
    // above the row's present one (read without an atomic: the row only rises, so a stale value is a low one) is not sent.
    // With an atomic per piece the walk of 400,000 edges into one vertex, 12/16 pattern, took 354 us, now 31; combined
    // by two launches of their own (the pieces' maxima stored), the walk and they took 37.  (Apart from the others'
    // atomics: one sequence for both made a loop of 1,000 vertices, 10/12, 268 us long instead of 263.)
    float m[4] = {o[0], o[1], o[2], o[3]};
    bool raise = true;
    if (__all(cur == __builtin_amdgcn_readfirstlane(cur)) && __popcll(__ballot(1)) == GL4) {
      for (int d = 1; d < G; ++d) {
        const int from = (g + d < G ? g + d : g + d - G) * L4 + j;
#pragma unroll
        for (int u = 0; u < 4; ++u) m[u] = fmaxf(m[u], __shfl(o[u], from, 64));
      }
      raise = g == 0;
    }
    if (raise) {
      float has[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) has[u] = __hip_atomic_load(row + u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (4 * j + u < Q && !(m[u] <= has[u])) atomic_raise(row + u, m[u]);
    }
  } else if (cur >= 0) {
    AC_WK_EMIT(cur);
  }
#undef AC_WK_EMIT
}

template <bool kWithVR, bool kArg, bool kPrune>
static void launch_walk_max_t(int B, int nb, hipStream_t st, int64_t nbundles, const Bundle* bundles,
                              const int* gslot, const int* bsrc, const int* bdst, const float* CE, const float* VR,
                              int VRs, int Q, int Qs, const QStat* qs, float* FMaxN, double* carry, int* FA,
                              int* carg, const float* bmin, const unsigned* CEp, const unsigned* bpack,
                              unsigned* CEpo, int* bstate) {
  switch (B) {
    case 1:
      hipLaunchKernelGGL((k_walk_max<kWithVR, 1, kArg, kPrune>), dim3(nb), dim3(kWalkBlock), 0, st, nbundles,
                         bundles, gslot, bsrc, bdst, CE, VR, VRs, Q, Qs, qs, FMaxN, carry, FA, carg, bmin, CEp, bpack,
                         CEpo, bstate);
      break;
    case 4:
      hipLaunchKernelGGL((k_walk_max<kWithVR, 4, kArg, kPrune>), dim3(nb), dim3(kWalkBlock), 0, st, nbundles,
                         bundles, gslot, bsrc, bdst, CE, VR, VRs, Q, Qs, qs, FMaxN, carry, FA, carg, bmin, CEp, bpack,
                         CEpo, bstate);
      break;
    default:
      hipLaunchKernelGGL((k_walk_max<kWithVR, 2, kArg, kPrune>), dim3(nb), dim3(kWalkBlock), 0, st, nbundles,
                         bundles, gslot, bsrc, bdst, CE, VR, VRs, Q, Qs, qs, FMaxN, carry, FA, carg, bmin, CEp, bpack,
                         CEpo, bstate);
      break;
  }
}

template <bool kWithVR, bool kArg>
static void launch_walk_max_p(int B, int nb, hipStream_t st, int64_t nbundles, const Bundle* bundles,
                              const int* gslot, const int* bsrc, const int* bdst, const float* CE, const float* VR,
                              int VRs, int Q, int Qs, const QStat* qs, float* FMaxN, double* carry, int* FA,
                              int* carg, const float* bmin, const unsigned* CEp, const unsigned* bpack,
                              unsigned* CEpo, int* bstate) {
  if (bmin)
    launch_walk_max_t<kWithVR, kArg, true>(B, nb, st, nbundles, bundles, gslot, bsrc, bdst, CE, VR, VRs, Q, Qs, qs,
                                           FMaxN, carry, FA, carg, bmin, CEp, bpack, CEpo, bstate);
  else
    launch_walk_max_t<kWithVR, kArg, false>(B, nb, st, nbundles, bundles, gslot, bsrc, bdst, CE, VR, VRs, Q, Qs, qs,
                                            FMaxN, carry, FA, carg, bmin, CEp, bpack, CEpo, bstate);
}

void launch_walk_max(int64_t nbundles, const Bundle* bundles, const int* gslot, const int* bsrc, const int* bdst,
                     const float* CE, const float* VR, int VRs, int Q, int Qs, const QStat* qs, float* FMaxN,
                     double* carry, int B, hipStream_t st, int* FA, int* carg, const float* bmin,
                     const unsigned* CEp, const unsigned* bpack, unsigned* CEp_out, int* bstate) {
  if (nbundles == 0) return;
  const int nb = (int)((nbundles + kWalkBlock / 64 - 1) / (kWalkBlock / 64));
  if (!bpack) CEp = CEp_out = nullptr;
  if (CEp_out) CEp = nullptr;  // packing on the way: the walk reads the FP32 rows
  if (VR && FA)
    launch_walk_max_p<true, true>(B, nb, st, nbundles, bundles, gslot, bsrc, bdst, CE, VR, VRs, Q, Qs, qs, FMaxN,
                                  carry, FA, carg, bmin, CEp, bpack, CEp_out, bstate);
  else if (VR)
    launch_walk_max_p<true, false>(B, nb, st, nbundles, bundles, gslot, bsrc, bdst, CE, VR, VRs, Q, Qs, qs, FMaxN,
                                   carry, FA, carg, bmin, CEp, bpack, CEp_out, bstate);
  else if (FA)
    launch_walk_max_p<false, true>(B, nb, st, nbundles, bundles, gslot, bsrc, bdst, CE, VR, VRs, Q, Qs, qs, FMaxN,
                                   carry, FA, carg, bmin, CEp, bpack, CEp_out, bstate);
  else
    launch_walk_max_p<false, false>(B, nb, st, nbundles, bundles, gslot, bsrc, bdst, CE, VR, VRs, Q, Qs, qs, FMaxN,
                                    carry, FA, carg, bmin, CEp, bpack, CEp_out, bstate);
}

// The base of a bundle's 24-bit cost codes from its least and largest cost bit patterns over columns q < Q, +inf
// excluded (lo > hi: no such cost).  The costs must lie strictly inside two binades (2^e, 2^(e+2)) of one biased
// exponent e >= 1: then each is its bit pattern minus base = e << 23, a code in [1, 2^24), and +inf (padding rows)
// codes as 0.  Positive floats order as their bit patterns, so the least and largest patterns decide: a least cost
// that is a power of two widens the window down one binade, and negative, zero, subnormal or NaN costs fall outside
// every window.  0 = the bundle keeps its FP32 rows.
__device__ __forceinline__ unsigned pack_base(unsigned lo, unsigned hi) {
  if (lo > hi || hi >= 0x7F800000u) return 0u;
  unsigned e = lo >> 23;
  if ((lo & 0x7FFFFFu) == 0u) e = e > 0u ? e - 1u : 0u;  // code 0 is +inf: the least cost must lie above the base
  return e >= 1u && hi - (e << 23) < (1u << 24) ? e << 23 : 0u;
}

// Per bundle and pattern edge, the least cost among the bundle's rows (padding rows are +inf): bmin[b][Qs].  One
// wave per bundle, as the walk; the groups' minima are merged through LDS.  With bpack != nullptr it also writes
// the bundle's cost-code base (pack_base), from the same pass over the rows.
__global__ __launch_bounds__(kWalkBlock) void k_bundle_min(int64_t nbundles, const Bundle* __restrict__ bundles,
                                                           const float* __restrict__ CE, int Q, int Qs,
                                                           float* __restrict__ bmin, unsigned* __restrict__ bpack) {
  __shared__ f4v red[kWalkBlock / 64][64];
  const int L4 = Qs / 4, G = 64 / L4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane / L4, j = lane - g * L4;
  const int64_t b = (int64_t)blockIdx.x * (kWalkBlock / 64) + wave;
  f4v m = f4v{INFINITY, INFINITY, INFINITY, INFINITY};
  unsigned lo = 0xFFFFFFFFu, hi = 0u;
  if (g < G && b < nbundles) {
    const Bundle Bd = bundles[b];
    const f4v* ce = reinterpret_cast<const f4v*>(CE) + (Bd.base + g) * L4 + j;
    // Eight rows in flight (past the end: the last one again), where a row at a time waited for each.
    for (int s0 = 0; s0 < Bd.len; s0 += 8) {
      f4v c[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) c[s] = __builtin_nontemporal_load(ce + (int64_t)min(s0 + s, Bd.len - 1) * G * L4);
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        m = f4v{fminf(m[0], c[s][0]), fminf(m[1], c[s][1]), fminf(m[2], c[s][2]), fminf(m[3], c[s][3])};
        if (bpack) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const unsigned x = __float_as_uint(c[s][u]);
            if (4 * j + u < Q && x != 0x7F800000u) {
              lo = min(lo, x);
              hi = max(hi, x);
            }
          }
        }
      }
    }
  }
  if (bpack) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo = min(lo, (unsigned)__shfl_xor((int)lo, o, 64));
      hi = max(hi, (unsigned)__shfl_xor((int)hi, o, 64));
    }
    if (lane == 0 && b < nbundles) bpack[b] = pack_base(lo, hi);
  }
  red[wave][lane] = m;
  __syncthreads();
  if (b < nbundles && lane < L4) {
    f4v a = red[wave][lane];
    for (int gg = 1; gg < G; ++gg) {
      const f4v c = red[wave][gg * L4 + lane];
      a = f4v{fminf(a[0], c[0]), fminf(a[1], c[1]), fminf(a[2], c[2]), fminf(a[3], c[3])};
    }
    reinterpret_cast<f4v*>(bmin)[b * L4 + lane] = a;
  }
}

void launch_bundle_min(int64_t nbundles, const Bundle* bundles, const float* CE, int Q, int Qs, float* bmin,
                       unsigned* bpack, hipStream_t st) {
  if (nbundles == 0) return;
  const int nb = (int)((nbundles + kWalkBlock / 64 - 1) / (kWalkBlock / 64));
  hipLaunchKernelGGL(k_bundle_min, dim3(nb), dim3(kWalkBlock), 0, st, nbundles, bundles, CE, Q, Qs, bmin, bpack);
}

// Bundle layout from the CSC arrays: one block per bundle writes its rows (step-major, run-minor).  rowmap[k] is
// the row of CSC position k.  brun[b * G + g] is the run walked by group g of bundle b (-1: none).
__global__ __launch_bounds__(256) void k_build_bundles(const Bundle* __restrict__ bundles, const int* __restrict__ brun,
                                                       const Run* __restrict__ runs, const int2* __restrict__ sd,
                                                       const int* __restrict__ eid, int G, int* __restrict__ bsrc,
                                                       int* __restrict__ bdst, int* __restrict__ beid,
                                                       int* __restrict__ rowmap) {
  const int64_t b = blockIdx.x;
  const Bundle Bd = bundles[b];
  const int nrow = Bd.len * G;
  for (int i = threadIdx.x; i < nrow; i += blockDim.x) {
    const int s = i / G, g = i - s * G;
    const int r = brun[b * G + g];
    const int64_t row = Bd.base + i;
    int src = 0, dst = -1, e = -1;
    if (r >= 0) {
      const Run R = runs[r];
      if (R.kb + s < R.ke) {
        const int k = R.kb + s;
        src = sd[k].x;
        dst = sd[k].y;
        e = eid[k];
        rowmap[k] = (int)row;
        if (s > 0 && sd[k - 1].y != dst) src |= kNewVertex;  // the run moves on to the next vertex (dst + 1)
      } else {
        dst = sd[R.ke - 1].y;
      }
    }
    bsrc[row] = src;
    bdst[row] = dst;
    beid[row] = e;
  }
}

void launch_build_bundles(int64_t nbundles, const Bundle* bundles, const int* brun, const Run* runs, const int2* sd,
                          const int* eid, int G, int* bsrc, int* bdst, int* beid, int* rowmap, hipStream_t st) {
  if (nbundles == 0) return;
  hipLaunchKernelGGL(k_build_bundles, dim3((unsigned)nbundles), dim3(256), 0, st, bundles, brun, runs, sd, eid, G,
                     bsrc, bdst, beid, rowmap);
}

__global__ void k_remap_ks(int64_t m, const int2* __restrict__ ks, const int* __restrict__ rowmap,
                           int2* __restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
    const int2 e = ks[i];
    out[i] = make_int2(rowmap[e.x], e.y);
  }
}

void launch_remap_ks(int64_t m, const int2* ks, const int* rowmap, int2* out, hipStream_t st) {
  if (m == 0) return;
  const int blocks = (int)std::min<int64_t>((m + 255) / 256, 1 << 16);
  hipLaunchKernelGGL(k_remap_ks, dim3(blocks), dim3(256), 0, st, m, ks, rowmap, out);
}

// The taped walks' pieces, as k_walk_src_fixup: the maxima, and the row of the best piece into FA.  Of equal pieces the
// first of the lowest group counts, however many waves share the vertex.
__global__ __launch_bounds__(64 * kFixWaves) void k_walk_max_fixup(SplitList L,
                                                                   const double* __restrict__ carry, int Q, int Qs,
                                                                   const QStat* __restrict__ qs,
                                                                   float* __restrict__ FMaxN,
                                                                   const int* __restrict__ carg, int* __restrict__ FA) {
  __shared__ double red[kFixWaves][64][4];
  __shared__ int rpiece[kFixWaves][64][4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, L4 = Qs / 4, G = 64 / L4;
  const FixTask f = fix_task(L, Qs);
  // Normalised as the walk normalises a vertex it finishes (one FP64 subtraction of mFE + lFE, rounded once), so a
  // recording walk leaves the same FMaxN as a plain one, whose pieces are normalised that way.
  auto finish = [&](int q, double m, int piece) {
    const int64_t o = (int64_t)f.S.v * Qs + q;
    FMaxN[o] = (float)(m - (q < Q ? qs[q].mFE + qs[q].lFE : 0.0));
    FA[o] = piece < 0 ? -1 : carg[(int64_t)(f.S.first + piece) * Qs + q];
  };
  if (f.few) {
    if (!f.active) return;
    double o[kFewPieces], m = -kInf;
    int a = -1;
#pragma unroll
    for (int c = 0; c < kFewPieces; ++c) o[c] = carry[(int64_t)(f.S.first + min(c, f.S.count - 1)) * Qs + f.j];
#pragma unroll
    for (int c = 0; c < kFewPieces; ++c)  // (past the last piece: that piece again, which changes nothing)
      if (o[c] > m) m = o[c], a = c;
    finish(f.j, m, a);
    return;
  }
  double mx[4] = {-kInf, -kInf, -kInf, -kInf};
  int at[4] = {-1, -1, -1, -1};
  if (f.active)
#pragma unroll 4
    for (int c = f.w * G + f.g; c < f.S.count; c += f.W * G) {
      const double4 o = *reinterpret_cast<const double4*>(carry + (int64_t)(f.S.first + c) * Qs + 4 * f.j);
      const double ov[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (ov[u] > mx[u]) {
          mx[u] = ov[u];
          at[u] = c;
        }
    }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    red[wave][lane][u] = mx[u];
    rpiece[wave][lane][u] = at[u];
  }
  __syncthreads();
  if (f.W > 1) {
    if (t < 256) {
      double m = red[0][t >> 2][t & 3];
      int a = rpiece[0][t >> 2][t & 3];
      for (int w = 1; w < kFixWaves; ++w) {
        const double x = red[w][t >> 2][t & 3];
        const int xa = rpiece[w][t >> 2][t & 3];
        if (x > m || (x == m && xa < a)) m = x, a = xa;
      }
      red[0][t >> 2][t & 3] = m;
      rpiece[0][t >> 2][t & 3] = a;
    }
    __syncthreads();
  }
  if (f.active && f.w == 0 && f.g == 0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      double m = -kInf;
      int a = -1;
      for (int gg = 0; gg < min(G, f.S.count); ++gg)  // groups that have a piece
        if (red[wave][gg * L4 + f.j][u] > m) {
          m = red[wave][gg * L4 + f.j][u];
          a = rpiece[wave][gg * L4 + f.j][u];
        }
      finish(4 * f.j + u, m, a);
    }
  }
}

void launch_walk_max_fixup(const SplitList& L, const double* carry, int Q, int Qs, const QStat* qs,
                           float* FMaxN, hipStream_t st, const int* carg, int* FA) {
  if (L.n == 0) return;
  hipLaunchKernelGGL(k_walk_max_fixup, dim3(fix_blocks(L, Qs)), dim3(64 * kFixWaves), 0, st, L, carry, Q, Qs, qs, FMaxN, carg, FA);
}

// ---------------------------------------------------------------------------------------------------------------
// Vertex passes.  A block takes tiles of VT (a power of two, <= 64) consecutive vertices.  The tile's rows of FMaxN and
// VFm (and, in mode A, of minCEo and lsO), contiguous in HBM, and of CV are staged in LDS as FP32, into rows padded to an
// odd stride; the next tile's rows are loaded into registers (coalesced float4 loads) while the current tile is
// computed, so the loads of one tile overlap the arithmetic of the previous one.  Each thread's LDS positions are the
// same in every tile and are kept in registers: forming them took ten integer divisions per thread and tile.
//   p-phase : a lane per (tile row, pattern vertex), VT lanes to a pattern vertex: a wave handles 64 / VT of them at a
//             time.  MU_pre = -CV + sum over the incidences of p in ascending q (FMax term before RMax term;
//             src/ac.hxx:164-170 made deterministic), FMax = max(fillF, FMaxN), RMax = max(fillR, VFm - LSE_RE).
//             Mode A keeps MU = MU_pre - LSE_MU in LDS (FP64), mode OUT writes it in dn x pn order, mode C accumulates
//             the column's log-sum-exp per lane.
//   q-phase : (mode A) a thread per (q, row): VF = MU[pd] - FMax, VR = MU[ps] - RMax (src/main.cu:165-176), stored
//             with coalesced writes, and the per-q maxima / edge log-sum-exps accumulated in registers.
// At R-MAT 22 (64-row tiles) passes A and C are bound by their streams; on small graphs, and with patterns whose rows
// fill a tile with few vertices, by the chain through one block: its tables, its tiles one after the other, the merge
// of its partials.  Hence short tiles where there are few (vertex_tile), lanes shared among pattern vertices, and
// merges that take one exponential however many partials they merge.  Passes A / C per launch, before (a wave per
// pattern vertex whatever the tile's height, isolated vertices on block 0's way, serial merges, a term at a time) and
// now: 1,000 vertices with a 10/12 pattern 20.0 / 8.5 -> 7.5 / 5.1 us; 50,001 with 40/70 48.9 / 44.4 -> 28.1 / 19.7 us;
// R-MAT 16 slabs of 128 pattern edges 98.5 / 108.3 -> 50 / 35 us; R-MAT 20 with 16/24 105.7 / 58.9 -> 97 / 42 us.

constexpr int kVTMax = 64;
// Staged tile limits: VT * Qs <= 2048 and VT * P <= 2048 floats, for every block size NT (256 or 512).
constexpr int kTileFloats = 2048;

// One incidence of a pattern vertex in the MU sums: its term is fmax(fill, guard(x - m - l)) with x the staged value
// at column col of the adjacent FMaxN | VFm tiles.  An FMax term has m = l = 0 (x - 0 - 0 = x exactly, -inf stays
// -inf), so both kinds take the same branch-free sequence.
struct IncRec {
  double fill, m, l;
  int col, pad;
};

// Partial sums of the MU sums (tiles of fewer than 64 rows): up to kTerms consecutive incidences of one pattern vertex.
constexpr int kTerms = 4;

static size_t vertex_lds_bytes(int mode, int VT, int P, int Q, int Qs, int nsum) {
  size_t b = (size_t)(2 * P) * sizeof(double);                               // MU normalisers
  if (VT < 64) b += (size_t)nsum * (VT * sizeof(double) + sizeof(int2)) + (size_t)(P + 1) * sizeof(int);  // partial sums
  b += (size_t)(2 * Q + 1) * sizeof(IncRec);                                 // incidence records (+ one pad)
  if (mode != kModeC) b += (size_t)(P + 1) * VT * sizeof(double);            // MU
  const int nst = mode == kModeA ? 4 : 2;                                    // staged [VT][Qs] arrays
  b += (size_t)VT * (nst * (Qs + 1) + (P + 1)) * sizeof(float);              // staged rows
  b += (size_t)(P + 1) * sizeof(int);                                        // incidence offsets
  if (mode == kModeOut) b += (size_t)VT * sizeof(int);                       // the tile's caller ids
  return (b + 15) / 16 * 16;
}

// Tiles wanted at least: one for each of the 256 CUs.
constexpr int kTilesWanted = 256;

int vertex_sums(int P, const int* inc_off, int2* sums, int* off) {
  int m = 0;
  for (int p = 0; p < P; ++p) {
    if (off) off[p] = m;
    for (int k = inc_off[p]; k < inc_off[p + 1]; k += kTerms, ++m)
      if (sums) sums[m] = make_int2(k, std::min(k + kTerms, inc_off[p + 1]));
  }
  if (off) off[P] = m;
  return m;
}

int vertex_tile(int64_t n, int P, int Q, int nsum) {
  const int Qs = std::max(4, (Q + 3) / 4 * 4);
  int vt = kVTMax;
  if (const char* e = std::getenv("AC_VERTEX_TILE")) {  // tuning override: rows per tile, 8, 16, 32 or 64
    const int v = std::atoi(e);
    if (v == 8 || v == 16 || v == 32 || v == 64) vt = v;
  } else {
    while (vt > 8 && (n + vt - 1) / vt < kTilesWanted) vt /= 2;
  }
  while (vt > 4 && (vertex_lds_bytes(kModeA, vt, P, Q, Qs, nsum) > 65536 || vt * Qs > kTileFloats ||
                    vt * P > kTileFloats))
    vt /= 2;
  return vt;
}

// Read-only inputs seen through the constant address space: loads at wave-uniform indexes become scalar loads, and
// branches on their values scalar branches.
typedef const __attribute__((address_space(4))) int cint_t;

// The isolated vertices' share, in closed form (a block of a vertex pass of its own writes it as one extra partial).
// Their FMaxN = VFm = -inf rows make MU_pre = -CV + K_p, K_p the sum of the fills of p's incidences (in the vertex
// pass's own operation sequence), so MU is largest at the least-cost isolated vertex and the column log-sum-exp is
// LSE(-CV) + K_p.  They have no out-edges: no edge terms.
__device__ double iso_kp(const VertexArgs& a, const IncRec* recs, const int* ioff, int p, double acc) {
  if (a.first) return acc;
  const int step = a.VT == 64 ? 1 : kTerms;
  for (int k = ioff[p]; k < ioff[p + 1]; k += step) {
    double s = fmax(recs[k].fill, -kInf);
    for (int u = 1; u < step && k + u < ioff[p + 1]; ++u) s += fmax(recs[k + u].fill, -kInf);
    acc += s;
  }
  return acc;
}

__device__ QPart iso_qpart(const VertexArgs& a, const IncRec* recs, const int* ioff, int q) {
  QPart w{-kInf, -kInf, lse_empty(), lse_empty(), -1, -1};
  if (!a.iso) return w;
  const int pd = a.pd[q], ps = a.ps[q];
  const double fm = fmax(a.qs[q].fillF, -kInf), rm = fmax(a.qs[q].fillR, -kInf);
  if (a.iso[pd].vmin >= 0) {
    const double mu = (iso_kp(a, recs, ioff, pd, -(double)a.iso[pd].cmin) - a.pst[pd].m) - a.pst[pd].l;
    w.vfmax = mu - fm;
    if (w.vfmax > -kInf) w.avf = a.iso[pd].vmin;  // as in the vertex pass, -inf records no vertex
  }
  if (a.iso[ps].vmin >= 0) {
    const double mu = (iso_kp(a, recs, ioff, ps, -(double)a.iso[ps].cmin) - a.pst[ps].m) - a.pst[ps].l;
    w.vrmax = mu - rm;
    if (w.vrmax > -kInf) w.avr = a.iso[ps].vmin;
  }
  return w;
}

__device__ Lse iso_lse(const VertexArgs& a, const IncRec* recs, const int* ioff, int p) {
  if (!a.iso || a.iso[p].vmin < 0) return lse_empty();
  const double m = iso_kp(a, recs, ioff, p, a.iso[p].m);
  return m > -kInf ? Lse{m, a.iso[p].t} : lse_empty();
}

constexpr int kPW = 4;  // mode C: pattern vertices per lane; VT * P <= kTileFloats = kPW * 512 covers every P

// NT threads per block (kVW = NT / 64 waves); block 0 of modes A and C writes the isolated vertices' partial (slot nb),
// the other nb blocks take the tiles.
// kFull: VT == 64, so a wave handles one pattern vertex at a time and its incidence structure is wave-uniform.
// kArgMax (mode A): also track the vertices of the column maxima (the adjoint's tape needs them).
// kPFC: CV values each thread prefetches per tile (VT * P <= NT * kPFC); fewer registers allow more resident waves.
template <int kMode, bool kFull, bool kArgMax, int NT, int kPFC = kTileFloats / NT>
__global__ __launch_bounds__(NT, kMode == kModeA ? (kPFC == 4 ? 4 : 3) : 4) void k_vertex(VertexArgs a) {
  constexpr int kVW = NT / 64, kPF4 = kTileFloats / 4 / NT, kUnroll = kMode == kModeA ? 2 : 4;
  constexpr bool kA = kMode == kModeA, kC = kMode == kModeC;
  constexpr bool kRows = kMode == kModeOut || kMode == kModeMU;  // MU tile staged, written back row by row
  extern __shared__ double lds[];
  const int Q = a.Q, P = a.P, Qs = a.Qs, VT = kFull ? 64 : a.VT;
  const int ldq = Qs + 1, ldp = P + 1;
  double* pmu = lds;                                   // [2][P]: m, l of LSE_MU
  IncRec* recs = reinterpret_cast<IncRec*>(pmu + 2 * P);  // [2Q + 1] incidence records, inc order
  const int nsum = kFull ? 0 : a.nsum;
  double* Ps = reinterpret_cast<double*>(recs + 2 * Q + 1);  // [nsum][VT] partial sums (tiles of fewer than 64 rows)
  double* MUs = Ps + nsum * VT;                        // [VT][P + 1] (modes A, OUT, MU)
  const int ldm = P + 1;
  int2* tasks = reinterpret_cast<int2*>(MUs + (kC ? 0 : ldm * VT));  // [nsum] incidences [x, y) of each partial sum
  float* Fs = reinterpret_cast<float*>(tasks + nsum);  // [VT][ldq] FMaxN
  float* Vs = Fs + VT * ldq;                           // [VT][ldq] VFm
  float* Ms = Vs + VT * ldq;                           // [VT][ldq] minCEo (mode A)
  float* Ls = Ms + (kA ? VT * ldq : 0);                // [VT][ldq] lsO (mode A)
  float* Cs = Ls + (kA ? VT * ldq : 0);                // [VT][ldp] CV
  int* ioff = reinterpret_cast<int*>(Cs + VT * ldp);   // [P + 1] incidence offsets
  int* soff = ioff + P + 1;                            // [P + 1] first partial sum of each pattern vertex
  int* Prow = soff + (kFull ? 0 : P + 1);              // [VT] caller id of each tile row (mode OUT)
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const bool sums = !a.first;
  cint_t* const c_incoff = (cint_t*)a.inc_off;
  const bool iso_block = (kA || kC) && blockIdx.x == 0;
  const int64_t G = (kA || kC) ? gridDim.x - 1 : gridDim.x;  // tile blocks
  const int64_t blk = (kA || kC) ? (int64_t)blockIdx.x - 1 : blockIdx.x;
  const int64_t ntiles = (a.n + VT - 1) / VT;

  const f4v* F4 = reinterpret_cast<const f4v*>(a.FMaxN);
  const f4v* V4 = reinterpret_cast<const f4v*>(a.VFm);
  const f4v* M4 = reinterpret_cast<const f4v*>(a.minCEo);
  const f4v* L4v = reinterpret_cast<const f4v*>(a.lsO);
  const int64_t L4q = Qs / 4, f_end4 = a.f_end * L4q, o_lo4 = a.o_lo * L4q, o_hi4 = a.o_hi * L4q,
                o_end4 = a.o_end * L4q;
  typedef f4v PfSet[4][kPF4];  // FMaxN, VFm (and in pass A minCEo, lsO)
  PfSet pf = {};
  float pc[kPFC] = {};
  int pp = 0;  // mode OUT: the caller id of tile row t
  // Mode OUT of some columns: what they need of a row, the same in every tile (bit k: quadruple k; kPF4 + k: CV value k).
  unsigned need = ~0u;
  if (kMode == kModeOut && a.ncol < P) {
    need = 0u;
#pragma unroll
    for (int k = 0; k < kPF4; ++k) {
      const int col = 4 * (t + k * NT) % Qs;
      if (col + 4 > a.q0 && col < a.q0 + a.nq) need |= 1u << k;
    }
#pragma unroll
    for (int k = 0; k < kPFC; ++k) {
      const int col = (t + k * NT) % P;
      if (col >= a.c0 && col < a.c0 + a.ncol) need |= 1u << (kPF4 + k);
    }
  }
  // Loads of a tile into the register set; indexes past the tile are clamped to its last element (loaded, never
  // used).
  auto prefetch = [&](int64_t tl) __attribute__((always_inline)) {
    const int64_t v0_ = tl * VT;
    const int nv_ = (int)((a.n - v0_) < VT ? (a.n - v0_) : VT);
    const int last4_ = nv_ * Qs / 4 - 1, lastc_ = nv_ * P - 1;
    const int64_t b4_ = v0_ * Qs / 4, bc_ = v0_ * P;
#pragma unroll
    for (int k = 0; k < kPF4; ++k) {
      if (kMode == kModeOut && !(need >> k & 1u)) continue;
      const int64_t g_ = b4_ + min(t + k * NT, last4_);
      const bool hasF_ = !kA || g_ < f_end4, hasO_ = !kA || g_ < o_lo4 || (g_ >= o_hi4 && g_ < o_end4);
      pf[0][k] = hasF_ ? F4[g_] : f4v{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      pf[1][k] = hasO_ ? V4[g_] : f4v{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (kA) {
        pf[2][k] = hasO_ ? M4[g_] : f4v{INFINITY, INFINITY, INFINITY, INFINITY};
        pf[3][k] = hasO_ ? L4v[g_] : f4v{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int k = 0; k < kPFC; ++k)
      if (kMode != kModeOut || (need >> (kPF4 + k) & 1u)) pc[k] = a.CV[bc_ + min(t + k * NT, lastc_)];
    if (kMode == kModeOut && a.perm) pp = a.perm[v0_ + min(t, nv_ - 1)];
  };
  if (!iso_block && blk < ntiles) prefetch(blk);  // in flight while the tables are built

  // A pattern edge's two records, written at their places: the values and the places load together.  (From the incidences
  // the code came first, then what it names, one memory latency more in every block: the loop of 50,001 vertices with 40/70
  // 4.076 -> 4.035 ms, of R-MAT 14 with 24/36 1.160 -> 1.153.)
  for (int k = t; k <= Q; k += NT) {
    if (k < Q) {
      const QStat x = a.qs[k];
      const int2 at = a.inc_at[k];
      recs[at.x] = IncRec{x.fillF, 0.0, 0.0, k, 0};
      recs[at.y] = IncRec{x.fillR, x.mRE, x.lRE, VT * ldq + k, 0};
    } else {
      recs[2 * Q] = IncRec{-kInf, 0.0, 0.0, 0, 0};  // read ahead of the last incidence, never used
    }
  }
  for (int i = t; i <= P; i += NT) ioff[i] = a.inc_off[i];
  if (!kFull) {
    for (int i = t; i < nsum; i += NT) tasks[i] = a.sums[i];
    for (int i = t; i <= P; i += NT) soff[i] = a.sum_off[i];
  }
  if (!kC)
    for (int i = t; i < P; i += NT) {
      pmu[i] = a.pst[i].m;
      pmu[P + i] = a.pst[i].l;
    }
  if (iso_block) {
    __syncthreads();
    if (kA)
      for (int i = t; i < Q; i += NT) a.qpart[i * (G + 1) + G] = iso_qpart(a, recs, ioff, i);
    else
      for (int i = t; i < P; i += NT) a.ppart[i * (G + 1) + G] = iso_lse(a, recs, ioff, i);
    return;
  }

  // This thread's LDS positions of its staged values: element i = t + k NT of the tile goes to row i / width, column
  // i % width of the padded rows (below 2^16, two to a register).
  unsigned off4 = 0, offc[(kPFC + 1) / 2];
#pragma unroll
  for (int k = 0; k < kPF4; ++k) {
    const int e = 4 * (t + k * NT), r = e / Qs;
    off4 |= (unsigned)(r * ldq + e - r * Qs) << (16 * k);
  }
#pragma unroll
  for (int k = 0; k < kPFC; ++k) {
    const int i = t + k * NT, r = i / P;
    const unsigned o = (unsigned)(r * ldp + i - r * P) & 0xFFFFu;
    offc[k / 2] = k & 1 ? offc[k / 2] | (o << 16) : o;
  }

  const int RQ = Q > 0 ? min(NT / Q, VT) : 0;  // rows side by side (more would only lengthen the merge)
  const bool qthread = t < RQ * Q;
  const int q = qthread ? t % Q : 0, rq = qthread ? t / Q : 0;
  // Read once: loads inside the tile loop would follow the loop's stores (possible aliases) and wait for every
  // outstanding load, the next tile's prefetch included.
  const int q_ps = kA && qthread ? a.ps[q] : 0, q_pd = kA && qthread ? a.pd[q] : 0;
  // The thread's pattern edge's fills and RE normaliser, in registers for the whole pass: an LDS table of them would
  // take pass A (VT = 64, 24 pattern edges) just past the 40 KB that lets four blocks share a CU.
  double fF = 0.0, fR = 0.0, mR = 0.0, lR = 0.0;
  if (kA && qthread) {
    const QStat x = a.qs[q];
    fF = x.fillF, fR = x.fillR, mR = x.mRE, lR = x.lRE;
  }
  double vfmax = -kInf, vrmax = -kInf;
  int avf = -1, avr = -1;
  Lse lre = lse_empty(), lfe = lse_empty();

  Lse pacc[kPW];
#pragma unroll
  for (int pi = 0; pi < kPW; ++pi) pacc[pi] = lse_empty();
  // Lane -> (tile row, one of the wave's pattern vertices); psweep pattern vertices per step of the block.
  const int prow = kFull ? lane : lane & (VT - 1);
  const int pfirst = kFull ? wave : wave * (64 / VT) + lane / VT, psweep = kFull ? kVW : kVW * (64 / VT);

  for (int64_t tile = blk; tile < ntiles; tile += G) {
    const int64_t v0 = tile * VT;
    const int nv = (int)((a.n - v0) < VT ? (a.n - v0) : VT);
    __syncthreads();  // tables written (first tile) / previous tile consumed
    {
      const int cnt4 = nv * Qs / 4, cntc = nv * P;
#pragma unroll
      for (int k = 0; k < kPF4; ++k)
        if (t + k * NT < cnt4) {
          const int o = (off4 >> (16 * k)) & 0xFFFF;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            Fs[o + u] = pf[0][k][u];
            Vs[o + u] = pf[1][k][u];
            if (kA) {
              Ms[o + u] = pf[2][k][u];
              Ls[o + u] = pf[3][k][u];
            }
          }
        }
#pragma unroll
      for (int k = 0; k < kPFC; ++k)
        if (t + k * NT < cntc) Cs[(offc[k / 2] >> (16 * (k & 1))) & 0xFFFF] = pc[k];
      if (kMode == kModeOut && a.perm && t < nv) Prow[t] = pp;
    }
    __syncthreads();
    if (tile + G < ntiles) prefetch(tile + G);
    // One incidence's term in tile row prow.
    auto term = [&](const IncRec& rc, float x) __attribute__((always_inline)) {
      const double d = ((double)x - rc.m) - rc.l;
      return fmax(rc.fill, x == -INFINITY ? -kInf : d);
    };
    // p-phase.  Tiles of fewer than 64 rows form the sums in two steps, so that a pattern vertex with many incidences
    // (a hub) is spread over the block: kTerms incidences per lane, then the partial sums in order.
    if (!kFull && sums) {
      const int v1 = kMode == kModeOut ? soff[a.c0 + a.ncol] : nsum;
      for (int v = (kMode == kModeOut ? soff[a.c0] : 0) + pfirst; v < v1; v += psweep)
        if (prow < nv) {
          const int2 ks = tasks[v];
          IncRec rc[kTerms];
          float x[kTerms];
#pragma unroll
          for (int u = 0; u < kTerms; ++u) rc[u] = recs[min(ks.x + u, ks.y - 1)];
#pragma unroll
          for (int u = 0; u < kTerms; ++u) x[u] = Fs[prow * ldq + rc[u].col];
          double s = term(rc[0], x[0]);
#pragma unroll
          for (int u = 1; u < kTerms; ++u)
            if (ks.x + u < ks.y) s += term(rc[u], x[u]);
          Ps[v * VT + prow] = s;
        }
      __syncthreads();
    }
    // MU_pre of row prow and pattern vertex p.
    auto mu_pre = [&](int p) __attribute__((always_inline)) {
      double acc = -(double)Cs[prow * ldp + p];
      if (!sums) return acc;
      if (!kFull) {
        const int v1 = soff[p + 1];
#pragma unroll 4
        for (int v = soff[p]; v < v1; ++v) acc += Ps[v * VT + prow];
        return acc;
      }
      // kUnroll terms at a time, their LDS reads all in flight; the sum is taken in order.  (A term by itself waits for
      // its record, then for its value: about 200 cycles.)
      const int k1 = c_incoff[p + 1];
      int k = c_incoff[p];
      for (; k + kUnroll <= k1; k += kUnroll) {
        IncRec rc[kUnroll];
        float x[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) rc[u] = recs[k + u];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) x[u] = Fs[prow * ldq + rc[u].col];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) acc += term(rc[u], x[u]);
      }
      IncRec rc = recs[k];
      for (; k < k1; ++k) {
        const IncRec nx = recs[k + 1];  // in flight while this term is formed
        acc += term(rc, Fs[prow * ldq + rc.col]);
        rc = nx;
      }
      return acc;
    };
    if (kC) {
#pragma unroll
      for (int pi = 0; pi < kPW; ++pi) {
        if (psweep * pi >= P) break;
        const int p = pfirst + psweep * pi;
        if (p < P) lse_add(pacc[pi], prow < nv ? mu_pre(p) : -kInf);
      }
    } else {
      const int p1 = kMode == kModeOut ? a.c0 + a.ncol : P;
      for (int p = (kMode == kModeOut ? a.c0 : 0) + pfirst; p < p1; p += psweep)
        if (prow < nv) MUs[prow * ldm + p] = (mu_pre(p) - pmu[p]) - pmu[P + p];
    }
    if (kRows) {
      // The tile's rows go out whole: consecutive threads write consecutive columns of a row.
      __syncthreads();
      const int w = kMode == kModeOut ? a.ncol : P;
      for (int e = t; e < nv * w; e += NT) {
        const int r = e / w, c = e - r * w;
        if (kMode == kModeMU)
          a.mu_out[(v0 + r) * P + c] = MUs[r * ldm + c];
        else
          a.out[(int64_t)(a.perm ? Prow[r] : v0 + r) * w + c] = (float)MUs[r * ldm + a.c0 + c];
      }
    }
    if (kA) {
      __syncthreads();
      if (qthread) {
        for (int r = rq; r < nv; r += RQ) {
          const int64_t i = (v0 + r) * Qs + q;
          const float mo = Ms[r * ldq + q];
          const float lo = Ls[r * ldq + q];
          const double fm = fmax(fF, (double)Fs[r * ldq + q]);
          const float vfm = Vs[r * ldq + q];
          const double rm = fmax(fR, vfm == -INFINITY ? -kInf : ((double)vfm - mR) - lR);
          const double vf = MUs[r * ldm + q_pd] - fm;
          const double vr = MUs[r * ldm + q_ps] - rm;
          if (kArgMax) {
            if (vf > vfmax) {  // rows ascend within a thread, so the first maximum is the lowest vertex
              vfmax = vf;
              avf = (int)(v0 + r);
            }
            if (vr > vrmax) {
              vrmax = vr;
              avr = (int)(v0 + r);
            }
          } else {
            vfmax = fmax(vfmax, vf);
            vrmax = fmax(vrmax, vr);
          }
          // A vertex without out-edges keeps VFm = -inf (as filled in the prep), is no gathered source and adds no
          // edge term.
          if (mo != INFINITY) {
            const double xx = vf - (double)mo;
            a.VR[(v0 + r) * a.VRs + q] = (float)vr;
            // The row's padding columns too (never read), so that whole 128-byte lines are written.
            if (q < a.VRs - Q) a.VR[(v0 + r) * a.VRs + Q + q] = 0.f;
            a.VFm_out[i] = (float)xx;
            lse_add_finite(lre, xx + (double)lo);
            lse_add_finite(lfe, (vr - (double)mo) + (double)lo);
          }
        }
      }
    }
  }
  __syncthreads();

  // Block partials, merged in a fixed order: the maxima first (every thread of a column finds them, which saves barriers;
  // a field's values lie together: 1,000 vertices with 10/12 took 9.4 us with whole partials, 7.5 now; R-MAT 18 27.1, 25.9),
  // then every accumulator rescaled to them at once (one exponential each, in parallel), then the sums.
  if (kA) {
    double* mre = lds;  // [6][NT]: maxima of RE and FE, max VF, max VR, rescaled sums of RE and FE; then the vertices
    double *mfe = mre + NT, *xvf = mfe + NT, *xvr = xvf + NT, *tre = xvr + NT, *tfe = tre + NT;
    int *xaf = reinterpret_cast<int*>(tfe + NT), *xar = xaf + NT;
    if (qthread) {
      mre[t] = lre.m, mfe[t] = lfe.m;
      xvf[t] = vfmax, xvr[t] = vrmax;
      if (kArgMax) xaf[t] = avf, xar[t] = avr;
    }
    __syncthreads();
    double Mre = -kInf, Mfe = -kInf;
    if (qthread) {
#pragma unroll 4
      for (int r = 0; r < RQ; ++r) {
        Mre = fmax(Mre, mre[r * Q + q]);
        Mfe = fmax(Mfe, mfe[r * Q + q]);
      }
      tre[t] = lse_rescaled(lre, Mre);
      tfe[t] = lse_rescaled(lfe, Mfe);
    }
    __syncthreads();
    if (t < Q) {  // (q == t)
      QPart acc{-kInf, -kInf, Lse{Mre, 0.0}, Lse{Mfe, 0.0}, -1, -1};
      bool ore = false, ofe = false;
#pragma unroll 4
      for (int r = 0; r < RQ; ++r) {
        const int i = r * Q + t;
        lse_sum_step(acc.re.t, ore, tre[i]);
        lse_sum_step(acc.fe.t, ofe, tfe[i]);
        if (kArgMax) {
          argmax_merge(acc.vfmax, acc.avf, xvf[i], xaf[i]);
          argmax_merge(acc.vrmax, acc.avr, xvr[i], xar[i]);
        } else {
          acc.vfmax = fmax(acc.vfmax, xvf[i]);
          acc.vrmax = fmax(acc.vrmax, xvr[i]);
        }
      }
      a.qpart[t * (G + 1) + blk] = acc;
    }
  } else if (kC) {
#pragma unroll
    for (int pi = 0; pi < kPW; ++pi) {
      if (psweep * pi >= P) break;
      const int p = pfirst + psweep * pi;
      const Lse w = lanes_lse_merge(pacc[pi], VT);
      if (p < P && prow == 0) a.ppart[p * (G + 1) + blk] = w;
    }
  }
}

// Pass A runs 256-thread blocks (its register use), the lighter modes 512-thread blocks (measured at R-MAT 22).
// Pass A tiles whose CV rows fit 4 values per thread take the variant with the shorter CV prefetch: 120 instead of
// 132 VGPRs, 4 instead of 3 resident waves per SIMD.
constexpr int kNA = 256, kNO = 512;
static bool short_cv(const VertexArgs& a) { return a.VT * a.P <= kNA * 4; }

typedef void (*VertexKernel)(VertexArgs);

template <bool kFull>
static VertexKernel vertex_kernel_t(int mode, const VertexArgs& a) {
  switch (mode) {
    case kModeA:
      if (a.track_arg) return short_cv(a) ? k_vertex<kModeA, kFull, true, kNA, 4> : k_vertex<kModeA, kFull, true, kNA>;
      return short_cv(a) ? k_vertex<kModeA, kFull, false, kNA, 4> : k_vertex<kModeA, kFull, false, kNA>;
    case kModeC:
      return k_vertex<kModeC, kFull, false, kNO>;
    case kModeMU:
      return k_vertex<kModeMU, kFull, false, kNO>;
    default:
      return k_vertex<kModeOut, kFull, false, kNO>;
  }
}

// The kernel a pass launches, its block size and dynamic LDS bytes.
static VertexKernel vertex_kernel(int mode, const VertexArgs& a, int* nt, size_t* lds) {
  const size_t tiles = vertex_lds_bytes(mode, a.VT, a.P, a.Q, a.Qs, a.nsum);
  *nt = mode == kModeA ? kNA : kNO;
  *lds = mode == kModeA ? std::max(tiles, kNA * (6 * sizeof(double) + 2 * sizeof(int))) : tiles;
  return a.VT == 64 ? vertex_kernel_t<true>(mode, a) : vertex_kernel_t<false>(mode, a);
}

void launch_vertex(int mode, const VertexArgs& a, int nblocks, hipStream_t st) {
  int nt = 0;
  size_t lds = 0;
  const VertexKernel k = vertex_kernel(mode, a, &nt, &lds);
  VertexArgs arg = a;
  void* args[] = {&arg};
  const int extra = mode == kModeA || mode == kModeC ? 1 : 0;  // the isolated vertices' block
  (void)hipLaunchKernel(reinterpret_cast<const void*>(k), dim3(nblocks + extra), dim3(nt), args, lds, st);
}

// Tile blocks of a vertex pass resident at once on the device (CUs x blocks per CU at the pass's registers and LDS,
// less the isolated vertices' block).
int vertex_resident_blocks(int mode, const VertexArgs& a) {
  int dev = 0, cus = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  int nt = 0;
  size_t lds = 0;
  const VertexKernel k = vertex_kernel(mode, a, &nt, &lds);
  const hipError_t e =
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, reinterpret_cast<const void*>(k), nt, lds);
  const int extra = mode == kModeA || mode == kModeC ? 1 : 0;
  return e == hipSuccess ? cus * std::max(per, 1) - extra : 0;
}

__global__ void k_gather_rows(int64_t n, int ncol, const int* __restrict__ perm, const float* __restrict__ in,
                              float* __restrict__ out) {
  const int64_t total = n * ncol;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / ncol, c = i - r * ncol;
    out[i] = in[(int64_t)perm[r] * ncol + c];
  }
}

void launch_gather_rows(int64_t n, int ncol, const int* perm, const float* in, float* out, hipStream_t st) {
  if (n * ncol == 0) return;
  const int blocks = (int)std::min<int64_t>((n * ncol + 255) / 256, 1 << 16);
  hipLaunchKernelGGL(k_gather_rows, dim3(blocks), dim3(256), 0, st, n, ncol, perm, in, out);
}

}  // namespace ac
