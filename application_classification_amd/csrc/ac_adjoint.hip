// Adjoint of the matcher (no counterpart in the reference): gradients of a loss on the output log-probabilities with
// respect to the per-dimension cdist weights, by reverse mode through the prep and every iteration.
//
// One iteration maps the state S_i = (MU_i, FMax_i, RMax_i) to S_{i+1} (src/main.cu:160-245):
//   VF = MU_i[pd] - FMax_i,  VR = MU_i[ps] - RMax_i,  fillR = max_v VF,  fillF = max_v VR
//   FMax_{i+1}[v] = max(fillF, max_{e->v} (VR[src e] - CE_e) - LSE_FE),  LSE_FE = log sum_e exp(VR[src e] - CE_e)
//   RMax_{i+1}[v] = max(fillR, max_{e: src=v} (VF[v] - CE_e) - LSE_RE)
//   MU_{i+1} = LSM_v(-CV + sum_{q: pd=p} FMax_{i+1} + sum_{q: ps=p} RMax_{i+1})
// Its adjoint, given (gMU, gFMax, gRMax) of S_{i+1}:
//   gZ = gMU - exp(MU_{i+1}) colsum_v(gMU)                        (log-softmax Jacobian, FP32)
//   gCV -= gZ;  gF = gFMax + gZ[pd],  gR = gRMax + gZ[ps]
//   max subgradients: to the recorded argmax in-edge (FMax) / the minimum-cost out-edge (RMax) when the edge term
//   wins, else to the fill, whose own subgradient goes to the recorded argmax vertex;
//   log-sum-exp over edges: sum_e exp(FE_e) routes -S_F = -sum_v gE_F to every edge; its vertex part is the closed
//   form  sum_{e: src=v} exp(VR[v] - CE_e - LSE_FE) = exp(VR[v] - LSE_FE - minCEo[v] + lsO[v]), and its edge-cost
//   part S_F exp(VR[src] - LSE_FE) exp(-CE_e) is accumulated per (src, q) in cD, so that the final gradient of every
//   edge cost is  gCE_e = (sparse argmax terms) + (cD[src e] + c_q) exp(-CE_e), formed once at the end.
// The weight gradients are then  dL/dw_k = sum gC / (2 C) (x_k - p_k)^2  over vertex and edge costs.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>

#include "ac_adjoint.hpp"

namespace ac {

namespace {

constexpr double kInf = __builtin_huge_val();
typedef float f4v __attribute__((ext_vector_type(4)));

}  // namespace

// Column sums of X[n][C] (C <= 256): per-block partials in a fixed order.
__global__ __launch_bounds__(256) void k_colsum(int64_t n, int C, const float* __restrict__ X, double* __restrict__ part) {
  __shared__ double red[256];
  const int t = threadIdx.x, RC = 256 / C;
  const bool active = t < RC * C;
  const int c = active ? t % C : 0;
  double s = 0.0;
  if (active)
    for (int64_t v = (int64_t)blockIdx.x * RC + t / C; v < n; v += (int64_t)gridDim.x * RC) s += (double)X[v * C + c];
  red[t] = s;
  __syncthreads();
  if (t < C) {
    double a = 0.0;
    for (int r = 0; r < RC; ++r) a += red[r * C + t];
    part[(int64_t)t * gridDim.x + blockIdx.x] = a;
  }
}

// out[c] = sum over parts of part[b * sb + c * sc].
__global__ __launch_bounds__(256) void k_sum_parts(int nparts, int64_t sb, int64_t sc, const double* __restrict__ part,
                                                   double* __restrict__ out) {
  // One block per column: lane l sums partials l, l + 256, ... in order (eight loads in flight before the adds), then
  // a fixed tree over the lanes.  The order is the same on every call.
  __shared__ double red[4];
  const int t = threadIdx.x, c = blockIdx.x;
  double a = 0.0;
  for (int b0 = t; b0 < nparts; b0 += 8 * 256) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int b = b0 + u * 256;
      v[u] = part[(b < nparts ? b : nparts - 1) * sb + c * sc];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (b0 + u * 256 < nparts) a += v[u];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
  if ((t & 63) == 0) red[t >> 6] = a;
  __syncthreads();
  if (t == 0) out[c] = ((red[0] + red[1]) + red[2]) + red[3];
}

// Log-softmax Jacobian of MU = LSM_v(Z): gMU <- gZ = gMU - exp(MU) colsum(gMU); gCV -= gZ.
__global__ __launch_bounds__(256) void k_bwd_out(int64_t total, int P, const double* __restrict__ MU,
                                                 const double* __restrict__ colsum, float* __restrict__ gMU,
                                                 float* __restrict__ gCV) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const float gz = gMU[i] - __expf((float)MU[i]) * (float)colsum[i % P];
    gMU[i] = gz;
    gCV[i] -= gz;
  }
}

// Max-subgradient routing of FMax / RMax of state S (thread per (v, q), q fixed per thread).  gF = -gVF + gZ[pd],
// gR = -gVR + gZ[ps], where gVF / gVR are the next state's (the step processed before this one; zero at the
// first): the gradients of this state's FMax / RMax through the next step's inputs.  The edge term takes the
// gradient where it is strictly above the fill.  Per-block partials part[4][Q][blocks]: sum gE_F, sum gE_R, fill gradient
// of fillF, of fillR.  gmax (nullable) receives the largest |gE_F| (as float bits, an atomic maximum: exact and
// order-free), which sets the fixed-point scale of the FMax edge terms' source sums.  gERsum accumulates
// gE_R per (v, q) over the steps: the RMax rows AO are the same in every step, so their edge terms are applied once.
// kOut: k_bwd_out's step for the rows of a tile first (T rows; T P <= kRouteTile), its gZ kept in LDS: gZ is read here
// only, and in a launch of its own it was written and read back.  Isolated vertices have no edge terms (FMaxN and VFm hold
// -inf), so their rows of S are not read, nor, with kOut, their zero rows of gEF and gER written.  Bound by its streams:
// R-MAT 18 with 12/16, a step's two launches 43 us, now 33.
constexpr int kRouteTile = 2048;
template <bool kOut>
__global__ __launch_bounds__(256) void k_bwd_route(BwdGraph G, BwdState S, const double* __restrict__ MU,
                                                   const double* __restrict__ colsum, const float* __restrict__ gMU,
                                                   float* __restrict__ gCV, const float* __restrict__ gVF,
                                                   const float* __restrict__ gVR, float* __restrict__ gEF,
                                                   float* __restrict__ gER, unsigned* __restrict__ gmax,
                                                   float* __restrict__ gERsum, double* __restrict__ part, int T) {
  __shared__ double red[256][4];
  __shared__ float gz[kOut ? kRouteTile : 1];
  __shared__ unsigned bmax;
  const int t = threadIdx.x, Q = G.Q, P = G.P, RQ = 256 / Q;
  if (t == 0) bmax = 0u;
  const bool active = t < RQ * Q;
  const int q = active ? t % Q : 0, rq = active ? t / Q : 0;
  double sF = 0.0, sR = 0.0, fF = 0.0, fR = 0.0;
  unsigned mx = 0u;
  const int pdq = G.pd[q], psq = G.ps[q];
  const QStat s = S.qs[q];
  for (int64_t v0 = (int64_t)blockIdx.x * T; v0 < G.n; v0 += (int64_t)gridDim.x * T) {
    const int nv = (int)min((int64_t)T, G.n - v0);
    __syncthreads();
    if (kOut) {
      for (int e = t; e < nv * P; e += 256) {
        const int64_t i = v0 * P + e;
        const float g = gMU[i] - __expf((float)MU[i]) * (float)colsum[e % P];
        gz[e] = g;
        gCV[i] -= g;
      }
      __syncthreads();
    }
    if (!active) continue;
#pragma unroll 2
    for (int r = rq; r < nv; r += RQ) {
      const int64_t i = (v0 + r) * G.Qs + q;
      float gF = -gVF[i], gR = -gVR[i];
      if (kOut) {
        gF += gz[r * P + pdq];
        gR += gz[r * P + psq];
      }
      if (v0 + r >= G.n_act) {
        fF += gF;
        fR += gR;
        if (!kOut) gEF[i] = gER[i] = 0.f;
        continue;
      }
      const float vfm = S.VFm[i];
      const bool eF = (double)S.FMaxN[i] > s.fillF;
      const bool eR = (vfm == -INFINITY ? -kInf : ((double)vfm - s.mRE) - s.lRE) > s.fillR;
      gEF[i] = eF ? gF : 0.f;
      gER[i] = eR ? gR : 0.f;
      if (eF) mx = max(mx, __float_as_uint(fabsf(gF)));
      if (eR && gR != 0.f) gERsum[i] += gR;
      if (eF) sF += gF; else fF += gF;
      if (eR) sR += gR; else fR += gR;
    }
  }
  if (gmax && mx) atomicMax(&bmax, mx);
  red[t][0] = sF;
  red[t][1] = sR;
  red[t][2] = fF;
  red[t][3] = fR;
  __syncthreads();
  if (gmax && t == 0 && bmax) atomicMax(gmax, bmax);
  if (t < Q)
    for (int k = 0; k < 4; ++k) {
      double a = 0.0;
      for (int r = 0; r < RQ; ++r) a += red[r * Q + t][k];
      part[((int64_t)k * Q + t) * gridDim.x + blockIdx.x] = a;
    }
}

// The fixed-point scale of the FMax edge terms' source sums: 2^(39 - shift - e) for the largest |gE_F| in
// [2^e, 2^(e+1)), so every term is below 2^(40 - shift) in magnitude.  A source's sum has at most its out-degree of
// terms, and shift (BwdGraph::fix_shift) leaves room for the graph's largest out-degree: up to 2^(23 + shift) terms
// stay inside int64.  A power of two, so scaling is exact and only the rounding to an integer (at 2^-(40 - shift)
// of the largest term) loses anything.
__device__ __forceinline__ int fix_exponent(unsigned gmax_bits, int shift) {
  const int e = (int)((gmax_bits >> 23) & 0xFFu) - 127;  // subnormal maxima: e = -127, a larger scale than needed
  return 39 - shift - max(-126, min(e, 127));
}

// The FMax edge term of (v, q), where it carries gradient gE = gEF[v][q] != 0: its recorded row FA[v][q] receives
// -gE in gCE (one term per (row, q) and step, so the float atomic adds the same two values in the same order as a
// plain update), and the row's source accumulates gE in the fixed-point sum gVRfix[src][q] (integer additions: exact,
// so the sum does not depend on their order).  FA rows exist only where the walk recorded a maximum (vertices with
// in-edges, bundles not pruned); a nonzero gradient implies one, and the row is bounds-checked besides.
__device__ __forceinline__ void fmax_edge_term(int64_t o, int q, int Qs, float ge, const int* __restrict__ FA,
                                               const int* __restrict__ bsrc, int64_t brows, float* __restrict__ gCE,
                                               unsigned long long* __restrict__ gVRfix, double fscale) {
  const int row = FA[o];
  if (row < 0 || row >= brows) return;
  unsafeAtomicAdd(gCE + (int64_t)row * Qs + q, -ge);
  if (gVRfix) {
    const int64_t src = bsrc[row] & ~kNewVertex;
    atomicAdd(gVRfix + src * Qs + q, (unsigned long long)__double2ll_rn((double)ge * fscale));
  }
}

// The prep's FMax edge terms (no source sums: the prep state has no VR).
__global__ void k_bwd_fscatter(int64_t n, int Q, int Qs, const float* __restrict__ gEF, const int* __restrict__ FA,
                               const int* __restrict__ bsrc, int64_t brows, float* __restrict__ gCE) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n * Qs; i += (int64_t)gridDim.x * blockDim.x) {
    const int q = (int)(i % Qs);
    if (q >= Q) continue;
    const float ge = gEF[i];
    if (ge != 0.f) fmax_edge_term(i, q, Qs, ge, FA, bsrc, brows, gCE, nullptr, 0.0);
  }
}

// Input side of one iteration (state S = S_i, scalars qs1 of S_{i+1}; red4 = {S_F, S_R, gfillF, gfillR}[Q]):
//   gVR = -S_F exp(VR - LSE_FE - minCEo + lsO) + [v = argmax VR] gfillF
//   gVF = gE_R - S_R exp(VF - LSE_RE - minCEo + lsO) + [v = argmax VF] gfillR
//   cD += S_F exp(VR - LSE_FE) + S_R exp(VF - LSE_RE)            (vertices with out-edges; FP64)
// and the FMax edge terms of the step (fmax_edge_term; FE: the step's gE_F, argmax rows and fixed-point scale), whose
// source sums go to gVRfix and are added to gVR by the vertex kernel that follows.
// A thread keeps its pattern edge and takes kIn vertices at a time, all their loads in flight.  Isolated vertices have no
// terms but those of the maxima's vertices.  Bound by its streams (14 values of 4 or 8 bytes per vertex and pattern edge)
// and three FP64 exponentials: R-MAT 18 with 12/16 in 51 us (66 with a flat index
// and the scalars read for every element; 57 with 8192 blocks, whose prologues follow each other).
constexpr int kIn = 2;
__global__ __launch_bounds__(256, 4) void k_bwd_in(BwdGraph G, BwdState S, const double* __restrict__ MU,
                                                const QStat* __restrict__ qs1, const double* __restrict__ red4,
                                                const float* __restrict__ gER, float* __restrict__ gVR,
                                                float* __restrict__ gVF, double* __restrict__ cD, FmaxTerms FE) {
  const int Q = G.Q, RQ = 256 / Q, t = threadIdx.x;
  if (t >= RQ * Q) return;
  const double fscale = ldexp(1.0, fix_exponent(*FE.gmax, G.fix_shift));
  const int q = t % Q, pdq = G.pd[q], psq = G.ps[q];
  const QStat s0 = S.qs[q], s1 = qs1[q];
  const double SF = red4[q], SR = red4[Q + q], gfF = red4[2 * Q + q], gfR = red4[3 * Q + q];
  const double lF = s1.mFE + s1.lFE, lR = s1.mRE + s1.lRE;
  const int64_t step = (int64_t)gridDim.x * RQ;
  for (int64_t v0 = (int64_t)blockIdx.x * RQ + t / Q; v0 < G.n; v0 += kIn * step) {
    double muF[kIn], muR[kIn], cd[kIn];
    float F[kIn], V[kIn], mo[kIn], ls[kIn], er[kIn], ge[kIn];
#pragma unroll
    for (int u = 0; u < kIn; ++u) {
      const int64_t v = v0 + u * step;
      mo[u] = INFINITY;
      er[u] = ge[u] = 0.f;
      if (v < G.n_act) {
        const int64_t o = v * G.Qs + q;
        mo[u] = G.minCEo[o];
        ls[u] = G.lsO[o];
        muF[u] = MU[v * G.P + pdq];
        muR[u] = MU[v * G.P + psq];
        F[u] = S.FMaxN[o];
        V[u] = S.VFm[o];
        cd[u] = cD[o];
        er[u] = gER[o];
        ge[u] = FE.gEF[o];
      }
    }
#pragma unroll
    for (int u = 0; u < kIn; ++u) {
      const int64_t v = v0 + u * step;
      if (v >= G.n) break;
      const int64_t o = v * G.Qs + q;
      double gvr = 0.0, gvf = (double)er[u];
      if (mo[u] != INFINITY) {
        const double VF = muF[u] - fmax(s0.fillF, (double)F[u]);
        const double VR = muR[u] - fmax(s0.fillR, V[u] == -INFINITY ? -kInf : ((double)V[u] - s0.mRE) - s0.lRE);
        const double eF = exp(VR - lF), eR = exp(VF - lR);
        const double wo = exp((double)ls[u] - (double)mo[u]);
        gvr -= SF * eF * wo;
        gvf -= SR * eR * wo;
        cD[o] = cd[u] + (SF * eF + SR * eR);
      }
      if (v == s1.vF) gvr += gfF;
      if (v == s1.vR) gvf += gfR;
      gVR[o] = (float)gvr;
      gVF[o] = (float)gvf;
      if (ge[u] != 0.f) fmax_edge_term(o, q, G.Qs, ge[u], FE.FA, FE.bsrc, FE.brows, FE.gCE, FE.gVRfix, fscale);
    }
  }
}

// The vertex side of a step back, one tile of T vertices per block iteration:
//   1. gVR[v][q] += gVRfix[v][q] 2^-k, the fixed-point sums of the step's FMax edge terms (where nonzero; the
//      accumulator is cleared for the next step), staged with gVF in LDS, four pattern edges to a thread;
//   2. gMU[v][p] = sum over the incidences of p (ascending q) of gVF (q ends at p) or gVR (q starts at p), and the thread's
//      (fixed p) part of the column sum of gMU, in FP64;
//   3. per-block partial column sums: part[p][b].
// The input state's FMax / RMax gradients are -gVF / -gVR, which k_bwd_route of the next step back reads directly.
// Bound by its streams: R-MAT 18 with 12/16 in 22.4 us (26.7 with single values staged and a column's sum left to one
// thread); by its tiles' latency on small graphs, hence
// short ones there (1,000 vertices, 10/12: 7.1 -> 3.8 us).
__global__ __launch_bounds__(256) void k_bwd_vtx(BwdGraph G, float* __restrict__ gVR, const float* __restrict__ gVF,
                                                 unsigned long long* __restrict__ gVRfix,
                                                 const unsigned* __restrict__ gmax, float* __restrict__ gMU,
                                                 double* __restrict__ part, int T) {
  typedef unsigned long long u4v __attribute__((ext_vector_type(4)));
  extern __shared__ float vsh[];  // [T][Qs] gVR, [T][Qs] gVF, then the incidence lists
  __shared__ double cs[256];
  const int Qs = G.Qs, P = G.P, t = threadIdx.x;
  float* tR = vsh;
  float* tF = tR + T * Qs;
  int* ioff = reinterpret_cast<int*>(tF + T * Qs);
  int* iinc = ioff + (P + 1);
  const int ninc = G.inc_off[P];
  for (int k = t; k <= P; k += 256) ioff[k] = G.inc_off[k];
  for (int k = t; k < ninc; k += 256) iinc[k] = G.inc[k];
  const double inv = ldexp(1.0, -fix_exponent(*gmax, G.fix_shift));
  const int64_t act4 = G.n_act * Qs / 4;  // isolated vertices are no edge's source
  const int RP = 256 / P, p = t % P, rp = t / P;
  double col = 0.0;
  for (int64_t v0 = (int64_t)blockIdx.x * T; v0 < G.n; v0 += (int64_t)gridDim.x * T) {
    const int nv = (int)min((int64_t)T, G.n - v0);
    __syncthreads();  // the lists are written (first tile) / the last tile is read
    for (int e = t; e < nv * Qs / 4; e += 256) {
      const int64_t o = v0 * Qs / 4 + e;
      f4v r = reinterpret_cast<const f4v*>(gVR)[o];
      u4v f = {0, 0, 0, 0};
      if (o < act4) f = reinterpret_cast<const u4v*>(gVRfix)[o];
      reinterpret_cast<f4v*>(tF)[e] = reinterpret_cast<const f4v*>(gVF)[o];
      if ((f[0] | f[1] | f[2] | f[3]) != 0) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (f[u] != 0) r[u] = (float)((double)r[u] + (double)(long long)f[u] * inv);
        reinterpret_cast<f4v*>(gVR)[o] = r;
        reinterpret_cast<u4v*>(gVRfix)[o] = u4v{0, 0, 0, 0};
      }
      reinterpret_cast<f4v*>(tR)[e] = r;
    }
    __syncthreads();
    if (rp < RP)
      for (int vl = rp; vl < nv; vl += RP) {
        float a = 0.f;
        for (int k = ioff[p]; k < ioff[p + 1]; ++k) {
          const int code = iinc[k];
          a += (code & 1) ? tR[vl * Qs + (code >> 1)] : tF[vl * Qs + (code >> 1)];
        }
        gMU[(v0 + vl) * P + p] = a;
        col += (double)a;
      }
  }
  cs[t] = col;
  __syncthreads();
  if (t < P) {
    for (int r = 1; r < RP; ++r) col += cs[r * P + t];
    part[(int64_t)t * gridDim.x + blockIdx.x] = col;
  }
}

// Fill subgradients of the prep state go to the argmax of MU0 = LSM(-CV) of the source / destination pattern vertex:
// fillF_q = max_v MU0[v][ps q], fillR_q = max_v MU0[v][pd q].  A thread per pattern vertex, its incidences in order.  And
// the prep's part of the edge costs' gradients, cq[q] = (S_F + S_R) exp(-LSE0), a thread per pattern edge (on the host it
// took a copy back, a wait and a copy; with the wait between the two weight sums, a training step at 1,000 vertices took
// 1,439 us in place of 1,343).
__global__ __launch_bounds__(256) void k_bwd_prep_fill(BwdGraph G, const double* __restrict__ red4,
                                                       const QStat* __restrict__ qs0, const int* __restrict__ am0,
                                                       float* __restrict__ gMU, double* __restrict__ cq) {
  const int t = threadIdx.x, Q = G.Q;
  if (t < Q) {
    const double lse0 = qs0[t].mFE + qs0[t].lFE;
    cq[t] = lse0 > -kInf && lse0 < kInf ? (red4[t] + red4[Q + t]) * exp(-lse0) : 0.0;
  }
  if (t < G.P && G.inc_off[t] < G.inc_off[t + 1]) {
    float a = gMU[(int64_t)am0[t] * G.P + t];
    for (int k = G.inc_off[t]; k < G.inc_off[t + 1]; ++k) {
      const int code = G.inc[k], q = code >> 1;
      a += (float)red4[((code & 1) ? 2 : 3) * Q + q];
    }
    gMU[(int64_t)am0[t] * G.P + t] = a;
  }
}

// Per column p of CV[n][P]: the lowest row of the minimum (the argmax of MU0 = LSM(-CV)).  Block partials.
__global__ __launch_bounds__(256) void k_col_argmin(int64_t n, int P, const float* __restrict__ CV, float* __restrict__ pv,
                                                    int* __restrict__ pi) {
  __shared__ float rv[256];
  __shared__ int ri[256];
  const int t = threadIdx.x, RP = 256 / P;
  const bool active = t < RP * P;
  const int p = active ? t % P : 0;
  float best = INFINITY;
  int bi = INT_MAX;
  if (active)
    for (int64_t v = (int64_t)blockIdx.x * RP + t / P; v < n; v += (int64_t)gridDim.x * RP) {
      const float x = CV[v * P + p];
      if (x < best) {
        best = x;
        bi = (int)v;
      }
    }
  rv[t] = best;
  ri[t] = bi;
  __syncthreads();
  if (t < P) {
    for (int r = 1; r < RP; ++r) {
      const float x = rv[r * P + t];
      const int xi = ri[r * P + t];
      if (x < best || (x == best && xi < bi)) {
        best = x;
        bi = xi;
      }
    }
    pv[(int64_t)blockIdx.x * P + t] = best;
    pi[(int64_t)blockIdx.x * P + t] = bi;
  }
}

// One block per column: the least of its blocks' minima, the lowest row on ties.
__global__ __launch_bounds__(256) void k_col_argmin_final(int nparts, int P, const float* __restrict__ pv,
                                                          const int* __restrict__ pi, int* __restrict__ am) {
  __shared__ float rv[256];
  __shared__ int ri[256];
  const int p = blockIdx.x, t = threadIdx.x;
  float best = INFINITY;
  int bi = INT_MAX;
  for (int b = t; b < nparts; b += 256) {
    const float x = pv[(int64_t)b * P + p];
    const int xi = pi[(int64_t)b * P + p];
    if (x < best || (x == best && xi < bi)) {
      best = x;
      bi = xi;
    }
  }
  rv[t] = best;
  ri[t] = bi;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w && (rv[t + w] < rv[t] || (rv[t + w] == rv[t] && ri[t + w] < ri[t]))) {
      rv[t] = rv[t + w];
      ri[t] = ri[t + w];
    }
    __syncthreads();
  }
  if (t == 0) am[p] = ri[0] == INT_MAX ? 0 : ri[0];
}

// Edge-cost gradients divided by twice the cost: G[row][q] = (gCE + (cD[src] + cq) exp(-CE)) / (2 CE), 0 for
// padding rows and zero costs (d sqrt(s) / ds is unbounded at 0; such a pair contributes nothing here).
// A group of Qs/4 lanes per row, four pattern edges to a lane: 16- and 32-byte accesses, no index division per element.
__global__ __launch_bounds__(256) void k_bwd_edge_coef(int64_t nrows, int Q, int Qs, const int* __restrict__ beid,
                                                       const int* __restrict__ bsrc, const float* __restrict__ CE,
                                                       const double* __restrict__ cD, const double* __restrict__ cq,
                                                       float* __restrict__ G) {
  const int L4 = Qs / 4, R = 256 / L4, r = threadIdx.x / L4, j = threadIdx.x - r * L4;
  if (r >= R) return;
  double c[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) c[u] = 4 * j + u < Q ? cq[4 * j + u] : 0.0;
  for (int64_t row = (int64_t)blockIdx.x * R + r; row < nrows; row += (int64_t)gridDim.x * R) {
    const int64_t o = row * L4 + j;
    f4v out = {0.f, 0.f, 0.f, 0.f};
    if (beid[row] >= 0) {
      const f4v ce4 = reinterpret_cast<const f4v*>(CE)[o], g4 = reinterpret_cast<const f4v*>(G)[o];
      const double4 d4 = reinterpret_cast<const double4*>(cD)[(int64_t)(bsrc[row] & ~kNewVertex) * L4 + j];
      const double dd[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double ce = (double)ce4[u];
        if (4 * j + u < Q && ce > 0.0 && ce != kInf) {
          const double g = (double)g4[u] + (dd[u] + c[u]) * exp(-ce);
          out[u] = (float)(g / (2.0 * ce));
        }
      }
    }
    reinterpret_cast<f4v*>(G)[o] = out;
  }
}

// Vertex-cost gradients divided by twice the cost (in place): G = gCV / (2 CV), 0 where CV = 0.
__global__ void k_bwd_vertex_coef(int64_t total, const float* __restrict__ CV, float* __restrict__ G) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const float c = CV[i];
    G[i] = c > 0.f ? G[i] / (2.f * c) : 0.f;
  }
}

// Outer-product sums over rows, for q < K, k < dim:  A[q][k] = sum_r G[r][q] x_r[k]^2,  B[q][k] = sum_r G[r][q]
// x_r[k],  C[q] = sum_r G[r][q],  x_r = feats[idx[r]] (rows with idx < 0 skipped), one block partial each.
// For the (q, k) block [q0, q0 + 16 NQT) x [k0, k0 + 16 NKT) they are GEMMs over the rows on FP64 matrix cores
// (v_mfma_f64_16x16x4f64, four rows per step).  A-operand lane
// i + 16k holds G[row k][q0 + i], B-operand lane j + 16k holds x[row k][k0 + j] (or its square), and D[4r +
// lane/16][lane%16] sits in register r.  Products of floats are exact in FP64; the sums are FP64.  The block's four
// waves are summed in order.
typedef double d4v __attribute__((ext_vector_type(4)));
template <int NQT, int NKT>
__global__ __launch_bounds__(256) void k_outer_mfma(int64_t nrows, const int* __restrict__ idx,
                                                    const float* __restrict__ feats, int dim,
                                                    const float* __restrict__ G, int Gs, int K, int q0, int k0,
                                                    double* __restrict__ part) {
  __shared__ double red[3][64][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = lane & 15, kr = lane >> 4;
  d4v accA[NQT][NKT], accB[NQT][NKT];
#pragma unroll
  for (int a = 0; a < NQT; ++a)
#pragma unroll
    for (int b = 0; b < NKT; ++b) accA[a][b] = accB[a][b] = d4v{0.0, 0.0, 0.0, 0.0};
  double cs[NQT];
#pragma unroll
  for (int a = 0; a < NQT; ++a) cs[a] = 0.0;
  // Steps of kOS x 4 rows, software-pipelined: the raw values of the next step are loaded while the current one
  // runs on the matrix cores, and the row ids one step earlier still, so that every load of a step issues at once.
  // All loads use valid (clamped) addresses and write each register once; the values that lie past K or dim or
  // belong to no row are zeroed when they are converted, so the loads stay in flight until then.
  constexpr int kOS = 4;
  const int64_t stride = (int64_t)gridDim.x * 4 * (4 * kOS);
  float gf[kOS][NQT], xf[kOS][NKT];
  int64_t srcl[kOS];  // source rows of the loaded step (-1: none)
  int sid[kOS];       // raw ids of the step after it
  auto load_ids = [&](int64_t r0, int* sv) {
#pragma unroll
    for (int h = 0; h < kOS; ++h) {
      const int64_t row = r0 + 4 * h + kr;
      sv[h] = idx[row < nrows ? row : nrows - 1];
    }
  };
  auto src_of = [&](int64_t r0, int h, int raw) -> int64_t {
    const int64_t row = r0 + 4 * h + kr;
    return row < nrows ? (int64_t)raw : -1;
  };
  auto load = [&](int64_t r0) {
#pragma unroll
    for (int h = 0; h < kOS; ++h) {
      const int64_t row = r0 + 4 * h + kr;
      const int64_t rc = row < nrows ? row : nrows - 1, sc = srcl[h] >= 0 ? srcl[h] : 0;
#pragma unroll
      for (int a = 0; a < NQT; ++a) {
        const int q = q0 + 16 * a + i;
        gf[h][a] = G[rc * Gs + (q < K ? q : K - 1)];
      }
#pragma unroll
      for (int b = 0; b < NKT; ++b) {
        const int k = k0 + 16 * b + i;
        xf[h][b] = feats[sc * dim + (k < dim ? k : dim - 1)];
      }
    }
  };
  int64_t r0 = ((int64_t)blockIdx.x * 4 + wave) * (4 * kOS);
  if (r0 < nrows) {
    int s0[kOS];
    load_ids(r0, s0);
#pragma unroll
    for (int h = 0; h < kOS; ++h) srcl[h] = src_of(r0, h, s0[h]);
    load(r0);
    load_ids(r0 + stride, sid);
  }
  for (; r0 < nrows; r0 += stride) {
    double g[kOS][NQT], x[kOS][NKT];
#pragma unroll
    for (int h = 0; h < kOS; ++h) {
      const bool ok = srcl[h] >= 0;
#pragma unroll
      for (int a = 0; a < NQT; ++a) g[h][a] = (ok && q0 + 16 * a + i < K) ? (double)gf[h][a] : 0.0;
#pragma unroll
      for (int b = 0; b < NKT; ++b) x[h][b] = (ok && k0 + 16 * b + i < dim) ? (double)xf[h][b] : 0.0;
    }
    // The next step's loads are issued unconditionally (past the last step they read clamped, valid rows and are
    // never used), so that no branch separates them from the loop back-edge.
#pragma unroll
    for (int h = 0; h < kOS; ++h) {
      int raw = sid[h];
      asm volatile("" : "+v"(raw));  // an empty register barrier: the id is first needed here
      srcl[h] = src_of(r0 + stride, h, raw);
    }
    load(r0 + stride);
    load_ids(r0 + 2 * stride, sid);
#pragma unroll
    for (int h = 0; h < kOS; ++h)
#pragma unroll
      for (int a = 0; a < NQT; ++a) {
        cs[a] += g[h][a];
#pragma unroll
        for (int b = 0; b < NKT; ++b) {
          accB[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(g[h][a], x[h][b], accB[a][b], 0, 0, 0);
          accA[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(g[h][a], x[h][b] * x[h][b], accA[a][b], 0, 0, 0);
        }
      }
  }
  // C: the four row slots of each column, then the waves.
#pragma unroll
  for (int a = 0; a < NQT; ++a) {
    cs[a] += __shfl_xor(cs[a], 16, 64);
    cs[a] += __shfl_xor(cs[a], 32, 64);
  }
  double* out = part + (int64_t)blockIdx.x * (2 * (int64_t)K * dim + K);
  auto block_sum = [&](d4v v) {
    __syncthreads();
    if (wave > 0)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave - 1][lane][r] = v[r];
    __syncthreads();
    if (wave == 0)
      for (int w = 0; w < 3; ++w)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] += red[w][lane][r];
    return v;
  };
#pragma unroll
  for (int a = 0; a < NQT; ++a)
#pragma unroll
    for (int b = 0; b < NKT; ++b)
#pragma unroll
      for (int which = 0; which < 2; ++which) {
        const d4v v = block_sum(which ? accB[a][b] : accA[a][b]);
        if (wave == 0)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int q = q0 + 16 * a + 4 * r + kr, k = k0 + 16 * b + i;
            if (q < K && k < dim) out[(which ? (int64_t)K * dim : 0) + (int64_t)q * dim + k] = v[r];
          }
      }
  if (k0 == 0)
#pragma unroll
    for (int a = 0; a < NQT; ++a) {
      const d4v v = block_sum(d4v{cs[a], 0.0, 0.0, 0.0});
      const int q = q0 + 16 * a + i;
      if (wave == 0 && kr == 0 && q < K) out[2 * (int64_t)K * dim + q] = v[0];
    }
}

// ---------------------------------------------------------------------------------------------------------------
// Launchers.

static int grid_for(int64_t total) { return (int)std::max<int64_t>(1, std::min<int64_t>((total + 255) / 256, 1 << 15)); }

// by_column: partials [C][nparts] (a column's together: whole lines to a block), else [nparts][C].
void launch_sum_parts(int nparts, int C, const double* part, double* out, bool by_column, hipStream_t st) {
  if (C == 0) return;
  hipLaunchKernelGGL(k_sum_parts, dim3(C), dim3(256), 0, st, nparts, by_column ? (int64_t)1 : (int64_t)C,
                     by_column ? (int64_t)nparts : (int64_t)1, part, out);
}

void launch_colsum(int64_t n, int C, const float* X, double* part, int nparts, double* out, hipStream_t st) {
  if (C == 0) return;
  hipLaunchKernelGGL(k_colsum, dim3(nparts), dim3(256), 0, st, n, C, X, part);
  launch_sum_parts(nparts, C, part, out, true, st);
}

void launch_bwd_out(const BwdGraph& G, const double* MU, const double* colsum, float* gMU, float* gCV, hipStream_t st) {
  hipLaunchKernelGGL(k_bwd_out, dim3(grid_for(G.n * G.P)), dim3(256), 0, st, G.n * G.P, G.P, MU, colsum, gMU, gCV);
}

void launch_bwd_route(const BwdGraph& G, const BwdState& S, const double* MU, const double* colsum, float* gMU,
                      float* gCV, const float* gVF, const float* gVR, float* gEF, float* gER, unsigned* gmax,
                      float* gERsum, double* part, int nparts, double* red4, hipStream_t st) {
  if (G.Q == 0) {
    if (MU) launch_bwd_out(G, MU, colsum, gMU, gCV, st);
    return;
  }
  // Rows per tile: every block has one, as far as LDS holds it.
  const int T = (int)std::min<int64_t>(std::max<int64_t>(16, (G.n + nparts - 1) / nparts), kRouteTile / G.P);
  hipLaunchKernelGGL(MU ? k_bwd_route<true> : k_bwd_route<false>, dim3(nparts), dim3(256), 0, st, G, S, MU, colsum, gMU,
                     gCV, gVF, gVR, gEF, gER, gmax, gERsum, part, T);
  launch_sum_parts(nparts, 4 * G.Q, part, red4, true, st);
}

void launch_bwd_in(const BwdGraph& G, const BwdState& S, const double* MU, const QStat* qs1, const double* red4,
                   const float* gER, float* gVR, float* gVF, double* cD, const FmaxTerms& FE, hipStream_t st) {
  if (G.Q == 0) return;
  const int64_t rows = kIn * (256 / G.Q);
  const int nb = (int)std::min<int64_t>((G.n + rows - 1) / rows, 1024);  // resident at once: the prologue is paid once
  hipLaunchKernelGGL(k_bwd_in, dim3(nb), dim3(256), 0, st, G, S, MU, qs1, red4, gER, gVR, gVF, cD, FE);
}

void launch_bwd_fscatter(const BwdGraph& G, const float* gEF, const int* FA, const int* bsrc, int64_t brows,
                         float* gCE, hipStream_t st) {
  if (G.Q == 0) return;
  hipLaunchKernelGGL(k_bwd_fscatter, dim3(grid_for(G.n * G.Qs)), dim3(256), 0, st, G.n, G.Q, G.Qs, gEF, FA, bsrc, brows,
                     gCE);
}

// RMax edge terms, once after the last step: the minimum-cost out-edge row AO[v][q] receives -gERsum[v][q] (the sum
// over the steps of gE_R[v][q]).  Each (row, q) belongs to one (v, q).
__global__ void k_bwd_rterms(int64_t n, int Q, int Qs, const float* __restrict__ gER, const int* __restrict__ AO,
                             int64_t brows, float* __restrict__ gCE) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n * Qs; i += (int64_t)gridDim.x * blockDim.x) {
    const int q = (int)(i % Qs);
    if (q >= Q) continue;
    const float g = gER[i];
    if (g == 0.f) continue;
    const int row = AO[i];
    if (row >= 0 && row < brows) gCE[(int64_t)row * Qs + q] += -g;
  }
}




void launch_bwd_rterms(const BwdGraph& G, const float* gERsum, const int* AO, int64_t brows, float* gCE,
                       hipStream_t st) {
  if (G.Q == 0) return;
  const int64_t nq = G.n * G.Qs;
  hipLaunchKernelGGL(k_bwd_rterms, dim3((unsigned)std::min<int64_t>((nq + 255) / 256, 1 << 16)), dim3(256), 0, st,
                     G.n, G.Q, G.Qs, gERsum, AO, brows, gCE);
}

// Vertices per tile: as LDS holds (32 KB of rows), 64 at most, and fewer where that leaves CUs idle.
static int bwd_vtx_tile(const BwdGraph& G) {
  return (int)std::min<int64_t>(std::min(64, 4096 / std::max(1, G.Qs)), std::max<int64_t>(16, (G.n + 1023) / 1024));
}

int bwd_vtx_blocks(const BwdGraph& G) {
  const int T = bwd_vtx_tile(G);
  return (int)std::max<int64_t>(1, std::min<int64_t>((G.n + T - 1) / T, 2048));
}

void launch_bwd_vtx(const BwdGraph& G, float* gVR, const float* gVF, unsigned long long* gVRfix, const unsigned* gmax,
                    float* gMU, double* part, hipStream_t st) {
  const int T = bwd_vtx_tile(G), nb = bwd_vtx_blocks(G);
  const size_t lds = (size_t)T * 2 * G.Qs * sizeof(float) + (size_t)(G.P + 1 + 2 * G.Q) * sizeof(int);
  hipLaunchKernelGGL(k_bwd_vtx, dim3(nb), dim3(256), lds, st, G, gVR, gVF, gVRfix, gmax, gMU, part, T);
}

void launch_bwd_prep_fill(const BwdGraph& G, const double* red4, const QStat* qs0, const int* am0, float* gMU, double* cq,
                          hipStream_t st) {
  if (G.Q == 0) return;
  hipLaunchKernelGGL(k_bwd_prep_fill, dim3(1), dim3(256), 0, st, G, red4, qs0, am0, gMU, cq);
}

void launch_col_argmin(int64_t n, int P, const float* CV, float* pv, int* pi, int nparts, int* am, hipStream_t st) {
  hipLaunchKernelGGL(k_col_argmin, dim3(nparts), dim3(256), 0, st, n, P, CV, pv, pi);
  hipLaunchKernelGGL(k_col_argmin_final, dim3(P), dim3(256), 0, st, nparts, P, pv, pi, am);
}

void launch_bwd_edge_coef(int64_t nrows, int Q, int Qs, const int* beid, const int* bsrc, const float* CE,
                          const double* cD, const double* cq, float* G, hipStream_t st) {
  if (nrows == 0) return;
  hipLaunchKernelGGL(k_bwd_edge_coef, dim3(grid_for(nrows * (Qs / 4))), dim3(256), 0, st, nrows, Q, Qs, beid, bsrc, CE, cD,
                     cq, G);
}

void launch_bwd_vertex_coef(int64_t total, const float* CV, float* G, hipStream_t st) {
  hipLaunchKernelGGL(k_bwd_vertex_coef, dim3(grid_for(total)), dim3(256), 0, st, total, CV, G);
}

void launch_outer_acc(int64_t nrows, const int* idx, const float* feats, int dim, const float* G, int Gs, int K,
                      double* part, int nparts, hipStream_t st) {
  // Blocks of at most 32 pattern columns, each covering every row once per launch: 32 features wide, or, where 16 columns
  // are left (half the products of a 32-column block would be padding), up to 64, so that G is read once for them.  Bound by
  // the products and the gathered rows: vertices and edges of a training step at R-MAT 18 (12/16, 32 features), 251 us
  // together, 398 in 32-column blocks.  (The edges' coefficients formed in here instead of by k_bwd_edge_coef: 397 against
  // 230 and 184 us, their FP64 exponentials waiting at this kernel's low occupancy.)
  auto launch = [&](auto kernel, int q0, int k0) {
    hipLaunchKernelGGL(kernel, dim3(nparts), dim3(256), 0, st, nrows, idx, feats, dim, G, Gs, K, q0, k0, part);
  };
  for (int q0 = 0; q0 < K; q0 += 32) {
    const bool narrow = K - q0 <= 16;
    for (int k0 = 0, w; k0 < dim; k0 += w) {
      const int left = dim - k0;
      w = left <= 16 ? 16 : left <= 32 || !narrow ? 32 : 64;
      if (narrow)
        launch(w == 16 ? k_outer_mfma<1, 1> : w == 32 ? k_outer_mfma<1, 2> : k_outer_mfma<1, 4>, q0, k0);
      else
        launch(w == 16 ? k_outer_mfma<2, 1> : k_outer_mfma<2, 2>, q0, k0);
    }
  }
}

}  // namespace ac
