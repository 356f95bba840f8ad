// __global__ kernels of libcsipm (included once, by csipm.hip).
#pragma once

#include "csipm_device.hpp"

namespace csipm {

// ===========================================================================
// Standalone packing maps (FP64, bit-exact for even sizes)
// ===========================================================================

// v[k1 + ld1*(k2 + N2*k3)] for every element of the (ld1, N2, N3) spectrum.
template <int D>
__global__ __launch_bounds__(256) void k_beta_to_dft(const double* __restrict__ beta,
                                                     cpx<double>* __restrict__ v, MapGeom g,
                                                     int ld1, int64_t total) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const int k1 = (int)(t % ld1);
  const int64_t r = t / ld1;
  const int k2 = D >= 2 ? (int)(r % g.n[1]) : 0;
  const int k3 = D >= 3 ? (int)(r / g.n[1]) : 0;
  v[t] = beta_to_dft_elem<D, double>(beta, k1, k2, k3, g);
}

// Gather form of DFT_to_beta, one beta index at a time
// (src/mapping_cpu_kernels.jl:11-21, 38-87, 109-351).  Decodes the block of
// index i, the element it represents and reads it from the half spectrum
// (3D second-half dim-1 elements: conjugate partner, Im negated).
__host__ __device__ __forceinline__ int self_index(int s, const MapGeom& g, int dim) {
  return s == 0 ? 0 : g.M[dim];
}

template <int D>
__host__ __device__ __forceinline__ double dft_to_beta_elem(const cpx<double>* __restrict__ v,
                                                            int64_t i, const MapGeom& g,
                                                            int ld1) {
#pragma clang fp contract(off)
  int e[3] = {0, 0, 0};   // represented element (full-spectrum coordinates)
  int comp = 0;           // 0 Re, 1 Im
  bool vertex = false;
  const int P1 = g.P[0], P2 = g.P[1], P3 = g.P[2];
  const int S2 = g.S[1], S3 = g.S[2];
  // R offset r -> index r+1 ; H offset h -> index M+1+h
  if (D == 1) {
    if (i < g.off[1]) {
      vertex = true;
      e[0] = self_index((int)i, g, 0);
    } else {
      const int64_t t = i - g.off[1];
      comp = (int)(t / P1);
      e[0] = (int)(t % P1) + 1;
    }
  } else if (D == 2) {
    if (i < g.off[1]) {
      vertex = true;
      e[0] = self_index((int)i / S2, g, 0);
      e[1] = self_index((int)i % S2, g, 1);
    } else if (i < g.off[2]) {
      const int64_t t = i - g.off[1];
      const int q = (int)(t / P2);
      comp = q & 1;
      e[0] = self_index(q >> 1, g, 0);
      e[1] = (int)(t % P2) + 1;
    } else if (i < g.off[3]) {
      const int64_t t = i - g.off[2];
      const int q = (int)(t / P1);
      comp = q & 1;
      e[1] = self_index(q >> 1, g, 1);
      e[0] = (int)(t % P1) + 1;
    } else {
      const int64_t t = i - g.off[3];
      const int q = (int)(t / g.P12);   // 0: Re(R,R) 1: Im(R,R) 2: Re(R,H) 3: Im(R,H)
      const int64_t u = t % g.P12;
      comp = q & 1;
      e[0] = (int)(u % P1) + 1;
      const int c2 = (int)(u / P1);
      e[1] = (q >= 2) ? g.M[1] + 1 + c2 : c2 + 1;
    }
  } else {
    if (i < g.off[1]) {
      vertex = true;
      const int t = (int)i;
      e[2] = self_index(t % S3, g, 2);
      e[1] = self_index((t / S3) % S2, g, 1);
      e[0] = self_index(t / (S3 * S2), g, 0);
    } else if (i < g.off[2]) {           // edges along dim 3, groups (s1, s2)
      const int64_t t = i - g.off[1];
      const int q = (int)(t / P3);
      comp = q & 1;
      const int grp = q >> 1;
      e[0] = self_index(grp / S2, g, 0);
      e[1] = self_index(grp % S2, g, 1);
      e[2] = (int)(t % P3) + 1;
    } else if (i < g.off[3]) {           // edges along dim 2, groups (s1, s3)
      const int64_t t = i - g.off[2];
      const int q = (int)(t / P2);
      comp = q & 1;
      const int grp = q >> 1;
      e[0] = self_index(grp / S3, g, 0);
      e[2] = self_index(grp % S3, g, 2);
      e[1] = (int)(t % P2) + 1;
    } else if (i < g.off[4]) {           // edges along dim 1, groups (s2, s3)
      const int64_t t = i - g.off[3];
      const int q = (int)(t / P1);
      comp = q & 1;
      const int grp = q >> 1;
      e[1] = self_index(grp / S3, g, 1);
      e[2] = self_index(grp % S3, g, 2);
      e[0] = (int)(t % P1) + 1;
    } else if (i < g.off[5]) {           // faces, self-conjugate dim 1
      const int64_t t = i - g.off[4];
      const int q = (int)(t / g.P23);
      const int64_t u = t % g.P23;
      comp = q & 1;
      e[0] = self_index(q >> 2, g, 0);
      const int c2 = (int)(u % P2);
      e[2] = (int)(u / P2) + 1;
      e[1] = ((q & 2) ? g.M[1] + 1 + c2 : c2 + 1);
    } else if (i < g.off[6]) {           // faces, self-conjugate dim 2
      const int64_t t = i - g.off[5];
      const int q = (int)(t / g.P13);
      const int64_t u = t % g.P13;
      comp = q & 1;
      e[1] = self_index(q >> 2, g, 1);
      const int c1 = (int)(u % P1);
      e[2] = (int)(u / P1) + 1;
      e[0] = ((q & 2) ? g.M[0] + 1 + c1 : c1 + 1);
    } else if (i < g.off[7]) {           // faces, self-conjugate dim 3
      const int64_t t = i - g.off[6];
      const int q = (int)(t / g.P12);
      const int64_t u = t % g.P12;
      comp = q & 1;
      e[2] = self_index(q >> 2, g, 2);
      const int c1 = (int)(u % P1);
      e[1] = (int)(u / P1) + 1;
      e[0] = ((q & 2) ? g.M[0] + 1 + c1 : c1 + 1);
    } else {                             // interior
      const int64_t t = i - g.off[7];
      const int q = (int)(t / g.P123);   // 2*blk + comp, blk: (R,R) (H,R) (R,H) (H,H)
      const int64_t u = t % g.P123;
      comp = q & 1;
      const int blk = q >> 1;
      const int c1 = (int)(u % P1);
      const int64_t u2 = u / P1;
      const int c2 = (int)(u2 % P2);
      e[2] = (int)(u2 / P2) + 1;
      e[0] = (blk & 1) ? g.M[0] + 1 + c1 : c1 + 1;
      e[1] = (blk & 2) ? g.M[1] + 1 + c2 : c2 + 1;
    }
  }
  double sign = 1.0;
  if (e[0] > g.M[0]) {  // second half of dim 1: read the conjugate partner
    e[0] = g.n[0] - e[0];
    e[1] = e[1] == 0 ? 0 : g.n[1] - e[1];
    e[2] = e[2] == 0 ? 0 : g.n[2] - e[2];
    sign = -1.0;
  }
  const cpx<double> val = v[e[0] + (int64_t)ld1 * (e[1] + (int64_t)g.n[1] * e[2])];
  const double sq2 = 1.4142135623730951;
  if (vertex) return val.x;
  if (comp == 0) return sq2 * val.x;
  return (sign * sq2) * val.y;
}

template <int D>
__global__ __launch_bounds__(256) void k_dft_to_beta(const cpx<double>* __restrict__ v,
                                                     double* __restrict__ beta, MapGeom g,
                                                     int ld1) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.N) return;
  beta[i] = dft_to_beta_elem<D>(v, i, g, ld1);
}

// ===========================================================================
// Destinations of the forward passes that end in beta (or u) space
// ===========================================================================
template <typename T>
struct Epi {
  int kind;             // 0: out[i] = value          1: condensed KKT epilogue
                        // 2: reduced (Schur) epilogue y = alpha (m + D x) + beta y, D in L1
  T* out;               // kind 0: the value; kind 2: m itself as well, when not null
  const T* xb;
  const T* xz;
  const T* L1;
  const T* L2;
  T* yb;
  T* yz;
  T alpha, beta;
  double* dot_part;     // per-block partial sums of x'y (CG p'q), or null
};

// The epilogue of a u-space element in two steps, so that a thread can issue
// the operand loads of several elements before it consumes any of them:
// epi_fetch_u loads what kind `e.kind` reads (always in range for el < U),
// epi_commit_u forms and stores the result and returns its x'y term.
template <typename T>
struct EpiOps {
  cpx<T> xb, xz, l1, l2, ob, oz;
};

template <typename T>
__device__ __forceinline__ EpiOps<T> epi_fetch_u(const Epi<T>& e, int64_t el) {
  EpiOps<T> o;
  const cpx<T> z = {(T)0, (T)0};
  o.xb = o.xz = o.l1 = o.l2 = o.ob = o.oz = z;
  if (e.kind == 0) return o;
  o.xb = reinterpret_cast<const cpx<T>*>(e.xb)[el];
  o.l1 = reinterpret_cast<const cpx<T>*>(e.L1)[el];
  if (e.beta != (T)0) o.ob = reinterpret_cast<const cpx<T>*>(e.yb)[el];
  if (e.kind == 2) return o;
  o.xz = reinterpret_cast<const cpx<T>*>(e.xz)[el];
  o.l2 = reinterpret_cast<const cpx<T>*>(e.L2)[el];
  if (e.beta != (T)0) o.oz = reinterpret_cast<const cpx<T>*>(e.yz)[el];
  return o;
}

template <typename T>
__device__ __forceinline__ double epi_commit_u(const Epi<T>& e, int64_t el, cpx<T> m,
                                               const EpiOps<T>& o) {
  if (e.kind == 0) {
    reinterpret_cast<cpx<T>*>(e.out)[el] = m;
    return 0.0;
  }
  if (e.kind == 2) {
    if (e.out) reinterpret_cast<cpx<T>*>(e.out)[el] = m;
    cpx<T> qb = {e.alpha * (m.x + o.l1.x * o.xb.x), e.alpha * (m.y + o.l1.y * o.xb.y)};
    if (e.beta != (T)0) {
      qb.x += e.beta * o.ob.x;
      qb.y += e.beta * o.ob.y;
    }
    reinterpret_cast<cpx<T>*>(e.yb)[el] = qb;
    return (double)o.xb.x * qb.x + (double)o.xb.y * qb.y;
  }
  cpx<T> qb = {e.alpha * (m.x + o.l1.x * o.xb.x + o.l2.x * o.xz.x),
               e.alpha * (m.y + o.l1.y * o.xb.y + o.l2.y * o.xz.y)};
  cpx<T> qz = {e.alpha * (o.l2.x * o.xb.x + o.l1.x * o.xz.x),
               e.alpha * (o.l2.y * o.xb.y + o.l1.y * o.xz.y)};
  if (e.beta != (T)0) {
    qb.x += e.beta * o.ob.x;
    qb.y += e.beta * o.ob.y;
    qz.x += e.beta * o.oz.x;
    qz.y += e.beta * o.oz.y;
  }
  reinterpret_cast<cpx<T>*>(e.yb)[el] = qb;
  reinterpret_cast<cpx<T>*>(e.yz)[el] = qz;
  return (double)o.xb.x * qb.x + (double)o.xb.y * qb.y + (double)o.xz.x * qz.x +
         (double)o.xz.y * qz.y;
}

// Global-memory phases of the pass kernels run in groups of stage_k<T>()
// elements per thread: fetch(i) issues the loads of element i (branch-free,
// on an index clamped into range), put(i, r) consumes them.  All fetches of
// a group come before its first put, so a thread has that many loads in
// flight instead of one.
template <typename T>
constexpr int stage_k() {
  return sizeof(T) == 4 ? 8 : 4;
}

// The members of a group past the end are skipped by a uniform branch: a small
// tile otherwise spent most of its instructions on clamped repeats.
template <int NT, int K, typename R, typename F, typename P>
__device__ __forceinline__ void staged(int total, F&& fetch, P&& put) {
  for (int g0 = 0; g0 < total; g0 += K * NT) {
    const int i0 = g0 + (int)threadIdx.x;
    R r[K];
#pragma unroll
    for (int j = 0; j < K; ++j)
      if (g0 + j * NT < total) r[j] = fetch(min(i0 + j * NT, total - 1));
#pragma unroll
    for (int j = 0; j < K; ++j)
      if (i0 + j * NT < total) put(i0 + j * NT, r[j]);
  }
}

// The same for the beta entries an element of the half spectrum feeds (none
// of them: an element that beta does not hold).
template <typename T>
struct BetaOps {
  EpiOps<T> o;        // operands of the real-part entry (.x) and the other (.y)
  uint32_t re, im;
  bool hit, vertex, neg;
};

// interior: 1 <= k1 <= P1 and D >= 2
template <int D, typename T>
__device__ __forceinline__ BetaOps<T> epi_fetch_beta(const Epi<T>& e, int k1, int k2, int k3,
                                                     const MapGeom& g, bool interior) {
  BetaOps<T> r;
  r.hit = true;
  r.vertex = false;
  if (D >= 2 && interior) {
    const BetaRow w = beta_row<D>(k2, k3, g);
    r.re = w.re + (uint32_t)(w.s * k1);
    r.im = r.re + w.d;
    r.neg = w.neg;
  } else {
    int64_t re, im;
    r.hit = scatter_targets<D>(k1, k2, k3, g, re, im, r.vertex, r.neg);
    r.re = r.hit ? (uint32_t)re : 0u;
    r.im = r.hit && !r.vertex ? (uint32_t)im : r.re;
  }
  const cpx<T> z = {(T)0, (T)0};
  r.o.xb = r.o.xz = r.o.l1 = r.o.l2 = r.o.ob = r.o.oz = z;
  if (e.kind == 0) return r;
  r.o.xb = {e.xb[r.re], e.xb[r.im]};
  r.o.l1 = {e.L1[r.re], e.L1[r.im]};
  if (e.beta != (T)0) r.o.ob = {e.yb[r.re], e.yb[r.im]};
  if (e.kind == 2) return r;
  r.o.xz = {e.xz[r.re], e.xz[r.im]};
  r.o.l2 = {e.L2[r.re], e.L2[r.im]};
  if (e.beta != (T)0) r.o.oz = {e.yz[r.re], e.yz[r.im]};
  return r;
}

// v: the spectrum value
template <typename T>
__device__ __forceinline__ double epi_commit_beta(const Epi<T>& e, cpx<T> v, const BetaOps<T>& r) {
  if (!r.hit) return 0.0;
  const T sq2 = (T)1.4142135623730951;
  const EpiOps<T>& o = r.o;
  cpx<T> m = {sq2 * v.x, sq2 * v.y};
  if (r.neg) m.y = -m.y;
  if (r.vertex) m.x = v.x;
  if (e.kind == 0) {
    e.out[r.re] = m.x;
    if (!r.vertex) e.out[r.im] = m.y;
    return 0.0;
  }
  if (e.kind == 2) {
    if (e.out) {
      e.out[r.re] = m.x;
      if (!r.vertex) e.out[r.im] = m.y;
    }
    cpx<T> qb = {e.alpha * (m.x + o.l1.x * o.xb.x), e.alpha * (m.y + o.l1.y * o.xb.y)};
    if (e.beta != (T)0) {
      qb.x += e.beta * o.ob.x;
      qb.y += e.beta * o.ob.y;
    }
    e.yb[r.re] = qb.x;
    if (!r.vertex) e.yb[r.im] = qb.y;
    return (double)o.xb.x * qb.x + (r.vertex ? 0.0 : (double)o.xb.y * qb.y);
  }
  cpx<T> qb = {e.alpha * (m.x + o.l1.x * o.xb.x + o.l2.x * o.xz.x),
               e.alpha * (m.y + o.l1.y * o.xb.y + o.l2.y * o.xz.y)};
  cpx<T> qz = {e.alpha * (o.l2.x * o.xb.x + o.l1.x * o.xz.x),
               e.alpha * (o.l2.y * o.xb.y + o.l1.y * o.xz.y)};
  if (e.beta != (T)0) {
    qb.x += e.beta * o.ob.x;
    qb.y += e.beta * o.ob.y;
    qz.x += e.beta * o.oz.x;
    qz.y += e.beta * o.oz.y;
  }
  e.yb[r.re] = qb.x;
  e.yz[r.re] = qz.x;
  double acc = (double)o.xb.x * qb.x + (double)o.xz.x * qz.x;
  if (!r.vertex) {
    e.yb[r.im] = qb.y;
    e.yz[r.im] = qz.y;
    acc += (double)o.xb.y * qb.y + (double)o.xz.y * qz.y;
  }
  return acc;
}

// per-block partial of a dot product (deterministic; finalised by a later kernel)
__device__ __forceinline__ void store_partial(double* part, double acc, int idx) {
  const double s = block_reduce(acc, OpSum());
  if (threadIdx.x == 0 && part) part[idx] = s;
}

// ===========================================================================
// FFT passes over the (H1, N2, N3) half spectrum.
//  lines: along dimension 2 (axis 1) or 3 (axis 2); a workgroup takes 2^lg
//         lines with consecutive k1, so global accesses are contiguous.
//  dim1:  dimension 1; two real lines per complex FFT of length N1
//         (z = x_a + i x_b), 2^lg pairs per workgroup.
//  col, row: the four-step passes of long 1D lines, below.
// One body runs them all (pass_body): a pass is a load, one or two turns of
// the line transform with a step between them, and a store.  Kernels exist for
// each combination the single-instance passes and the batched chains use, and
// one that takes the steps from PassArgs: a batch of several dimensionalities
// runs the passes at one position of all its chains in one launch of that
// kernel, side by side instead of one after another.  It is the slower one for
// passes of one kind (registers and branches of all steps: 255 x 255 FP64 31.9
// against 39.4 us an apply, 49999 FP32 45 against 59 us) and much the faster
// one for a mix (48 requests of the serving stream's mix, launches of one kind
// on two streams 70 ms a solve, mixed launches 57 ms).
// Sources: SRC_BUF (scratch spectrum), SRC_BETA (gather from beta through the
// packing map), SRC_U (spectrum-ordered beta), SRC_REAL (real samples, dim 1).
// Destinations likewise, the beta / u ones with the epilogue Epi.
// ===========================================================================
enum { SRC_BUF = 0, SRC_BETA = 1, SRC_REAL = 2, SRC_U = 3 };
enum { DST_BUF = 0, DST_BETA = 1, DST_REAL = 2, DST_U = 3 };
enum { MODE_MTM = 0, MODE_C2R = 1, MODE_R2C = 2 };
// four-step passes (see below)
enum { C_FIRST = 0, C_REAL_IN = 1, C_MID = 2, C_LAST = 3, C_MID_C2R = 4 };
enum { R_MTM = 0, R_C2R = 1, R_R2C = 2, R_CONV_INV = 3, R_CONV_FWD = 4 };

// the steps of a pass
enum {   // load
  LD_LINES_BUF_FWD, LD_LINES_BUF_INV, LD_LINES_U2, LD_LINES_U3, LD_LINES_BETA2, LD_LINES_BETA3,
  LD_DIM1_BUF, LD_DIM1_U, LD_DIM1_BETA, LD_DIM1_REAL,
  LD_COL_FIRST_U, LD_COL_FIRST_BETA, LD_COL_REAL, LD_COL_BUF_FWD, LD_COL_BUF_INV,
  LD_ROW_FWD, LD_ROW_INV, LD_ROW_REAL
};
enum {   // between the two turns (MID_NONE: one turn)
  MID_NONE, MID_DIM1_MASK, MID_COL, MID_ROW_MASK, MID_ROW_CONV_INV, MID_ROW_CONV_FWD
};
enum {   // store
  ST_LINES_BUF_FWD, ST_LINES_BUF_INV, ST_LINES_U2, ST_LINES_U3, ST_LINES_BETA2, ST_LINES_BETA3,
  ST_DIM1_BUF, ST_DIM1_U, ST_DIM1_BETA, ST_DIM1_REAL,
  ST_COL_BUF_FWD, ST_COL_BUF_INV, ST_COL_U, ST_COL_BETA, ST_COL_REAL,
  ST_ROW_FWD, ST_ROW_INV, ST_ROW_REAL
};

template <typename T>
struct PassArgs {
  int ld, mid, st;      // the pass (LD_*, MID_*, ST_*)
  MapGeom g;
  const FftPlan* plan;  // device-resident
  const cpx<T>* tw;     // the plan's twiddles, stage by stage
  int axis;      // line passes: 1 or 2
  int H1;
  int lg;        // log2 of lines (pairs) per workgroup
  int ps;        // LDS line stride
  int ntile1;    // line passes: tiles along k1
  int nlines;    // dimension 1: real lines N2*N3
  int npairs;
  uint32_t h1m;  // ceil(2^32 / H1)
  uint32_t n1m;  // ceil(2^32 / N1)
  cpx<T>* buf;
  const T* beta_in;
  const cpx<T>* u_in;
  const T* real_in;
  T* real_out;
  Epi<T> epi;
  const uint32_t* miss;  // bit set = missing sample (nullable)
  T scale;
  const int* done;
  // line transform: length len; bs = 1 selects Bluestein's chirp-z form, in
  // which case plan is the convolution FFT of length M >= 2 len - 1; bs = 2
  // selects Rader's form for a prime len, plan being the FFT of length len -
  // 1; bs = 3 the dense form, dense its coefficients (see dense_dft)
  int len;
  int bs;
  const cpx<T>* chirp;  // w_n = exp(-i pi n^2 / len), n < len
  const cpx<T>* bfw;    // FFT_M(b) / M of the forward kernel b = conj(w) (wrapped);
                        // Rader: FFT_{L-1}(b) / (L-1) of b_j = exp(-2 pi i g^-j / L)
  const T* dense;       // dense form: cosine, then sine tiles
  const int* rperm;     // Rader: [e] row of element e in the convolution order
                        // (e = 0: row L), [L + m] element g^-m mod L of output m
  // long 1D lines (four-step): the length-F transform (F = len, or the
  // Bluestein length when obs) as A columns x B rows, position col + A*row
  int A, B, F;
  int obs;              // outer Bluestein: chirp / bfw are of length len / F
  uint32_t am;          // ceil(2^32 / A)
  const cpx<T>* twF;    // exp(-2 pi i j / F), j < F
};

// Dense form of the forward DFT for line lengths L <= 511 that no plan of the
// radices covers, on the matrix cores: with H = L / 2 and, for j = 1 ..
// (L - 1) / 2, a_j = x_j + x_{L-j} and b_j = x_j - x_{L-j} (a_0 = x_0, and
// a_H = x_H when L is even),
//   X_k = sum_j a_j cos(2 pi j k / L) - i sum_j b_j sin(2 pi j k / L),
// X_{L-k} the same with + i: two real matrix products of about H x H with the
// tile's 2 nl real columns.  a and b replace x in LDS rows j and L - j; a wave
// takes output tiles of 16 k by 16 columns, eight accumulators each (C and S)
// at most four at a time, and the outputs replace a and b when all waves have
// read them.  The coefficients come packed in lane order, 64 to a 16 x 4 tile
// (the wave reads them from the L2, one load feeding N products).
// What bounds it: the products take L^2 / 128 cycles a line and CU in FP32 (L^2
// / 64 in FP64), which is 17% of the time of a 127^3 line pass (FP64 23%): its
// waves wait 60% of theirs for memory and LDS, since in a tile of 8 lines each
// load of a coefficient feeds one product.  At 185^3 the matrix cores are busy
// 41%, and the waves wait half their time to issue.  Rader's and Bluestein's
// forms of such lengths spent over a thousand cycles a line on two transforms
// and the moves between, in twice the LDS rows: the operator product of 127^3
// took 187 us in FP32 and 71 with this (185^3: 400 to 243, FP64 784 to 392).
// tiles of the coefficient matrices: ceil((H + 1) / 16) by ceil((H + 1) / 4)
// (cosine) and by ceil(((L - 1) / 2) / 4) (sine), the latter two made even
// (zero tiles; their rows stay inside the line for L > 16)
__host__ __device__ __forceinline__ int dense_mt(int L) { return (L / 2 + 16) / 16; }
__host__ __device__ __forceinline__ int dense_kc(int L) { return (L / 2 + 8) / 8 * 2; }
__host__ __device__ __forceinline__ int dense_ks(int L) { return ((L - 1) / 2 + 7) / 8 * 2; }

// acc += coefficients (tile 0 at p[u], 64 entries a tile) x rows of x: tile kt
// takes rows r0 + step * (4 kt + lane / 16); two tiles a turn, the next two
// loaded before the products of these.  The products are summed in parts of 8
// (lines up to 127, U = 1) or 32: one chain over the whole line rounds as often
// as it has terms.  M^T M off by, FP32 / FP64: 127 x 127 in one chain 3.1e-7 /
// 5.7e-16, in parts of 8 2.0e-7 / 3.6e-16 (Rader's form 3.2e-7 / 7.2e-16, the
// radix plan of 116 x 124 2.1e-7 / 3.9e-16); 509 x 2100 4.5e-7 / 8.3e-16 in one
// chain, 2.5e-7 / 4.7e-16 in parts of 32 (Bluestein's 3.0e-7 / 7.1e-16; parts of 8
// took 185^3 in FP64 from 406 to 432 us)
template <typename T, int U, int N>
__device__ __forceinline__ void dense_product(Vec4<T> (&acc)[U][N], const T* const (&p)[U],
                                              int tiles, const T* x, int r0, int step, int rs,
                                              const int (&col)[N]) {
  const int kk = ((int)threadIdx.x & 63) >> 4;
  T q[2][U], qn[2][U];
  Vec4<T> part[U][N];
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int v = 0; v < N; ++v) part[u][v] = Vec4<T>{0, 0, 0, 0};
    q[0][u] = p[u][0];
    q[1][u] = p[u][64];
  }
#pragma unroll 1
  for (int kt = 0; kt < tiles; kt += 2) {
    const int nx = min(kt + 2, tiles - 2) * 64;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      qn[0][u] = p[u][nx];
      qn[1][u] = p[u][nx + 64];
    }
    T b[2][N];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int v = 0; v < N; ++v) b[h][v] = x[(r0 + step * (4 * (kt + h) + kk)) * rs + col[v]];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int v = 0; v < N; ++v) part[u][v] = mfma16x16x4(q[h][u], b[h][v], part[u][v]);
    if (U == 1 || (kt & 6) == 6 || kt + 2 >= tiles) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int v = 0; v < N; ++v) {
          acc[u][v] += part[u][v];
          part[u][v] = Vec4<T>{0, 0, 0, 0};
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      q[0][u] = qn[0][u];
      q[1][u] = qn[1][u];
    }
  }
}

// U k-tiles of a wave (k-tile wave + u NT / 64) by N column tiles
template <typename T, int NT, int U, int N>
__device__ __forceinline__ void dense_tiles(cpx<T>* lds, const T* __restrict__ coef, int L,
                                            int cols, int rs) {
  constexpr int W = NT / 64;
  const int wave = uniform((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
  const int n = lane & 15;
  const int Mt = dense_mt(L), Kc = dense_kc(L), Ks = dense_ks(L);
  T* x = reinterpret_cast<T*>(lds);
  Vec4<T> c[U][N], s[U][N];
  const T* ac[U];
  const T* as[U];
  int col[N];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int mt = min(wave + u * W, Mt - 1);   // tiles past the last: repeated, not stored
    ac[u] = coef + (int64_t)mt * Kc * 64 + lane;
    as[u] = coef + ((int64_t)Mt * Kc + (int64_t)mt * Ks) * 64 + lane;
#pragma unroll
    for (int v = 0; v < N; ++v) c[u][v] = s[u][v] = Vec4<T>{0, 0, 0, 0};
  }
#pragma unroll
  for (int v = 0; v < N; ++v) col[v] = min(n + 16 * v, cols - 1);
  // columns of the cosine matrix: a_j in row j; rows past H hold other finite
  // values of the same column and meet zero coefficients.  Of the sine
  // matrix: b_j in row L - j
  dense_product<T, U, N>(c, ac, Kc, x, 0, 1, rs, col);
  dense_product<T, U, N>(s, as, Ks, x, L - 1, -1, rs, col);
  __syncthreads();
  const bool im = n & 1;   // column pairs hold real and imaginary parts
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int mt = wave + u * W;
#pragma unroll
    for (int v = 0; v < N; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const T other = lane_swap(s[u][v][i]);
        const T plus = c[u][v][i] + other, minus = c[u][v][i] - other;
        const int k = 16 * mt + mfma_row<T>(lane, i);
        if (mt < Mt && k <= L / 2 && n + 16 * v < cols) {
          x[k * rs + col[v]] = im ? minus : plus;
          if (k > 0 && 2 * k != L) x[(L - k) * rs + col[v]] = im ? plus : minus;
        }
      }
  }
  __syncthreads();
}

template <typename T, int NT>
__device__ __forceinline__ void dense_dft(cpx<T>* lds, const T* __restrict__ coef, int L,
                                          int lg, int ps) {
  const int nl = 1 << lg;
  for (int idx = threadIdx.x; idx < ((L - 1) / 2) << lg; idx += NT) {
    const int line = idx & (nl - 1), j = 1 + (idx >> lg);
    cpx<T>*p = lds + j * ps + line, *q = lds + (L - j) * ps + line;
    const cpx<T> x = *p, y = *q;
    *p = cadd(x, y);
    *q = csub(x, y);
  }
  __syncthreads();
  const int cols = 2 << lg, rs = 2 * ps;
  const int u = (dense_mt(L) + NT / 64 - 1) / (NT / 64);
  if (u == 1) {
    if (lg <= 3) dense_tiles<T, NT, 1, 1>(lds, coef, L, cols, rs);
    else if (lg == 4) dense_tiles<T, NT, 1, 2>(lds, coef, L, cols, rs);
    else dense_tiles<T, NT, 1, 4>(lds, coef, L, cols, rs);
  } else if (u == 2) {
    if (lg <= 3) dense_tiles<T, NT, 2, 1>(lds, coef, L, cols, rs);
    else dense_tiles<T, NT, 2, 2>(lds, coef, L, cols, rs);
  } else if (u == 3) {
    dense_tiles<T, NT, 3, 1>(lds, coef, L, cols, rs);
  } else {
    dense_tiles<T, NT, 4, 1>(lds, coef, L, cols, rs);
  }
}

// the same as a call, for the kernels of mixed launches: its registers are
// not added to those of their other steps (a mixed launch of 48 requests, FP32,
// 256 threads: inlined 31.5 us and 31 of 128 registers spilled, called 28.0)
template <typename T>
using LdsTile = __attribute__((address_space(3))) cpx<T>*;
template <typename T, int NT>
__device__ __noinline__ void dense_dft_call(LdsTile<T> lds, const T* coef, int L, int lg, int ps) {
  dense_dft<T, NT>((cpx<T>*)lds, coef, L, lg, ps);
}

// Forward DFT of length a.len of the 2^lg lines in LDS ([element][line],
// stride ps), in place.  Direct: the Stockham plan.  Bluestein (lengths with a
// prime factor above 31): X_k = w_k sum_n (x_n w_n) conj(w_{k-n}), the
// convolution by FFT_M, pointwise product with the precomputed kernel
// spectrum, inverse FFT_M.  LDS must hold M rows.
// Rader (prime L = p, bs = 2), with g a primitive root mod p:
//   X_0 = x_0 + sum_{n>0} x_n,   X_{g^-m} = x_0 + sum_q x_{g^q} w^{g^(q-m)}
// (w = exp(-2 pi i / p)), a cyclic convolution of length p - 1 of
// a_q = x_{g^q} with b_j = w^{g^-j}, done by FFT_{p-1}, the pointwise product
// with the precomputed FFT_{p-1}(b) / (p - 1) and the inverse FFT_{p-1}.
// LDS rows of a tile: 0..p-1 the line in natural order, p..2p-2 the
// convolution (row p + q), 2p-1 x_0 and 2p X_0 (= x_0 + A_0, the DC term of
// FFT_{p-1}(a)).  The two permutations move between disjoint rows, one
// element at a time.
//
// One copy of the FFT per kernel: the inverse transforms (of a pass, and of
// the convolutions) run the forward code on values with real and imaginary
// part exchanged, and both transforms of a convolution are turns of one loop.
// With an inlined copy for every direction and form (ten in the dimension-1
// pass) a launch ran each copy once, cold: the short launches of single
// problems waited for instruction fetches as much as for data.
template <typename T, int E, int NT>
__device__ __forceinline__ void line_dft(cpx<T>* lds, const PassArgs<T>& a, int pl, int lg,
                                         int ps) {
  const int L = a.len, M = plan_word(pl, 0), nl = 1 << lg;
  constexpr int K = stage_k<T>();
  cpx<T>* conv = lds;
  // the table loads of each phase are issued in groups (staged) so that a
  // thread has several in flight instead of waiting for each before its move
  if (a.bs == 2) {
    conv = lds + L * ps;
    const int* __restrict__ perm = a.rperm;
    staged<NT, 8, int>(
        L << lg, [&](int idx) { return perm[idx >> lg]; },   // e = 0: q = p - 1, the x_0 row
        [&](int idx, int q) {
          const int line = idx & (nl - 1), e = idx >> lg;
          conv[q * ps + line] = lds[e * ps + line];
        });
    __syncthreads();
  } else if (a.bs == 1) {
    staged<NT, K, cpx<T>>(
        M << lg, [&](int idx) { return a.chirp[min(idx >> lg, L - 1)]; },
        [&](int idx, const cpx<T>& w) {
          const int line = idx & (nl - 1), e = idx >> lg;
          cpx<T>* q = lds + e * ps + line;
          *q = e < L ? cmul(*q, w) : cpx<T>{(T)0, (T)0};
        });
    __syncthreads();
  }
  cpx<T>* x0row = lds + (2 * L - 1) * ps;   // Rader
  cpx<T>* X0row = lds + 2 * L * ps;
  const int turns = a.bs ? 2 : 1;
#pragma unroll 1
  for (int t = 0; t < turns; ++t) {
    lds_fft<T, E, NT>(conv, pl, lg, ps, a.tw);
    if (t == 0 && a.bs) {
      // the product with the kernel spectrum, exchanged for the inverse FFT
      const cpx<T>* __restrict__ B = a.bfw;
      const bool rader = a.bs == 2;
      staged<NT, K, cpx<T>>(
          M << lg, [&](int idx) { return B[idx >> lg]; },
          [&](int idx, const cpx<T>& bk) {
            const int line = idx & (nl - 1), e = idx >> lg;
            cpx<T>* q = conv + e * ps + line;
            const cpx<T> v = *q;
            if (rader && e == 0) X0row[line] = cadd(x0row[line], v);
            *q = cswap(cmul(v, bk));
          });
      __syncthreads();
    }
  }
  if (a.bs == 2) {
    // X_{g^-m} = x_0 + c_m into row g^-m (1..p-1); the last index: X_0 into row 0
    const int* __restrict__ perm = a.rperm;
    staged<NT, 8, int>(
        L << lg, [&](int idx) { return perm[L + min(idx >> lg, L - 2)]; },
        [&](int idx, int row) {
          const int line = idx & (nl - 1), m = idx >> lg;
          if (m < L - 1)
            lds[row * ps + line] = cadd(cswap(conv[m * ps + line]), x0row[line]);
          else
            lds[line] = X0row[line];
        });
    __syncthreads();
  } else if (a.bs == 1) {
    staged<NT, K, cpx<T>>(
        L << lg, [&](int idx) { return a.chirp[idx >> lg]; },
        [&](int idx, const cpx<T>& w) {
          const int line = idx & (nl - 1), e = idx >> lg;
          cpx<T>* q = lds + e * ps + line;
          *q = cmul(cswap(*q), w);
        });
    __syncthreads();
  }
}

__device__ __forceinline__ int udiv(int a, int d, uint32_t m) { return d == 1 ? a : fdiv(a, m); }

// Workgroups are dispatched to the 8 XCDs round robin (block b on XCD b % 8),
// each XCD with its own L2.  xcd_block() numbers the blocks so that blocks
// b, b + 8, b + 16, .. (one XCD) take consecutive numbers: adjacent tiles,
// which share the cache lines at their edges, then meet in one L2.  A
// bijection of [0, gridDim.x); the last gridDim.x % 8 blocks keep their own.
__device__ __forceinline__ int xcd_block() {
  const int b = (int)blockIdx.x, q = (int)gridDim.x >> 3;
  return b >= (q << 3) ? b : (b & 7) * q + (b >> 3);
}

// a fetched source value: mode -1 = outside the tile (zero), otherwise the
// u_scale map of an SRC_U or SRC_BETA load (SRC_BUF: the value as loaded)
template <typename T>
struct Raw {
  cpx<T> w;
  int mode;
};

template <typename T, int SRC>
__device__ __forceinline__ cpx<T> raw_value(const Raw<T>& r) {
  if (r.mode < 0) return {(T)0, (T)0};
  return SRC == SRC_BUF ? r.w : u_scale(r.w, r.mode);
}

// the source value of element (k1, k2, k3); interior: 1 <= k1 <= P1 and D >= 2
template <int D, typename T, int SRC>
__device__ __forceinline__ Raw<T> spec_fetch(const PassArgs<T>& a, int k1, int k2, int k3,
                                             bool interior) {
  Raw<T> r;
  if (SRC == SRC_U) {
    r.w = a.u_in[u_src<D>(k1, k2, k3, a.g, a.H1, r.mode)];
    return r;
  }
  if (D >= 2 && interior) {
    const BetaRow w = beta_row<D>(k2, k3, a.g);
    const uint32_t re = w.re + (uint32_t)(w.s * k1);
    r.mode = w.neg ? 2 : 0;
    r.w = {a.beta_in[re], a.beta_in[re + w.d]};
    return r;
  }
  // beta_to_dft_elem's entries (an element that beta does not hold reads its
  // partner's, conjugate)
  Cat c1 = cat_of(k1, a.g, 0);
  Cat c2 = D >= 2 ? cat_of(k2, a.g, 1) : Cat{0, 0};
  Cat c3 = D >= 3 ? cat_of(k3, a.g, 2) : Cat{0, 0};
  r.mode = 0;
  if (!is_rep<D>(c1, c2, c3)) {
    c1 = cat_mirror(c1, a.g.P[0]);
    c2 = cat_mirror(c2, a.g.P[1]);
    c3 = cat_mirror(c3, a.g.P[2]);
    r.mode = 2;
  }
  int64_t bs;
  bool vertex;
  const int64_t re = rep_index<D>(c1, c2, c3, a.g, bs, vertex);
  if (vertex) r.mode = 1;
  r.w = {a.beta_in[re], a.beta_in[re + (vertex ? 0 : bs)]};
  return r;
}

// a value on its way into or out of the LDS tile of a pass whose transform is
// forward (FWD) or inverse (held exchanged, see line_dft)
template <bool FWD, typename T>
__device__ __forceinline__ cpx<T> tile_value(cpx<T> v) {
  return FWD ? v : cswap(v);
}

// a spectrum value read from LDS with its epilogue operands
template <typename T>
struct Fetched {
  cpx<T> m;
  EpiOps<T> ops;
};
template <typename T>
struct FetchedBeta {
  cpx<T> m;
  BetaOps<T> ops;
};

// block -> instance map of a vector launch over several instances
struct BSeg {
  const int* inst;   // instance of each block
  const int* first;  // first block of each instance (n + 1 entries)
};

// the tile of a line pass (tile = its index within the pass) into LDS
template <typename T, int NT, int D, int SRC, bool FWD>
__device__ __forceinline__ void lines_load(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int L = a.len;
  const int lg = a.lg, nl = 1 << lg;
  const int tile1 = tile % a.ntile1;
  const int o = tile / a.ntile1;
  const int k10 = tile1 << lg;
  const int nv = min(nl, a.H1 - k10);
  // element indexes of the half spectrum fit 31 bits
  const int s2 = a.H1, s3 = a.H1 * a.g.n[1];
  const int sl = a.axis == 1 ? s2 : s3;
  const int base = k10 + (a.axis == 1 ? o * s3 : o * s2);
  const int total = L << lg;
  constexpr int K = stage_k<T>();
  // a tile whose k1 are all representatives (1 <= k1 <= P1) reads and writes
  // u at the scratch index with the plain sqrt2 scalings of u_to_v / v_to_u
  const bool interior = k10 >= 1 && k10 + nv - 1 <= a.g.P[0];
  if (SRC == SRC_U && interior) {
    staged<NT, K, Raw<T>>(
        total,
        [&](int idx) {
          const int line = idx & (nl - 1), el = idx >> lg;
          Raw<T> r;
          r.mode = line < nv ? 0 : -1;
          r.w = a.u_in[base + (line < nv ? line : 0) + el * sl];
          return r;
        },
        [&](int idx, const Raw<T>& r) { lds[idx] = tile_value<FWD>(raw_value<T, SRC>(r)); });
  } else {
  staged<NT, K, Raw<T>>(
      total,
      [&](int idx) {
        const int line = idx & (nl - 1), el = idx >> lg;
        const bool ok = line < nv;
        const int k1 = k10 + (ok ? line : 0);
        Raw<T> r;
        r.mode = 0;
        if (SRC == SRC_BUF) {
          r.w = a.buf[base + (k1 - k10) + el * sl];
        } else {
          const int k2 = a.axis == 1 ? el : o;
          const int k3 = a.axis == 1 ? o : el;
          r = spec_fetch<D, T, SRC>(a, k1, k2, k3, interior);
        }
        if (!ok) r.mode = -1;
        return r;
      },
      [&](int idx, const Raw<T>& r) { lds[idx] = tile_value<FWD>(raw_value<T, SRC>(r)); });
  }
}

// ... and out of it; returns the thread's share of x'y
template <typename T, int NT, int D, int DST, bool FWD>
__device__ __forceinline__ double lines_store(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int L = a.len;
  const int lg = a.lg, nl = 1 << lg;
  const int tile1 = tile % a.ntile1;
  const int o = tile / a.ntile1;
  const int k10 = tile1 << lg;
  const int nv = min(nl, a.H1 - k10);
  // element indexes of the half spectrum fit 31 bits
  const int s2 = a.H1, s3 = a.H1 * a.g.n[1];
  const int sl = a.axis == 1 ? s2 : s3;
  const int base = k10 + (a.axis == 1 ? o * s3 : o * s2);
  const int total = L << lg;
  constexpr int K = stage_k<T>();
  // a tile whose k1 are all representatives (1 <= k1 <= P1) reads and writes
  // u at the scratch index with the plain sqrt2 scalings of u_to_v / v_to_u
  const bool interior = k10 >= 1 && k10 + nv - 1 <= a.g.P[0];
  double acc = 0.0;
  if (DST == DST_BUF) {
    staged<NT, K, cpx<T>>(
        total, [&](int idx) { return tile_value<FWD>(lds[idx]); },
        [&](int idx, const cpx<T>& v) {
          const int line = idx & (nl - 1), el = idx >> lg;
          if (line < nv) a.buf[base + line + el * sl] = v;
        });
  } else if (DST == DST_U && interior) {
    staged<NT, (K > 2 ? K / 2 : 1), Fetched<T>>(
        total,
        [&](int idx) {
          const int line = idx & (nl - 1), el = idx >> lg;
          Fetched<T> f;
          f.m = lds[idx];
          f.ops = epi_fetch_u(a.epi, base + (line < nv ? line : 0) + el * sl);
          return f;
        },
        [&](int idx, const Fetched<T>& f) {
          const int line = idx & (nl - 1), el = idx >> lg;
          if (line >= nv) return;
          acc += epi_commit_u(a.epi, base + line + el * sl, scale_sq2(f.m), f.ops);
        });
  } else if (DST == DST_U) {
    staged<NT, (K > 2 ? K / 2 : 1), Fetched<T>>(
        total,
        [&](int idx) {
          const int line = idx & (nl - 1), el = idx >> lg;
          const int k1 = k10 + (line < nv ? line : 0);
          const int k2 = a.axis == 1 ? el : o;
          const int k3 = a.axis == 1 ? o : el;
          Fetched<T> f;
          f.m = lds[idx];
          f.ops = epi_fetch_u(a.epi, k1 + a.H1 * (k2 + a.g.n[1] * k3));
          return f;
        },
        [&](int idx, const Fetched<T>& f) {
          const int line = idx & (nl - 1), el = idx >> lg;
          if (line >= nv) return;
          const int k1 = k10 + line;
          const int k2 = a.axis == 1 ? el : o;
          const int k3 = a.axis == 1 ? o : el;
          const int e = k1 + a.H1 * (k2 + a.g.n[1] * k3);
          acc += epi_commit_u(a.epi, e, v_to_u<D, T>(f.m, k1, k2, k3, a.g), f.ops);
        });
  } else {
    staged<NT, (K > 2 ? K / 2 : 1), FetchedBeta<T>>(
        total,
        [&](int idx) {
          const int line = idx & (nl - 1), el = idx >> lg;
          const int k1 = k10 + (line < nv ? line : 0);
          const int k2 = a.axis == 1 ? el : o;
          const int k3 = a.axis == 1 ? o : el;
          FetchedBeta<T> f;
          f.m = lds[idx];
          f.ops = epi_fetch_beta<D>(a.epi, k1, k2, k3, a.g, interior);
          return f;
        },
        [&](int idx, const FetchedBeta<T>& f) {
          const int line = idx & (nl - 1);
          if (line < nv) acc += epi_commit_beta(a.epi, f.m, f.ops);
        });
  }
  return acc;
}

// staged values of the dim-1 pass
template <typename T>
struct Pair {
  cpx<T> A, B;
  int mode;
};

template <typename T>
struct Masked {
  cpx<T> z;
  uint32_t wa, wb;
};

template <typename T>
struct Fetched2 {
  cpx<T> X, Y;
  EpiOps<T> ops;
};

// the mask words of a dimension-1 tile's lines are loaded with the tile (into
// LDS) rather than per element between the transforms: a line's N1 samples
// span at most mask_row(N1) words
constexpr int kMaskWords = 640;
__device__ __forceinline__ int mask_row(int N1) { return (N1 + 31) / 32 + 1; }
template <typename T>
__device__ __forceinline__ bool mask_staged(const PassArgs<T>& a) {
  return a.miss && (2 << a.lg) * mask_row(a.len) <= kMaskWords;
}

// the tile of a dimension-1 pass from the spectrum, exchanged (the first
// transform is inverse), and its mask words
template <typename T, int NT, int D, int SRC>
__device__ __forceinline__ void dim1_load(const PassArgs<T>& a, cpx<T>* lds, uint32_t* mw,
                                          int tile) {
  const int N1 = a.len, H1 = a.H1;
  const int lg = a.lg, np = 1 << lg, ps = a.ps;
  const int p0 = tile << lg;
  const int nl1 = a.nlines - 1;
  constexpr int K = stage_k<T>();
  (void)np, (void)nl1, (void)N1, (void)H1;
  const bool even = (N1 & 1) == 0;
  // the mask words of the tile's lines are loaded with the tile (into LDS)
  // rather than per element between the transforms: a line's N1 samples
  // span at most W words
  constexpr int kMR = (kMaskWords + NT - 1) / NT;
  const int W = mask_row(N1);
  const int nlt = 2 * np;
  const bool stage_mask = mask_staged(a);
  uint32_t mreg[kMR];
  if (stage_mask) {
    const int64_t nwords = ((int64_t)a.nlines * N1 + 31) >> 5;
#pragma unroll
    for (int r = 0; r < kMR; ++r) {
      const int i = threadIdx.x + r * NT;
      const int ll = i / W, j = i - ll * W;
      const int64_t l = 2 * (int64_t)p0 + ll;
      const int64_t w = ((l * N1) >> 5) + j;
      const bool ok = i < nlt * W && l < a.nlines && w < nwords;
      const uint32_t v = a.miss[ok ? w : 0];
      mreg[r] = ok ? v : 0u;
    }
  }
  const int tot = H1 << lg;
  staged<NT, K, Pair<T>>(
      tot,
      [&](int idx) {
        const int p = udiv(idx, H1, a.h1m);
        const int k = idx - p * H1;
        const int la = 2 * (p0 + p);
        Pair<T> r;
        r.mode = 0;
        r.B = {(T)0, (T)0};
        if (SRC == SRC_BUF) {
          r.A = a.buf[min(la, nl1) * H1 + k];
          r.B = a.buf[min(la + 1, nl1) * H1 + k];
        } else {   // 1D: a single line
          const Raw<T> w = spec_fetch<D, T, SRC>(a, k, 0, 0, false);
          r.A = w.w;
          r.mode = w.mode;
        }
        return r;
      },
      [&](int idx, const Pair<T>& r) {
        const int p = udiv(idx, H1, a.h1m);
        const int k = idx - p * H1;
        const int la = 2 * (p0 + p), lb = la + 1;
        const cpx<T> zero = {(T)0, (T)0};
        cpx<T> A = la < a.nlines ? (SRC == SRC_BUF ? r.A : u_scale(r.A, r.mode)) : zero;
        cpx<T> B = (SRC == SRC_BUF && lb < a.nlines) ? r.B : zero;
        if (k == 0 || (even && k == H1 - 1)) {  // DC / Nyquist of a real line are real
          A.y = 0;
          B.y = 0;
        }
        // A + i B and its Hermitian partner, exchanged: the transform is inverse
        lds[k * ps + p] = {A.y + B.x, A.x - B.y};
        if (k > 0 && N1 - k != k) lds[(N1 - k) * ps + p] = {B.x - A.y, A.x + B.y};
      });
  if (stage_mask) {
#pragma unroll
    for (int r = 0; r < kMR; ++r)
      if ((int)threadIdx.x + r * NT < kMaskWords) mw[threadIdx.x + r * NT] = mreg[r];
  }
}

// ... from real samples
template <typename T, int NT>
__device__ __forceinline__ void dim1_load_real(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int N1 = a.len, H1 = a.H1;
  const int lg = a.lg, np = 1 << lg, ps = a.ps;
  const int p0 = tile << lg;
  const int nl1 = a.nlines - 1;
  constexpr int K = stage_k<T>();
  (void)np, (void)nl1, (void)N1, (void)H1;
  const int totr = N1 << lg;
  staged<NT, K, cpx<T>>(
      totr,
      [&](int idx) {
        const int p = udiv(idx, N1, a.n1m);
        const int n = idx - p * N1;
        const int la = 2 * (p0 + p);
        return cpx<T>{a.real_in[(int64_t)min(la, nl1) * N1 + n],
                      a.real_in[(int64_t)min(la + 1, nl1) * N1 + n]};
      },
      [&](int idx, const cpx<T>& r) {
        const int p = udiv(idx, N1, a.n1m);
        const int n = idx - p * N1;
        const int la = 2 * (p0 + p), lb = la + 1;
        const T xa = la < a.nlines ? r.x * a.scale : (T)0;
        const T xb = lb < a.nlines ? r.y * a.scale : (T)0;
        lds[n * ps + p] = {xa, xb};
      });
}

// the samples after the inverse transform (exchanged in LDS), masked and
// scaled: in place and unexchanged for the forward transform, or (C2R) out
template <typename T, int NT, bool C2R>
__device__ __forceinline__ void dim1_mask(const PassArgs<T>& a, cpx<T>* lds, const uint32_t* mw,
                                          int tile) {
  const int N1 = a.len, H1 = a.H1;
  const int lg = a.lg, np = 1 << lg, ps = a.ps;
  const int p0 = tile << lg;
  const int nl1 = a.nlines - 1;
  constexpr int K = stage_k<T>();
  (void)np, (void)nl1, (void)N1, (void)H1;
  const int W = mask_row(N1);
  const bool stage_mask = mask_staged(a);
  const int totr = N1 << lg;
  if (!C2R && (stage_mask || !a.miss) && np <= NT) {
    // the mask in place from LDS: a thread keeps one line pair p (NT is a
    // multiple of np), so its lines, their staged mask rows and the bit
    // offset of sample 0 in their first word are fixed; per sample only
    // the word and bit of o + n are formed
    const int p = (int)threadIdx.x & (np - 1);
    const int dn = NT >> lg;
    const int la = 2 * (p0 + p), lb = la + 1;
    const T sa0 = la < a.nlines ? a.scale : (T)0;
    const T sb0 = lb < a.nlines ? a.scale : (T)0;
    const int oa = (int)(((int64_t)la * N1) & 31), ob = (int)(((int64_t)lb * N1) & 31);
    const uint32_t* ra = mw + (2 * p) * W;
    const uint32_t* rb = ra + W;
    cpx<T>* q = lds + ((int)threadIdx.x >> lg) * ps + p;
    for (int n = (int)threadIdx.x >> lg; n < N1; n += dn, q += dn * ps) {
      T sa = sa0, sb = sb0;
      if (stage_mask) {
        const int ta = oa + n, tb = ob + n;
        if ((ra[ta >> 5] >> (ta & 31)) & 1u) sa = (T)0;
        if ((rb[tb >> 5] >> (tb & 31)) & 1u) sb = (T)0;
      }
      const cpx<T> z = *q;   // (line b, line a): exchanged
      *q = {z.y * sa, z.x * sb};
    }
    return;
  }
staged<NT, K, Masked<T>>(
    totr,
    [&](int idx) {
      const int p = idx & (np - 1);
      const int n = idx >> lg;
      const int la = 2 * (p0 + p);
      Masked<T> r;
      r.z = cswap(lds[n * ps + p]);
      r.wa = r.wb = 0u;
      if (stage_mask) {
        const int64_t sa = (int64_t)la * N1 + n, sb = sa + N1;
        r.wa = mw[(2 * p) * W + (int)((sa >> 5) - (((int64_t)la * N1) >> 5))];
        r.wb = mw[(2 * p + 1) * W + (int)((sb >> 5) - (((int64_t)(la + 1) * N1) >> 5))];
      } else if (a.miss) {
        r.wa = a.miss[((int64_t)min(la, nl1) * N1 + n) >> 5];
        r.wb = a.miss[((int64_t)min(la + 1, nl1) * N1 + n) >> 5];
      }
      return r;
    },
    [&](int idx, const Masked<T>& r) {
      const int p = idx & (np - 1);
      const int n = idx >> lg;
      const int la = 2 * (p0 + p), lb = la + 1;
      const int64_t sa_i = (int64_t)la * N1 + n, sb_i = (int64_t)lb * N1 + n;
      const bool ma = (r.wa >> (sa_i & 31)) & 1u;
      const bool mb = (r.wb >> (sb_i & 31)) & 1u;
      const T sa = (la < a.nlines && !ma) ? a.scale : (T)0;
      const T sb = (lb < a.nlines && !mb) ? a.scale : (T)0;
      cpx<T> z = r.z;
      z.x *= sa;
      z.y *= sb;
      if (C2R) {
        if (la < a.nlines) a.real_out[sa_i] = z.x;
        if (lb < a.nlines) a.real_out[sb_i] = z.y;
      } else {
        lds[n * ps + p] = z;
      }
    });
}

// the forward transform's two real lines out of the tile
template <typename T, int NT, int D, int DST>
__device__ __forceinline__ double dim1_store(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int N1 = a.len, H1 = a.H1;
  const int lg = a.lg, np = 1 << lg, ps = a.ps;
  const int p0 = tile << lg;
  const int nl1 = a.nlines - 1;
  constexpr int K = stage_k<T>();
  (void)np, (void)nl1, (void)N1, (void)H1;
  double acc = 0.0;
  const int tot = H1 << lg;
  const T half = (T)0.5;
  if (DST == DST_BUF) {
    staged<NT, K, Pair<T>>(
        tot,
        [&](int idx) {
          const int p = udiv(idx, H1, a.h1m);
          const int k = idx - p * H1;
          Pair<T> r;
          r.A = lds[k * ps + p];
          r.B = lds[(k == 0 ? 0 : N1 - k) * ps + p];
          r.mode = 0;
          return r;
        },
        [&](int idx, const Pair<T>& r) {
          const int p = udiv(idx, H1, a.h1m);
          const int k = idx - p * H1;
          const int la = 2 * (p0 + p), lb = la + 1;
          if (la >= a.nlines) return;
          const cpx<T> X = r.A, Y = r.B;
          const cpx<T> Va = {half * (X.x + Y.x), half * (X.y - Y.y)};
          const cpx<T> Vb = {half * (X.y + Y.y), half * (Y.x - X.x)};
          a.buf[la * H1 + k] = Va;
          if (lb < a.nlines) a.buf[lb * H1 + k] = Vb;
        });
  } else if (DST == DST_U) {   // 1D: line 0 only
    staged<NT, (K > 2 ? K / 2 : 1), Fetched2<T>>(
        tot,
        [&](int idx) {
          const int p = udiv(idx, H1, a.h1m);
          const int k = idx - p * H1;
          Fetched2<T> f;
          f.X = lds[k * ps + p];
          f.Y = lds[(k == 0 ? 0 : N1 - k) * ps + p];
          f.ops = epi_fetch_u(a.epi, k);
          return f;
        },
        [&](int idx, const Fetched2<T>& f) {
          const int p = udiv(idx, H1, a.h1m);
          const int k = idx - p * H1;
          if (2 * (p0 + p) >= a.nlines) return;
          const cpx<T> Va = {half * (f.X.x + f.Y.x), half * (f.X.y - f.Y.y)};
          acc += epi_commit_u(a.epi, k, v_to_u<D, T>(Va, k, 0, 0, a.g), f.ops);
        });
  } else {   // 1D: line 0 only
    staged<NT, (K > 2 ? K / 2 : 1), FetchedBeta<T>>(
        tot,
        [&](int idx) {
          const int p = udiv(idx, H1, a.h1m);
          const int k = idx - p * H1;
          const cpx<T> X = lds[k * ps + p], Y = lds[(k == 0 ? 0 : N1 - k) * ps + p];
          FetchedBeta<T> f;
          f.m = {half * (X.x + Y.x), half * (X.y - Y.y)};
          f.ops = epi_fetch_beta<D>(a.epi, k, 0, 0, a.g, false);
          return f;
        },
        [&](int idx, const FetchedBeta<T>& f) {
          if (2 * (p0 + udiv(idx, H1, a.h1m)) < a.nlines) acc += epi_commit_beta(a.epi, f.m, f.ops);
        });
  }
  return acc;
}

// ===========================================================================
// Long 1D lines: the length-F DFT in four steps over the (B rows x A columns)
// view of the scratch spectrum (position col + A*row).  Column passes
// transform along rows (length B, stride A, 2^lg adjacent columns per
// workgroup), row passes along columns (length A, contiguous, 2^lg rows).
// Direct (F = N):
//   MTM   col FIRST (inverse, twiddle)  row MTM (inverse, mask at the time
//         index t = row + B*col, forward, twiddle)  col LAST (forward, epilogue)
// Bluestein (F = M >= 2N - 1, chirp w_n = exp(-i pi n^2/N)):
//   MTM   col FIRST (x conj(w), forward, twiddle)  row CONV_INV (forward,
//         x FFT_M(w)/M = conj(bfw), inverse, twiddle)  col MID (inverse, x conj(w), mask,
//         x w, forward, twiddle)  row CONV_FWD  col LAST (inverse, x w, epilogue)
// ===========================================================================
// (unstaged: groups of loads held in registers were slower here, 44 -> 48 us
// for 49999 samples in FP32 and 57 -> 66 ms for a mixed batch)
__device__ __forceinline__ bool miss_bit(const uint32_t* m, int64_t s) {
  return m && ((m[s >> 5] >> (s & 31)) & 1u);
}

template <typename T>
__device__ __forceinline__ cpx<T> twf(const PassArgs<T>& a, int64_t j, bool inv) {
  cpx<T> w = a.twF[j];
  if (inv) w.y = -w.y;
  return w;
}

template <typename T>
__device__ __forceinline__ cpx<T> chirp_at(const PassArgs<T>& a, int64_t n, bool conj_) {
  cpx<T> w = a.chirp[n];
  if (conj_) w.y = -w.y;
  return w;
}

// spectrum value k (< N) of a Hermitian line held as its half (k < H1)
template <typename T, int SRC>
__device__ __forceinline__ cpx<T> half_load(const PassArgs<T>& a, int64_t k) {
  const bool far = k >= a.H1;
  const cpx<T> v =
      raw_value<T, SRC>(spec_fetch<1, T, SRC>(a, (int)(far ? a.len - k : k), 0, 0, false));
  return {v.x, far ? -v.y : v.y};
}

// FWD: the pass's first transform is forward (else the tile holds exchanged
// values, see line_dft)
template <typename T, int NT, int MODE, int SRC, bool FWD>
__device__ __forceinline__ void col_load(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int A = a.A, B = a.B, lg = a.lg, nl = 1 << lg;
  const int64_t N = a.len;
  const bool bs = a.obs != 0;
  const int c0 = tile << lg;
  const int nv = min(nl, A - c0);
  for (int idx = threadIdx.x; idx < (B << lg); idx += NT) {
    const int line = idx & (nl - 1), r = idx >> lg;
    const int64_t n = c0 + line + (int64_t)A * r;
    cpx<T> v = {(T)0, (T)0};
    if (line < nv) {
      if (MODE == C_FIRST) {
        if (n < N) {
          v = half_load<T, SRC>(a, n);
          v = bs ? cmul(v, chirp_at(a, n, true)) : cswap(v);   // direct: inverse first
        }
      } else if (MODE == C_REAL_IN) {
        if (n < N) {
          v = {a.real_in[n] * a.scale, (T)0};
          if (bs) v = cmul(v, chirp_at(a, n, false));
        }
      } else {
        v = tile_value<FWD>(a.buf[n]);
      }
    }
    lds[r * nl + line] = v;
  }
}

// outer Bluestein, between the convolutions (exchanged values in LDS):
// conv -> x_n = conj(w_n) conv_n, masked real part; then x w for the forward
// transform, or (C2R) out
template <typename T, int NT, bool C2R>
__device__ __forceinline__ void col_mid(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int A = a.A, B = a.B, lg = a.lg, nl = 1 << lg;
  const int64_t N = a.len;
  const int c0 = tile << lg;
  const int nv = min(nl, A - c0);
  for (int idx = threadIdx.x; idx < (B << lg); idx += NT) {
    const int line = idx & (nl - 1), r = idx >> lg;
    const int64_t n = c0 + line + (int64_t)A * r;
    cpx<T>* q = lds + r * nl + line;
    T xr = (T)0;
    if (line < nv && n < N && !miss_bit(a.miss, n))
      xr = cmul(cswap(*q), chirp_at(a, n, true)).x * a.scale;
    if (C2R) {
      if (line < nv && n < N) a.real_out[n] = xr;
    } else {
      const cpx<T> w = n < N ? chirp_at(a, n, false) : cpx<T>{(T)0, (T)0};
      *q = {xr * w.x, xr * w.y};
    }
  }
}

// FWD: the pass's last transform was forward.  Into the scratch spectrum (with
// the four-step twiddle: conjugate after an inverse transform) or, the last
// pass, into beta / u
template <typename T, int NT, int DST, bool FWD>
__device__ __forceinline__ double col_store(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int A = a.A, B = a.B, lg = a.lg, nl = 1 << lg;
  const bool bs = a.obs != 0;
  const int c0 = tile << lg;
  const int nv = min(nl, A - c0);
  double acc = 0.0;
  for (int idx = threadIdx.x; idx < (B << lg); idx += NT) {
    const int line = idx & (nl - 1), r = idx >> lg;
    if (line >= nv) continue;
    const int col = c0 + line;
    cpx<T> v = tile_value<FWD>(lds[r * nl + line]);
    if (DST == DST_BUF) {
      v = cmul(v, twf(a, (int64_t)col * r, !FWD));
      a.buf[col + (int64_t)A * r] = v;
    } else {
      const int64_t k = col + (int64_t)A * r;
      if (k < a.H1) {
        if (bs) v = cmul(cswap(v), chirp_at(a, k, false));   // ends in the inverse transform
        if constexpr (DST == DST_U)
          acc += epi_commit_u(a.epi, k, v_to_u<1, T>(v, (int)k, 0, 0, a.g), epi_fetch_u(a.epi, k));
        else
          acc += epi_commit_beta(a.epi, v, epi_fetch_beta<1>(a.epi, (int)k, 0, 0, a.g, false));
      }
    }
  }
  return acc;
}

template <typename T, int NT, bool REAL, bool FWD>
__device__ __forceinline__ void row_load(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int A = a.A, B = a.B, lg = a.lg, nl = 1 << lg, ps = a.ps;
  const int r0 = tile << lg;
  const int nv = min(nl, B - r0);
  for (int idx = threadIdx.x; idx < (A << lg); idx += NT) {
    const int line = udiv(idx, A, a.am);
    const int c = idx - line * A;
    const int row = r0 + line;
    cpx<T> v = {(T)0, (T)0};
    if (line < nv) {
      if (REAL) v = {a.real_in[row + (int64_t)B * c] * a.scale, (T)0};
      else v = a.buf[c + (int64_t)A * row];
    }
    lds[c * ps + line] = tile_value<FWD>(v);
  }
}

// direct: the samples after the inverse transform (exchanged), masked
template <typename T, int NT, bool C2R>
__device__ __forceinline__ void row_mask(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int A = a.A, B = a.B, lg = a.lg, nl = 1 << lg, ps = a.ps;
  const int r0 = tile << lg;
  const int nv = min(nl, B - r0);
  for (int idx = threadIdx.x; idx < (A << lg); idx += NT) {
    const int line = udiv(idx, A, a.am);
    const int c = idx - line * A;
    const int64_t t = r0 + line + (int64_t)B * c;
    cpx<T>* q = lds + c * ps + line;
    const T xr = (line < nv && !miss_bit(a.miss, t)) ? q->y * a.scale : (T)0;
    if (C2R) {
      if (line < nv) a.real_out[t] = xr;
    } else {
      *q = {xr, (T)0};
    }
  }
}

// the product with the kernel spectrum, exchanged for the inverse FFT (the
// inverse kernel is the conjugate of the forward one, and both are even, so
// its spectrum is the conjugate too)
template <typename T, int NT, bool INV>
__device__ __forceinline__ void row_conv(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int A = a.A, B = a.B, lg = a.lg, nl = 1 << lg, ps = a.ps;
  const int r0 = tile << lg;
  const int nv = min(nl, B - r0);
  for (int idx = threadIdx.x; idx < (A << lg); idx += NT) {
    const int line = udiv(idx, A, a.am);
    const int c = idx - line * A;
    cpx<T>* q = lds + c * ps + line;
    if (line < nv) {
      cpx<T> bk = a.bfw[r0 + line + (int64_t)B * c];
      if (INV) bk.y = -bk.y;
      *q = cswap(cmul(*q, bk));
    }
  }
}

// FWD as in col_store
template <typename T, int NT, bool FWD>
__device__ __forceinline__ void row_store(const PassArgs<T>& a, cpx<T>* lds, int tile) {
  const int A = a.A, B = a.B, lg = a.lg, nl = 1 << lg, ps = a.ps;
  const int r0 = tile << lg;
  const int nv = min(nl, B - r0);
  for (int idx = threadIdx.x; idx < (A << lg); idx += NT) {
    const int line = udiv(idx, A, a.am);
    const int c = idx - line * A;
    if (line >= nv) continue;
    const int row = r0 + line;
    const cpx<T> v = tile_value<FWD>(lds[c * ps + line]);
    a.buf[c + (int64_t)A * row] = cmul(v, twf(a, (int64_t)row * c, !FWD));
  }
}

// one workgroup's tile of a pass; LD, MID, ST < 0: the steps PassArgs names.
// FORM: the line transforms it is compiled for, FORM_FFT (direct, Rader,
// Bluestein), FORM_DENSE or any (together they take more registers: the FP32
// 256^3 product 357 against 374 us)
enum { FORM_FFT = 0, FORM_DENSE = 1, FORM_ANY = 2 };
// args: the kernel's arguments in memory, where it loads them again.  The 3D
// line store to beta uses most of them; held from the load on, they went
// through the transform as spilled scalars, read back one by one in the store's
// loops, a fifth of the kernel's vector instructions.  (Adjoint of 256^3 FP32
// 148 -> 138 us, FP64 240 -> 221; the dense kernels, 127^3, took 1% longer with
// it, and the store to a 2D beta 3%.)
template <typename T>
using ArgsPtr = const __attribute__((address_space(4))) PassArgs<T>*;
template <typename T>
__device__ __forceinline__ PassArgs<T> load_args(ArgsPtr<T> p) {
  asm volatile("" : "+s"(p));   // (not the values loaded before)
  return *(const PassArgs<T>*)p;
}
template <typename T, int NT, int E, int LD, int MID, int ST, int FORM>
__device__ __forceinline__ void pass_body(const PassArgs<T>& a, int tile,
                                          ArgsPtr<T> args = nullptr) {
  const int ld = LD < 0 ? a.ld : LD, mid = MID < 0 ? a.mid : MID, st = ST < 0 ? a.st : ST;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  cpx<T>* lds = reinterpret_cast<cpx<T>*>(smem_raw);
  __shared__ uint32_t mw[kMaskWords];
  // finished instances: the flag is read beside the loads, not before them
  const int dflag = a.done ? *a.done : 0;
  const int pl = plan_load(a.plan);
  constexpr bool kShort = NT * E <= 4096;   // line, column and row tiles
  switch (ld) {
    case LD_DIM1_BUF: dim1_load<T, NT, 2, SRC_BUF>(a, lds, mw, tile); break;
    case LD_DIM1_U: dim1_load<T, NT, 1, SRC_U>(a, lds, mw, tile); break;
    case LD_DIM1_BETA: dim1_load<T, NT, 1, SRC_BETA>(a, lds, mw, tile); break;
    case LD_DIM1_REAL: dim1_load_real<T, NT>(a, lds, tile); break;
    default:
      if constexpr (kShort) {
        switch (ld) {
          case LD_LINES_BUF_FWD: lines_load<T, NT, 3, SRC_BUF, true>(a, lds, tile); break;
          case LD_LINES_BUF_INV: lines_load<T, NT, 3, SRC_BUF, false>(a, lds, tile); break;
          case LD_LINES_U2: lines_load<T, NT, 2, SRC_U, false>(a, lds, tile); break;
          case LD_LINES_U3: lines_load<T, NT, 3, SRC_U, false>(a, lds, tile); break;
          case LD_LINES_BETA2: lines_load<T, NT, 2, SRC_BETA, false>(a, lds, tile); break;
          case LD_LINES_BETA3: lines_load<T, NT, 3, SRC_BETA, false>(a, lds, tile); break;
          case LD_COL_FIRST_U: col_load<T, NT, C_FIRST, SRC_U, false>(a, lds, tile); break;
          case LD_COL_FIRST_BETA: col_load<T, NT, C_FIRST, SRC_BETA, false>(a, lds, tile); break;
          case LD_COL_REAL: col_load<T, NT, C_REAL_IN, SRC_REAL, true>(a, lds, tile); break;
          case LD_COL_BUF_FWD: col_load<T, NT, C_LAST, SRC_BUF, true>(a, lds, tile); break;
          case LD_COL_BUF_INV: col_load<T, NT, C_LAST, SRC_BUF, false>(a, lds, tile); break;
          case LD_ROW_FWD: row_load<T, NT, false, true>(a, lds, tile); break;
          case LD_ROW_INV: row_load<T, NT, false, false>(a, lds, tile); break;
          case LD_ROW_REAL: row_load<T, NT, true, true>(a, lds, tile); break;
          default: break;
        }
      }
  }
  if (dflag) return;
  __syncthreads();
#pragma unroll 1
  for (int turn = 0;; ++turn) {
    if constexpr (LD >= LD_COL_FIRST_U) {   // four-step passes transform directly
      lds_fft<T, E, NT>(lds, pl, a.lg, a.ps, a.tw);
    } else if constexpr (FORM == FORM_DENSE) {
      dense_dft<T, NT>(lds, a.dense, a.len, a.lg, a.ps);
    } else {
      bool fft = true;
      if constexpr (FORM == FORM_ANY && NT == 256) {   // (dense tiles run on 256 threads)
        if (a.bs == 3) {
          dense_dft_call<T, NT>((LdsTile<T>)lds, a.dense, a.len, a.lg, a.ps);
          fft = false;
        }
      }
      if (fft) line_dft<T, E, NT>(lds, a, pl, a.lg, a.ps);
    }
    if (turn == 1 || mid == MID_NONE) break;
    switch (mid) {
      case MID_DIM1_MASK: dim1_mask<T, NT, false>(a, lds, mw, tile); break;
      default:
        if constexpr (kShort) {
          switch (mid) {
            case MID_COL: col_mid<T, NT, false>(a, lds, tile); break;
            case MID_ROW_MASK: row_mask<T, NT, false>(a, lds, tile); break;
            case MID_ROW_CONV_INV: row_conv<T, NT, true>(a, lds, tile); break;
            case MID_ROW_CONV_FWD: row_conv<T, NT, false>(a, lds, tile); break;
            default: break;
          }
        }
    }
    __syncthreads();
  }
  double acc = 0.0;
  switch (st) {
    case ST_DIM1_BUF: dim1_store<T, NT, 2, DST_BUF>(a, lds, tile); return;
    case ST_DIM1_REAL: dim1_mask<T, NT, true>(a, lds, mw, tile); return;
    case ST_DIM1_U: acc = dim1_store<T, NT, 1, DST_U>(a, lds, tile); break;
    case ST_DIM1_BETA: acc = dim1_store<T, NT, 1, DST_BETA>(a, lds, tile); break;
    default:
      if constexpr (kShort) {
        switch (st) {
          case ST_LINES_BUF_FWD: lines_store<T, NT, 3, DST_BUF, true>(a, lds, tile); return;
          case ST_LINES_BUF_INV: lines_store<T, NT, 3, DST_BUF, false>(a, lds, tile); return;
          case ST_LINES_U2: acc = lines_store<T, NT, 2, DST_U, true>(a, lds, tile); break;
          case ST_LINES_U3: acc = lines_store<T, NT, 3, DST_U, true>(a, lds, tile); break;
          case ST_LINES_BETA2: acc = lines_store<T, NT, 2, DST_BETA, true>(a, lds, tile); break;
          case ST_LINES_BETA3:
            if constexpr (ST == ST_LINES_BETA3 && FORM == FORM_FFT)
              acc = lines_store<T, NT, 3, DST_BETA, true>(load_args<T>(args), lds, tile);
            else
              acc = lines_store<T, NT, 3, DST_BETA, true>(a, lds, tile);
            break;
          case ST_COL_BUF_FWD: col_store<T, NT, DST_BUF, true>(a, lds, tile); return;
          case ST_COL_BUF_INV: col_store<T, NT, DST_BUF, false>(a, lds, tile); return;
          case ST_COL_U: acc = col_store<T, NT, DST_U, true>(a, lds, tile); break;
          case ST_COL_BETA: acc = col_store<T, NT, DST_BETA, true>(a, lds, tile); break;
          case ST_COL_REAL: col_mid<T, NT, true>(a, lds, tile); return;
          case ST_ROW_FWD: row_store<T, NT, true>(a, lds, tile); return;
          case ST_ROW_INV: row_store<T, NT, false>(a, lds, tile); return;
          case ST_ROW_REAL: row_mask<T, NT, true>(a, lds, tile); return;
          default: break;
        }
      }
  }
  if (a.epi.dot_part) store_partial(a.epi.dot_part, acc, tile);
}

// waves per SIMD asked of the compiler for the pass kernels (of 512 registers
// a SIMD lane: 96 per thread in FP32, 168 in FP64; a 1024-thread workgroup
// needs four waves, 128 registers).  The dense and the mixed FP32 ones keep
// four as well, nothing spilled at 128 registers: a mixed launch of 512 threads
// 39.2 to 36.0 us (70 spilled at 96), the dense product of 127^3 80 to 77.
// The mixed FP64 ones two (256 threads 82 to 73 us; 106 spilled at 168)
template <typename T, int NT, int E, int LD, int FORM>
constexpr int pass_waves() {
  if (E == 16 || NT >= 1024 || (sizeof(T) == 4 && (LD < 0 || FORM == FORM_DENSE))) return 4;
  if (LD < 0) return 2;
  return sizeof(T) == 4 ? 5 : 3;
}

// a pass of one instance
template <typename T, int NT, int E, int LD, int MID, int ST, int FORM>
__global__ __launch_bounds__(NT, (pass_waves<T, NT, E, LD, FORM>())) void k_pass(PassArgs<T> a) {
  if constexpr (ST == ST_LINES_BETA3 && FORM == FORM_FFT) {
    const ArgsPtr<T> args = (ArgsPtr<T>)__builtin_amdgcn_kernarg_segment_ptr();
    pass_body<T, NT, E, LD, MID, ST, FORM>(load_args<T>(args), xcd_block(), args);
  } else {
    pass_body<T, NT, E, LD, MID, ST, FORM>(a, xcd_block());
  }
}

// member and tile of a block of a launch over several instances; member < 0:
// a filler
struct BlockMap {
  int member, tile;
};

// passes of several instances (LD < 0: each its own kind): the host's block map keeps
// adjacent tiles of an instance on one XCD (block b runs on XCD b % 8).
template <typename T, int NT, int E, int LD, int MID, int ST, int FORM>
__global__ __launch_bounds__(NT, (pass_waves<T, NT, E, LD, FORM>())) void kb_pass(
    const PassArgs<T>* __restrict__ tab, const BlockMap* __restrict__ map) {
  const int i = uniform(map[blockIdx.x].member), tile = uniform(map[blockIdx.x].tile);
  if (i < 0) return;
  const PassArgs<T> a = tab[i];  // loaded before any store: stays in scalar registers
  pass_body<T, NT, E, LD, MID, ST, FORM>(a, tile);
}

// beta <-> u (exact: a signed permutation), one thread per half-spectrum element.
// sign = 0 moves a diagonal (L1, L2, P..) instead: the same permutation, no signs.
template <int D, typename T>
__global__ __launch_bounds__(256) void k_beta_to_u(const T* __restrict__ beta, cpx<T>* u,
                                                   MapGeom g, int H1, int64_t nc, int sign) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nc) return;
  const int k1 = (int)(e % H1);
  const int64_t r = e / H1;
  const int k2 = (int)(r % g.n[1]);
  const int k3 = (int)(r / g.n[1]);
  int64_t re, im;
  bool vertex, neg;
  cpx<T> w = {(T)0, (T)0};
  if (scatter_targets<D>(k1, k2, k3, g, re, im, vertex, neg)) {
    w.x = beta[re];
    if (!vertex) w.y = (neg && sign) ? -beta[im] : beta[im];
  }
  u[e] = w;
}

template <int D, typename T>
__global__ __launch_bounds__(256) void k_u_to_beta(const cpx<T>* __restrict__ u, T* beta,
                                                   MapGeom g, int H1, int64_t nc, int sign) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nc) return;
  const int k1 = (int)(e % H1);
  const int64_t r = e / H1;
  const int k2 = (int)(r % g.n[1]);
  const int k3 = (int)(r / g.n[1]);
  int64_t re, im;
  bool vertex, neg;
  if (scatter_targets<D>(k1, k2, k3, g, re, im, vertex, neg)) {
    const cpx<T> w = u[e];
    beta[re] = w.x;
    if (!vertex) beta[im] = (neg && sign) ? -w.y : w.y;
  }
}

// bit i set when u slot i holds a beta entry (32 slots = 16 elements per thread)
template <int D>
__global__ __launch_bounds__(256) void k_u_valid(uint32_t* bits, MapGeom g, int H1, int64_t nc) {
  const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w * 16 >= nc) return;
  uint32_t word = 0;
  for (int j = 0; j < 16; ++j) {
    const int64_t e = w * 16 + j;
    if (e >= nc) break;
    const int k1 = (int)(e % H1);
    const int64_t r = e / H1;
    const int k2 = (int)(r % g.n[1]);
    const int k3 = (int)(r / g.n[1]);
    int64_t re, im;
    bool vertex, neg;
    if (scatter_targets<D>(k1, k2, k3, g, re, im, vertex, neg)) {
      word |= 1u << (2 * j);
      if (!vertex) word |= 1u << (2 * j + 1);
    }
  }
  bits[w] = word;
}

__device__ __forceinline__ bool slot_valid(const uint32_t* v, int64_t i) {
  return (v[i >> 5] >> (i & 31)) & 1u;
}

// ===========================================================================
// Vector kernels: preconditioner and CG
// ===========================================================================

// fft_kkt.jl:297-305.  The reference forms Minv = 1/(1+L1),
// S = 1/(L1 - L2^2 Minv), P12 = -L2 S Minv, P11 = Minv + Minv L2 S L2 Minv.  With
// det = (1+L1) L1 - L2^2 = L1 + 4 s1 s2 these are exactly P11 = L1/det,
// P12 = -L2/det, P22 = (1+L1)/det, evaluated here without the cancellation of
// L1 - L2^2 Minv when s1 and s2 differ by many orders of magnitude.
template <typename T>
__device__ __forceinline__ void precond_entries(T a, T b, T& l1, T& l2, T& p11, T& p12, T& p22) {
  l1 = a + b;
  l2 = a - b;
  const T inv = (T)1 / (l1 + (T)4 * a * b);
  p11 = l1 * inv;
  p12 = -l2 * inv;
  p22 = ((T)1 + l1) * inv;
}

template <typename T>
__global__ __launch_bounds__(256) void k_precond_build(const T* __restrict__ s1,
                                                       const T* __restrict__ s2, T* L1, T* L2,
                                                       T* P11, T* P12, T* P22, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  T l1, l2, p11, p12, p22;
  precond_entries<T>(s1[i], s2[i], l1, l2, p11, p12, p22);
  L1[i] = l1;
  L2[i] = l2;
  P11[i] = p11;
  P12[i] = p12;
  P22[i] = p22;
}

// fft_kkt.jl:81-82
template <typename T>
__global__ __launch_bounds__(256) void k_precond_apply(const T* __restrict__ x, T* y,
                                                       const T* __restrict__ P11,
                                                       const T* __restrict__ P12,
                                                       const T* __restrict__ P22, T alpha,
                                                       T beta, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const T xb = x[i], xz = x[n + i];
  T yb = alpha * (P11[i] * xb + P12[i] * xz);
  T yz = alpha * (P12[i] * xb + P22[i] * xz);
  if (beta != (T)0) {
    yb += beta * y[i];
    yz += beta * y[n + i];
  }
  y[i] = yb;
  y[n + i] = yz;
}

// per-block partials of up to 8 quantities: part[q * gridDim.x + block]
template <int NQ>
__device__ __forceinline__ void store_partials(double* part, const double (&acc)[NQ],
                                               const int (&ops)[NQ]) {
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    double r;
    if (ops[q] == 0) r = block_reduce(acc[q], OpSum());
    else if (ops[q] == 1) r = block_reduce(acc[q], OpMax());
    else r = block_reduce(acc[q], OpMin());
    if (threadIdx.x == 0) part[q * gridDim.x + blockIdx.x] = r;
  }
}

// ===========================================================================
// FFTNLPModel and the full KKT operators (elementwise, op precision T)
// ===========================================================================

// sum y^2, sum beta * Mtz0, sum c  (fft_model.jl:73)
template <typename T>
__global__ __launch_bounds__(256) void k_obj_parts(const T* __restrict__ y,
                                                   const T* __restrict__ x,
                                                   const T* __restrict__ mtz0, int64_t n,
                                                   double* part) {
  double a[3] = {0, 0, 0};
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double yi = y[i];
    a[0] += yi * yi;
    a[1] += (double)x[i] * (double)mtz0[i];
    a[2] += (double)x[n + i];
  }
  const int ops[3] = {0, 0, 0};
  store_partials<3>(part, a, ops);
}

// g_b = MtM beta - Mtz0 (in place on g_b), g_c = lambda  (fft_model.jl:77-89)
template <typename T>
__global__ __launch_bounds__(256) void k_grad_tail(T* g, const T* __restrict__ mtz0, T lam,
                                                   int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    g[i] = g[i] - mtz0[i];
    g[n + i] = lam;
  }
}

// c_b = -beta - c, c_c = beta - c  (fft_model.jl:91-101)
template <typename T>
__global__ __launch_bounds__(256) void k_cons(const T* __restrict__ x, T* cv, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const T b = x[i], c = x[n + i];
    cv[i] = -b - c;
    cv[n + i] = b - c;
  }
}

// full KKT product after M^T M x_beta is in Mb (fft_kkt.jl:239-246)
template <typename T>
__global__ __launch_bounds__(256) void k_kkt_full(const T* __restrict__ x, T* y,
                                                  const T* __restrict__ Mb, T alpha, T beta,
                                                  int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const T xb = x[i], xz = x[n + i], xs1 = x[2 * n + i], xs2 = x[3 * n + i];
    const T xy1 = x[4 * n + i], xy2 = x[5 * n + i];
    T o0 = alpha * (Mb[i] - xy1 + xy2);
    T o1 = -alpha * (xy1 + xy2);
    T o2 = -alpha * xy1;
    T o3 = -alpha * xy2;
    T o4 = alpha * (-xb - xz - xs1);
    T o5 = alpha * (xb - xz - xs2);
    if (beta != (T)0) {
      o0 += beta * y[i];
      o1 += beta * y[n + i];
      o2 += beta * y[2 * n + i];
      o3 += beta * y[3 * n + i];
      o4 += beta * y[4 * n + i];
      o5 += beta * y[5 * n + i];
    }
    y[i] = o0;
    y[n + i] = o1;
    y[2 * n + i] = o2;
    y[3 * n + i] = o3;
    y[4 * n + i] = o4;
    y[5 * n + i] = o5;
  }
}

// J^T y (fft_kkt.jl:253-275)
template <typename T>
__global__ __launch_bounds__(256) void k_jtprod(const T* __restrict__ x, T* y, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const T y1 = x[i], y2 = x[n + i];
    y[i] = -y1 + y2;
    y[n + i] = -y1 - y2;
    y[2 * n + i] = -y1;
    y[3 * n + i] = -y2;
  }
}

// 6N KKT right-hand side -> condensed 2N right-hand side (fft_kkt.jl:333-335)
template <typename T>
__global__ __launch_bounds__(256) void k_condense(const T* __restrict__ w,
                                                  const T* __restrict__ s1,
                                                  const T* __restrict__ s2, T* b, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const T w1 = w[i], w2 = w[n + i], w3 = w[2 * n + i], w4 = w[3 * n + i];
    const T w5 = w[4 * n + i], w6 = w[5 * n + i], a = s1[i], c = s2[i];
    b[i] = w1 - w3 + w4 - a * w5 + c * w6;
    b[n + i] = w2 - w3 - w4 - a * w5 - c * w6;
  }
}

// condensed solution -> 6N solution, in place on w (fft_kkt.jl:344-350)
template <typename T>
__global__ __launch_bounds__(256) void k_unpack(T* w, const T* __restrict__ x,
                                                const T* __restrict__ s1,
                                                const T* __restrict__ s2, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const T a = s1[i], c = s2[i];
    const T w1 = x[i], w2 = x[n + i];
    T w3 = w[2 * n + i], w4 = w[3 * n + i], w5 = w[4 * n + i], w6 = w[5 * n + i];
    w5 = -(w3 + a * (w1 + w2 + w5));
    w6 = -(w4 + c * (-w1 + w2 + w6));
    w3 = (w3 + w5) / a;
    w4 = (w4 + w6) / c;
    w[i] = w1;
    w[n + i] = w2;
    w[2 * n + i] = w3;
    w[3 * n + i] = w4;
    w[4 * n + i] = w5;
    w[5 * n + i] = w6;
  }
}

}  // namespace csipm
