// Device-side building blocks of libcsipm: complex arithmetic, the Hermitian
// beta <-> DFT packing geometry, Stockham butterflies and block reductions.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "radix_consts.hpp"

namespace csipm {

// ---------------------------------------------------------------------------
// complex numbers (interleaved re, im; 16 B for double, 8 B for float)
// ---------------------------------------------------------------------------
template <typename T>
struct alignas(2 * sizeof(T)) cpx {
  T x, y;
};

template <typename T>
__device__ __forceinline__ cpx<T> cadd(cpx<T> a, cpx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ cpx<T> csub(cpx<T> a, cpx<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T>
__device__ __forceinline__ cpx<T> cmul(cpx<T> a, cpx<T> b) {
  return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T>
__device__ __forceinline__ cpx<T> mul_mi(cpx<T> a) { return {a.y, -a.x}; }   // a * (-i)
// real and imaginary part exchanged: swap(DFT(swap(x))) is the inverse DFT
template <typename T>
__device__ __forceinline__ cpx<T> cswap(cpx<T> a) { return {a.y, a.x}; }

// ---------------------------------------------------------------------------
// Packing geometry.  Per dimension d of length n: M = n/2, P = (n-1)/2,
// self-conjugate indices S = {0, M} (n even) or {0} (n odd), representatives
// R = 1..P, second half H = M+1..M+P, conjugate partner (n - k) mod n.
// The beta vector is the reference's block sequence (vertices, edges, faces,
// interior; Re block then Im block), src/mapping_cpu_kernels.jl:1-351.
// ---------------------------------------------------------------------------
struct MapGeom {
  int d;
  int n[3], M[3], P[3], S[3];
  int64_t N;
  int64_t P12, P13, P23, P123;
  // block offsets; 3D: V, Ek, Ej, Ei, Fi, Fj, Fk, I.  2D: V, Er, Ec, C.
  // 1D: V, R.
  int64_t off[8];
};

// Geometry of the packing for sizes n[0..dim-1] (trailing sizes 1).
inline MapGeom make_map_geom(int dim, const int n_in[3]) {
  MapGeom g{};
  g.d = dim;
  for (int i = 0; i < 3; ++i) {
    const int n = i < dim ? n_in[i] : 1;
    g.n[i] = n;
    g.M[i] = n / 2;
    g.P[i] = (n - 1) / 2;
    g.S[i] = (n % 2 == 0) ? 2 : 1;
  }
  g.N = (int64_t)g.n[0] * g.n[1] * g.n[2];
  g.P12 = (int64_t)g.P[0] * g.P[1];
  g.P13 = (int64_t)g.P[0] * g.P[2];
  g.P23 = (int64_t)g.P[1] * g.P[2];
  g.P123 = g.P12 * g.P[2];
  const int64_t S1 = g.S[0], S2 = g.S[1], S3 = g.S[2];
  const int64_t P1 = g.P[0], P2 = g.P[1], P3 = g.P[2];
  for (int i = 0; i < 8; ++i) g.off[i] = 0;
  if (dim == 1) {
    g.off[1] = S1;
  } else if (dim == 2) {
    g.off[1] = S1 * S2;
    g.off[2] = g.off[1] + 2 * S1 * P2;
    g.off[3] = g.off[2] + 2 * S2 * P1;
  } else {
    g.off[1] = S1 * S2 * S3;
    g.off[2] = g.off[1] + 2 * S1 * S2 * P3;
    g.off[3] = g.off[2] + 2 * S1 * S3 * P2;
    g.off[4] = g.off[3] + 2 * S2 * S3 * P1;
    g.off[5] = g.off[4] + 4 * S1 * g.P23;
    g.off[6] = g.off[5] + 4 * S2 * g.P13;
    g.off[7] = g.off[6] + 4 * S3 * g.P12;
  }
  return g;
}

// category of index k: c = 0 (S, v = slot 0/1), 1 (R, v = k-1), 2 (H, v = k-M-1)
struct Cat {
  int c;
  int v;
};

__host__ __device__ __forceinline__ Cat cat_of(int k, const MapGeom& g, int dim) {
  const int n = g.n[dim], M = g.M[dim], P = g.P[dim];
  if (k == 0) return {0, 0};
  if (((n & 1) == 0) && k == M) return {0, 1};
  if (k <= P) return {1, k - 1};
  return {2, k - M - 1};
}

__host__ __device__ __forceinline__ Cat cat_mirror(Cat a, int P) {
  if (a.c == 1) return {2, P - 1 - a.v};
  if (a.c == 2) return {1, P - 1 - a.v};
  return a;
}

// Is the class a representative read directly by DFT_to_beta?
//  3D: the last non-self dimension is in R; 2D: the first non-self dimension
//  is in R; 1D: not in H.  (All-self classes are vertices.)
template <int D>
__host__ __device__ __forceinline__ bool is_rep(Cat c1, Cat c2, Cat c3) {
  if (D == 1) return c1.c != 2;
  if (D == 2) {
    if (c1.c != 0) return c1.c == 1;
    return c2.c != 2;
  }
  if (c3.c != 0) return c3.c == 1;
  if (c2.c != 0) return c2.c == 1;
  return c1.c != 2;
}

// beta index of the Re part of a representative class; bs = distance to the
// Im part; vertex = no Im part and no sqrt(2).
template <int D>
__host__ __device__ __forceinline__ int64_t rep_index(Cat c1, Cat c2, Cat c3, const MapGeom& g,
                                             int64_t& bs, bool& vertex) {
  vertex = false;
  if (D == 1) {
    if (c1.c == 0) { vertex = true; bs = 0; return c1.v; }
    bs = g.P[0];
    return g.off[1] + c1.v;
  }
  if (D == 2) {
    if (c1.c == 0 && c2.c == 0) { vertex = true; bs = 0; return g.off[0] + c1.v * g.S[1] + c2.v; }
    if (c1.c == 0) { bs = g.P[1]; return g.off[1] + 2 * (int64_t)c1.v * g.P[1] + c2.v; }
    if (c2.c == 0) { bs = g.P[0]; return g.off[2] + 2 * (int64_t)c2.v * g.P[0] + c1.v; }
    bs = g.P12;
    return g.off[3] + (c2.c == 2 ? 2 * g.P12 : 0) + c1.v + (int64_t)g.P[0] * c2.v;
  }
  const int S2 = g.S[1], S3 = g.S[2];
  const int64_t P1 = g.P[0], P2 = g.P[1], P3 = g.P[2];
  if (c1.c == 0 && c2.c == 0 && c3.c == 0) {
    vertex = true; bs = 0;
    return g.off[0] + (c1.v * S2 + c2.v) * S3 + c3.v;
  }
  if (c1.c == 0 && c2.c == 0) { bs = P3; return g.off[1] + 2 * (int64_t)(c1.v * S2 + c2.v) * P3 + c3.v; }
  if (c1.c == 0 && c3.c == 0) { bs = P2; return g.off[2] + 2 * (int64_t)(c1.v * S3 + c3.v) * P2 + c2.v; }
  if (c2.c == 0 && c3.c == 0) { bs = P1; return g.off[3] + 2 * (int64_t)(c2.v * S3 + c3.v) * P1 + c1.v; }
  if (c1.c == 0) {
    bs = g.P23;
    return g.off[4] + 4 * (int64_t)c1.v * g.P23 + (c2.c == 2 ? 2 * g.P23 : 0) + c2.v + P2 * c3.v;
  }
  if (c2.c == 0) {
    bs = g.P13;
    return g.off[5] + 4 * (int64_t)c2.v * g.P13 + (c1.c == 2 ? 2 * g.P13 : 0) + c1.v + P1 * c3.v;
  }
  if (c3.c == 0) {
    bs = g.P12;
    return g.off[6] + 4 * (int64_t)c3.v * g.P12 + (c1.c == 2 ? 2 * g.P12 : 0) + c1.v + P1 * c2.v;
  }
  bs = g.P123;
  const int blk = (c1.c == 2 ? 1 : 0) + (c2.c == 2 ? 2 : 0);
  return g.off[7] + 2 * (int64_t)blk * g.P123 + c1.v + P1 * (c2.v + P2 * c3.v);
}

// beta -> spectrum element (k1, k2, k3): the per-element formula of
// src/mapping_cpu_kernels.jl:363-738.  Representatives read (b_re + i b_im)/sqrt2,
// other elements are conjugates of their partner, (b_re - i b_im)/sqrt2;
// vertices are real.  Each part is one IEEE division by the double sqrt(2).
template <int D, typename T, typename BT>
__host__ __device__ __forceinline__ cpx<T> beta_to_dft_elem(const BT* __restrict__ beta, int k1, int k2,
                                                  int k3, const MapGeom& g) {
#pragma clang fp contract(off)
  Cat c1 = cat_of(k1, g, 0);
  Cat c2 = D >= 2 ? cat_of(k2, g, 1) : Cat{0, 0};
  Cat c3 = D >= 3 ? cat_of(k3, g, 2) : Cat{0, 0};
  bool neg = false;
  if (!is_rep<D>(c1, c2, c3)) {
    c1 = cat_mirror(c1, g.P[0]);
    c2 = cat_mirror(c2, g.P[1]);
    c3 = cat_mirror(c3, g.P[2]);
    neg = true;
  }
  int64_t bs;
  bool vertex;
  const int64_t re = rep_index<D>(c1, c2, c3, g, bs, vertex);
  const T sq2 = (T)1.4142135623730951;
  if (vertex) return {(T)beta[re], (T)0};
  const T a = (T)beta[re];
  const T b = (T)beta[re + bs];
  return {a / sq2, (neg ? -b : b) / sq2};
}

// Targets of a half-spectrum element in DFT_to_beta: beta indices reading its
// real and imaginary parts.  Returns false if no beta entry reads it.
//   scale_im = +1 (direct read) or -1 (3D mirror blocks read -Im of this element)
template <int D>
__host__ __device__ __forceinline__ bool scatter_targets(int k1, int k2, int k3, const MapGeom& g,
                                                int64_t& re, int64_t& im, bool& vertex,
                                                bool& neg_im) {
  Cat c1 = cat_of(k1, g, 0);
  Cat c2 = D >= 2 ? cat_of(k2, g, 1) : Cat{0, 0};
  Cat c3 = D >= 3 ? cat_of(k3, g, 2) : Cat{0, 0};
  int64_t bs;
  neg_im = false;
  if (is_rep<D>(c1, c2, c3)) {
    re = rep_index<D>(c1, c2, c3, g, bs, vertex);
    im = re + bs;
    return true;
  }
  if (c1.c != 1) return false;  // redundant conjugate inside a self-conjugate plane
  c1 = cat_mirror(c1, g.P[0]);
  c2 = cat_mirror(c2, g.P[1]);
  c3 = cat_mirror(c3, g.P[2]);
  re = rep_index<D>(c1, c2, c3, g, bs, vertex);
  im = re + bs;
  neg_im = true;
  return true;
}

// The same for the interior of dimension 1 (1 <= k1 <= P1, D >= 2), a row
// (k2, k3) at a time: every such element reads / feeds two beta entries, at
//   re + s * k1  and  d further,
// with the imaginary part negated when neg (the mirror blocks, where k1 runs
// backwards).  32-bit arithmetic: beta has at most 2^31 entries.
struct BetaRow {
  uint32_t re, d;
  int s;
  bool neg;
};

template <int D>
__host__ __device__ __forceinline__ BetaRow beta_row(int k2, int k3, const MapGeom& g) {
  const uint32_t P1 = (uint32_t)g.P[0], P2 = (uint32_t)g.P[1];
  const Cat c2 = cat_of(k2, g, 1);
  uint32_t v2 = (uint32_t)c2.v;
  if (D == 2) {
    if (c2.c == 0) return {(uint32_t)g.off[2] + 2u * v2 * P1 - 1u, P1, 1, false};
    return {(uint32_t)g.off[3] + (c2.c == 2 ? 2u * (uint32_t)g.P12 : 0u) + P1 * v2 - 1u,
            (uint32_t)g.P12, 1, false};
  }
  const uint32_t P3 = (uint32_t)g.P[2];
  const Cat c3 = cat_of(k3, g, 2);
  uint32_t v3 = (uint32_t)c3.v;
  const bool neg = c3.c == 2 || (c3.c == 0 && c2.c == 2);
  // the class of the representative (the mirror element's when neg)
  const bool h2 = neg ? c2.c == 1 : c2.c == 2;   // dimension 2 in its second half
  if (neg && c2.c != 0) v2 = P2 - 1u - v2;
  if (neg && c3.c != 0) v3 = P3 - 1u - v3;
  uint32_t base, d;
  if (c2.c == 0 && c3.c == 0) {
    d = P1;
    base = (uint32_t)g.off[3] + 2u * (v2 * (uint32_t)g.S[2] + v3) * P1;
  } else if (c2.c == 0) {
    d = (uint32_t)g.P13;
    base = (uint32_t)g.off[5] + (4u * v2 + (neg ? 2u : 0u)) * d + P1 * v3;
  } else if (c3.c == 0) {
    d = (uint32_t)g.P12;
    base = (uint32_t)g.off[6] + (4u * v3 + (neg ? 2u : 0u)) * d + P1 * v2;
  } else {
    d = (uint32_t)g.P123;
    base = (uint32_t)g.off[7] + 2u * ((neg ? 1u : 0u) + (h2 ? 2u : 0u)) * d + P1 * (v2 + P2 * v3);
  }
  // k1 - 1 forwards, P1 - 1 - (k1 - 1) backwards
  if (neg) return {base + P1, d, -1, true};
  return {base - 1u, d, 1, false};
}

// ---------------------------------------------------------------------------
// Radix-R DFT butterflies on registers, forward: exp(-2 pi i jk/R).  There is
// no inverse form: inverse = swap . forward . swap with swap exchanging real
// and imaginary parts, which the passes fold into their LDS loads and stores.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void dft2(cpx<T>* v) {
  cpx<T> a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}

template <typename T>
__device__ __forceinline__ void dft4(cpx<T>* v) {
  cpx<T> t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
  cpx<T> t2 = cadd(v[1], v[3]), t3 = mul_mi(csub(v[1], v[3]));
  v[0] = cadd(t0, t2);
  v[2] = csub(t0, t2);
  v[1] = cadd(t1, t3);
  v[3] = csub(t1, t3);
}

template <typename T>
__device__ __forceinline__ void dft8(cpx<T>* v) {
  cpx<T> e[4] = {v[0], v[2], v[4], v[6]};
  cpx<T> o[4] = {v[1], v[3], v[5], v[7]};
  dft4(e);
  dft4(o);
  const T h = (T)0.70710678118654752440;
  // w^1 = (h, -h), w^2 = -i, w^3 = (-h, -h)
  cpx<T> w1o = {h * (o[1].x + o[1].y), h * (o[1].y - o[1].x)};
  cpx<T> w2o = mul_mi(o[2]);
  cpx<T> w3o = {h * (-o[3].x + o[3].y), h * (-o[3].y - o[3].x)};
  v[0] = cadd(e[0], o[0]);
  v[4] = csub(e[0], o[0]);
  v[1] = cadd(e[1], w1o);
  v[5] = csub(e[1], w1o);
  v[2] = cadd(e[2], w2o);
  v[6] = csub(e[2], w2o);
  v[3] = cadd(e[3], w3o);
  v[7] = csub(e[3], w3o);
}

template <typename T>
__device__ __forceinline__ void dft16(cpx<T>* v) {
  // 4 x 4: columns of stride 4, twiddle, rows
  cpx<T> a[4][4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
#pragma unroll
    for (int p = 0; p < 4; ++p) a[q][p] = v[q + 4 * p];
    dft4(a[q]);
  }
  // twiddle a[q][p] *= w16^(q*p)
  const T c1 = (T)0.92387953251128675613, s1 = (T)0.38268343236508977173;
  const T h = (T)0.70710678118654752440;
#pragma unroll
  for (int q = 1; q < 4; ++q) {
#pragma unroll
    for (int p = 1; p < 4; ++p) {
      const int m = q * p;  // 1..9
      T c, s;
      switch (m) {
        case 1: c = c1; s = s1; break;
        case 2: c = h; s = h; break;
        case 3: c = s1; s = c1; break;
        case 4: c = 0; s = 1; break;
        case 6: c = -h; s = h; break;
        default: c = -c1; s = -s1; break;  // m == 9: angle 9*pi/8 -> cos=-c1, sin=-s1
      }
      const cpx<T> w = {c, -s};
      a[q][p] = cmul(a[q][p], w);
    }
  }
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    cpx<T> r[4] = {a[0][p], a[1][p], a[2][p], a[3][p]};
    dft4(r);
#pragma unroll
    for (int q = 0; q < 4; ++q) v[p + 4 * q] = r[q];
  }
}

// odd R = 2H+1: X[k] = x0 + sum_j a_j cos(2pi jk/R) - i sum_j b_j sin(2pi jk/R)
// with a_j = x_j + x_{R-j}, b_j = x_j - x_{R-j}
template <typename T, int R>
__device__ __forceinline__ void dft_odd(cpx<T>* v) {
  constexpr int H = (R - 1) / 2;
  cpx<T> a[H], b[H];
#pragma unroll
  for (int j = 1; j <= H; ++j) {
    a[j - 1] = cadd(v[j], v[R - j]);
    b[j - 1] = csub(v[j], v[R - j]);
  }
  const cpx<T> x0 = v[0];
  cpx<T> y0 = x0;
#pragma unroll
  for (int j = 0; j < H; ++j) y0 = cadd(y0, a[j]);
#pragma unroll
  for (int k = 1; k <= H; ++k) {
    T re = x0.x, im = x0.y, sre = 0, sim = 0;
#pragma unroll
    for (int j = 1; j <= H; ++j) {
      const int m = (j * k) % R;
      const T c = (T)OddRadix<R>::c[m];
      const T s = (T)OddRadix<R>::s[m];
      re += a[j - 1].x * c;
      im += a[j - 1].y * c;
      sre += b[j - 1].y * s;
      sim += b[j - 1].x * s;
    }
    v[k] = {re + sre, im - sim};
    v[R - k] = {re - sre, im + sim};
  }
  v[0] = y0;
}

// the same, writing X[k] to dst[k * stride] as it is formed: a_j and b_j
// overwrite the inputs in place and no output array is held
template <typename T, int R>
__device__ __forceinline__ void dft_odd_store(cpx<T>* v, cpx<T>* __restrict__ dst, int stride) {
  constexpr int H = (R - 1) / 2;
  const cpx<T> x0 = v[0];
  cpx<T> y0 = x0;
#pragma unroll
  for (int j = 1; j <= H; ++j) {
    const cpx<T> a = cadd(v[j], v[R - j]);
    const cpx<T> b = csub(v[j], v[R - j]);
    v[j] = a;
    v[R - j] = b;
    y0 = cadd(y0, a);
  }
  dst[0] = y0;
  // one output after another: scheduled across outputs the (H x H) products
  // took hundreds of registers in FP64
#pragma unroll
  for (int k = 1; k <= H; ++k) {
    T re = x0.x, im = x0.y, sre = 0, sim = 0;
#pragma unroll
    for (int j = 1; j <= H; ++j) {
      const T c = (T)OddRadix<R>::c[(j * k) % R], s = (T)OddRadix<R>::s[(j * k) % R];
      re += v[j].x * c;
      im += v[j].y * c;
      sre += v[R - j].y * s;
      sim += v[R - j].x * s;
    }
    dst[k * stride] = {re + sre, im - sim};
    dst[(R - k) * stride] = {re - sre, im + sim};
    if constexpr (R >= 11) __builtin_amdgcn_sched_barrier(0);
  }
}

template <typename T, int R>
__device__ __forceinline__ void dft(cpx<T>* v) {
  if constexpr (R == 2) dft2(v);
  else if constexpr (R == 4) dft4(v);
  else if constexpr (R == 8) dft8(v);
  else if constexpr (R == 16) dft16(v);
  else dft_odd<T, R>(v);
}

// ---------------------------------------------------------------------------
// Stockham autosort FFT of 2^lg lines of length L held in LDS in
// [element][line] order: element e of line l at lds[e * ps + l] (ps >= 2^lg,
// the line stride, padded where the load loops would otherwise conflict).
// Stage s with radix R after Ns = product of earlier radices: butterfly j
// reads elements j + r*L/R, multiplies input r by exp(-2 pi i r k/(Ns*R)),
// k = j mod Ns, and writes elements (j - k)*R + k + r*Ns.  Butterflies are
// numbered b = j * 2^lg + l, so the lines of a tile run on adjacent lanes and
// share twiddles.  A thread takes ceil(E / R) butterflies; the caller
// guarantees that NT threads then cover the (L / R) 2^lg of every stage.
// What bounds a stage: the number of waves a SIMD holds.  With E = 16 (two
// radix-9..15 butterflies and their twiddles per thread) the FP64 passes
// took 248-260 registers, one or two waves per SIMD, and the 1024-thread ones
// spilled 1300 registers; E = 8 with the waves per SIMD asked for by
// pass_waves() keeps three (FP64) or five (FP32).  Twiddles are laid out per stage in the order in
// which adjacent lanes read them: strided reads from one table of the length
// L cost a cache line per lane.
// Measured (before -> after, with tile_grows' tiles): line passes of the FP64
// 256^3 apply 72 -> 65 and 70 -> 57 us (270 MB each, 4.1-4.7 TB/s), its
// dimension-1 pass 140 -> 123 us (107 since radices 29 and 31 are matrix_stage's
// and the pass kernels no longer spill); 509 x 384 FP64 (Bluestein) 19 -> 13 us.
// ---------------------------------------------------------------------------
constexpr int kMaxStages = 15;

struct FftStage {
  int radix;
  int ns;        // product of the radices of earlier stages
  int tw;        // first twiddle of the stage (ns > 1): w^(r k), k < ns, at tw + (r - 1) ns + k
  uint32_t nsm;  // ceil(2^32 / ns), ns >= 2: j / ns = umulhi(j, nsm)
};

// 64 words: a wave holds the whole plan in one register, word l in lane l
// (plan_word), so a stage's parameters cost no memory access.  Read from
// memory stage by stage (the stores in between keep the compiler from scalar
// loads), each stage waited for two dependent L1 / L2 round trips.
struct FftPlan {
  int L;
  int nstages;
  int variant;   // which radix order (the host planner's, names the twiddle table)
  int pad;
  FftStage st[kMaxStages];
};
static_assert(sizeof(FftPlan) == 64 * sizeof(int), "one plan word per lane");

__device__ __forceinline__ int plan_load(const FftPlan* __restrict__ p) {
  return reinterpret_cast<const int*>(p)[threadIdx.x & 63];
}
__device__ __forceinline__ int plan_word(int pl, int w) {
  return __builtin_amdgcn_readlane(pl, w);
}

// a wave-uniform value into a scalar register (the value must be uniform)
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// exact for a, d <= 2^16 (host checks the plan limits)
__device__ __forceinline__ int fdiv(int a, uint32_t m) { return (int)__umulhi((uint32_t)a, m); }

// 15-point DFT by the prime-factor (Good-Thomas) split 15 = 3 x 5, which
// needs no twiddles: with x read at n = (5a + 3b) mod 15 and X written at
// k = (10 k1 + 6 k2) mod 15, X = DFT3 over a of DFT5 over b (W15^(nk) =
// W3^(a k1) W5^(b k2) for these maps).  3 five-point and 5 three-point
// transforms instead of the 15-point pair form's 7 x 7 products.
template <typename T>
__device__ __forceinline__ void dft15_store(cpx<T>* v, cpx<T>* __restrict__ dst, int stride) {
  cpx<T> y[3][5];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
#pragma unroll
    for (int b = 0; b < 5; ++b) y[a][b] = v[(5 * a + 3 * b) % 15];
    dft_odd<T, 5>(y[a]);
  }
#pragma unroll
  for (int k2 = 0; k2 < 5; ++k2) {
    cpx<T> z[3] = {y[0][k2], y[1][k2], y[2][k2]};
    dft_odd<T, 3>(z);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) dst[((10 * k1 + 6 * k2) % 15) * stride] = z[k1];
  }
}

// The matrix cores: 16 x 16 x 4 products, FP32 and FP64.
template <typename T>
using Vec4 = T __attribute__((ext_vector_type(4)));

__device__ __forceinline__ Vec4<float> mfma16x16x4(float a, float b, Vec4<float> c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ Vec4<double> mfma16x16x4(double a, double b, Vec4<double> c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// row of accumulator i in a 16 x 16 tile (column: lane & 15)
template <typename T>
__device__ __forceinline__ int mfma_row(int lane, int i) {
  return sizeof(T) == 4 ? 4 * (lane >> 4) + i : (lane >> 4) + 4 * i;
}
// the value of lane ^ 1
__device__ __forceinline__ float lane_swap(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ double lane_swap(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// A stage of radix 29 or 31 on the matrix cores.  With H = (R - 1) / 2, a_j =
// x_j + x_{R-j} and b_j = x_j - x_{R-j} (x twiddled, a_0 = x_0), the butterfly
//   X_k = sum_j a_j cos(2 pi j k / R) - i sum_j b_j sin(2 pi j k / R)
// is one 16-row tile of cosines times a and one of sines times b, eight
// products for the 16 real columns of eight butterflies; X_{R-k} is the same
// with + i.  A wave takes every (NT / 64)-th column tile and stores it when all
// waves have read theirs.
// What bounds it: per column tile eight products of 32 cycles and as many LDS
// reads.  As a butterfly a thread, its outputs in a loop, the radices kept one
// wave in four busy and spilled 200 registers in FP64 (the pass kernels spill
// up to 13 now): operator product 248^3 FP32 358 -> 272 us, FP64 583 -> 433;
// 217 x 217 FP32 41.5 -> 24.1; 961 FP64 29.4 -> 13.3.  The outputs divided among
// the waves instead: 248^3 FP32 333, FP64 799 (every wave spilled); a and b
// formed in LDS first: 290, 461.
template <typename T, int R, int NT>
__device__ __forceinline__ void matrix_stage(cpx<T>* __restrict__ lds, int L, int Ns, uint32_t nsm,
                                             int lg, int ps, const cpx<T>* __restrict__ tw) {
  constexpr int H = (R - 1) / 2, W = NT / 64;
  static_assert(H < 16, "one tile of output rows");
  // column tiles of a wave: a plan gives a thread at most 16 elements
  constexpr int NV = (2 * 16 * NT / R + 16 * W - 1) / (16 * W);
  const int nb = L / R, nl = 1 << lg, total = nb << lg;
  int tid = (int)threadIdx.x;   // (opaque: as in stockham_stage)
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63, wave = uniform(tid >> 6), n = lane & 15, kk = lane >> 4;
  const bool im = n & 1;   // column pairs hold real and imaginary parts
  const int tiles = (2 * total + 15) >> 4, rs = 2 * ps;
  // input rows j = 4 kt + kk and R - j, and their coefficients in output n
  T cc[4], ss[4];
  int lo[4], hi[4];
#pragma unroll
  for (int kt = 0; kt < 4; ++kt) {
    const int j = 4 * kt + kk;
    cc[kt] = j <= H ? (T)OddRadix<R>::c[(j * n) % R] : (T)0;
    ss[kt] = j <= H ? (T)OddRadix<R>::s[(j * n) % R] : (T)0;
    lo[kt] = j * nb * rs;
    hi[kt] = (j ? R - j : 0) * nb * rs;
  }
  T* x = reinterpret_cast<T*>(lds);
  Vec4<T> c[NV], s[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (wave + v * W >= tiles) continue;
    const int col = min((wave + v * W) * 16 + n, 2 * total - 1), b = col >> 1, jb = b >> lg;
    const T* src = x + jb * rs + 2 * (b & (nl - 1)) + (col & 1);
    const int k = Ns > 1 ? jb - fdiv(jb, nsm) * Ns : 0;
    c[v] = s[v] = Vec4<T>{0, 0, 0, 0};
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      const int j = 4 * kt + kk;
      T y = src[lo[kt]], z = src[hi[kt]];
      if (Ns > 1) {
        cpx<T> w = {(T)1, (T)0}, u = w;
        if (j > 0) {
          w = tw[(j - 1) * Ns + k];
          u = tw[(R - j - 1) * Ns + k];
        }
        const T yo = lane_swap(y), zo = lane_swap(z);
        y = y * w.x + (im ? yo : -yo) * w.y;
        z = z * u.x + (im ? zo : -zo) * u.y;
      }
      // (zeros where the coefficients are zero, so that an infinity stays one)
      const T a = j > H ? (T)0 : j ? y + z : y, d = j > H || j == 0 ? (T)0 : y - z;
      c[v] = mfma16x16x4(cc[kt], a, c[v]);
      s[v] = mfma16x16x4(ss[kt], d, s[v]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (wave + v * W >= tiles) continue;
    const int col = (wave + v * W) * 16 + n, b = col >> 1, j = b >> lg;
    const int k = Ns > 1 ? j - fdiv(j, nsm) * Ns : 0;
    T* dst = x + ((j - k) * R + k) * rs + 2 * (b & (nl - 1)) + (col & 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const T other = lane_swap(s[v][i]);
      const T plus = c[v][i] + other, minus = c[v][i] - other;
      const int r = mfma_row<T>(lane, i);
      if (col < 2 * total && r <= H) {
        dst[r * Ns * rs] = im ? minus : plus;
        if (r > 0) dst[(R - r) * Ns * rs] = im ? plus : minus;
      }
    }
  }
  __syncthreads();
}

template <typename T, int R, int E, int NT>
__device__ __forceinline__ void stockham_stage(cpx<T>* __restrict__ lds, int L, int Ns,
                                               uint32_t nsm, int lg, int ps,
                                               const cpx<T>* __restrict__ tw) {
  constexpr int NQ = (E + R - 1) / R;
  // twiddles loaded before the LDS reads they multiply (the rest, of the large
  // radices, in groups as the registers allow)
  constexpr int CH = sizeof(T) == 4 ? (R <= 17 ? R - 1 : 8) : (R <= 9 ? R - 1 : 6);
  const int nb = L / R;
  const int nl = 1 << lg;
  const int total = nb << lg;
  // an opaque copy of the lane index: keeps the compiler from hoisting every
  // stage's per-lane address arithmetic out of the caller's stage loop (the
  // hoisted values of all radix cases would stay live across the whole FFT)
  int tid = (int)threadIdx.x;
  asm volatile("" : "+v"(tid));
  cpx<T> v[NQ][R];
  int out[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    // idle lanes read nothing: 16-byte reads of one address by many lanes are
    // serialised (3000 cycles a stage when they repeated the last butterfly)
    const int b = tid + q * NT;
    if (b < total) {
      const int j = b >> lg;
      const int line = b & (nl - 1);
      const cpx<T>* src = lds + j * ps + line;
      if (Ns > 1) {
        const int k = j - fdiv(j, nsm) * Ns;
        out[q] = ((j - k) * R + k) * ps + line;
#pragma unroll
        for (int r0 = 1; r0 < R; r0 += CH) {
          cpx<T> w[CH];
#pragma unroll
          for (int r = r0; r < r0 + CH && r < R; ++r) w[r - r0] = tw[(r - 1) * Ns + k];
          if (r0 == 1) {
#pragma unroll
            for (int r = 0; r < R; ++r) v[q][r] = src[r * nb * ps];
          }
#pragma unroll
          for (int r = r0; r < r0 + CH && r < R; ++r) v[q][r] = cmul(v[q][r], w[r - r0]);
        }
      } else {
        out[q] = j * R * ps + line;
#pragma unroll
        for (int r = 0; r < R; ++r) v[q][r] = src[r * nb * ps];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (tid + q * NT < total) {
      cpx<T>* dst = lds + out[q];
      if constexpr (R == 2 || R == 4 || R == 8 || R == 16) {
        dft<T, R>(v[q]);
#pragma unroll
        for (int r = 0; r < R; ++r) dst[r * Ns * ps] = v[q][r];
      } else if constexpr (R == 15) {
        dft15_store<T>(v[q], dst, Ns * ps);
      } else {
        dft_odd_store<T, R>(v[q], dst, Ns * ps);
      }
    }
  }
  __syncthreads();
}

// forward DFT of the tile; pl: the wave's plan register (plan_load)
template <typename T, int E, int NT>
__device__ __forceinline__ void lds_fft(cpx<T>* lds, int pl, int lg, int ps,
                                        const cpx<T>* __restrict__ tw) {
  const int L = plan_word(pl, 0), nst = plan_word(pl, 1);
#pragma unroll 1
  for (int s = 0; s < nst; ++s) {
    const int w = 4 + 4 * s;
    const int ns = plan_word(pl, w + 1);
    const cpx<T>* __restrict__ tws = tw + plan_word(pl, w + 2);
    const uint32_t nsm = (uint32_t)plan_word(pl, w + 3);
    switch (plan_word(pl, w)) {
      case 2: stockham_stage<T, 2, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 3: stockham_stage<T, 3, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 4: stockham_stage<T, 4, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 5: stockham_stage<T, 5, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 7: stockham_stage<T, 7, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 8: stockham_stage<T, 8, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 9: stockham_stage<T, 9, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 11: stockham_stage<T, 11, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 13: stockham_stage<T, 13, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 15: stockham_stage<T, 15, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 16: stockham_stage<T, 16, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 17: stockham_stage<T, 17, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 19: stockham_stage<T, 19, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 23: stockham_stage<T, 23, E, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 29: matrix_stage<T, 29, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      case 31: matrix_stage<T, 31, NT>(lds, L, ns, nsm, lg, ps, tws); break;
      default: break;  // the host planner only emits the radices above
    }
  }
}

// ---------------------------------------------------------------------------
// Spectrum-ordered copy of beta ("u"): one complex slot per half-spectrum
// element e = k1 + H1*(k2 + N2*k3); stored elements hold
// u = sqrt(2) * v (v.x for vertices, whose Im slot is 0), redundant
// conjugates in the self-conjugate dim-1 planes hold 0.  Relative to beta it
// is a permutation with sign flips (the 3D mirror blocks' Im parts), so dot
// products, the diagonal KKT terms and the CG iterates carry over exactly,
// while the FFT passes read and write it along contiguous lines.
// ---------------------------------------------------------------------------
template <int D, typename T>
__host__ __device__ __forceinline__ cpx<T> u_to_v(const cpx<T>* __restrict__ u, int k1, int k2,
                                                  int k3, const MapGeom& g, int H1) {
#pragma clang fp contract(off)
  const T sq2 = (T)1.4142135623730951;
  const Cat c1 = cat_of(k1, g, 0);
  const int64_t e = k1 + (int64_t)H1 * (k2 + (int64_t)g.n[1] * k3);
  if (c1.c == 1) {
    const cpx<T> w = u[e];
    return {w.x / sq2, w.y / sq2};
  }
  const Cat c2 = D >= 2 ? cat_of(k2, g, 1) : Cat{0, 0};
  const Cat c3 = D >= 3 ? cat_of(k3, g, 2) : Cat{0, 0};
  if (is_rep<D>(c1, c2, c3)) {
    const cpx<T> w = u[e];
    if (c2.c == 0 && c3.c == 0) return {w.x, (T)0};
    return {w.x / sq2, w.y / sq2};
  }
  const int m2 = k2 == 0 ? 0 : g.n[1] - k2;
  const int m3 = k3 == 0 ? 0 : g.n[2] - k3;
  const cpx<T> w = u[k1 + (int64_t)H1 * (m2 + (int64_t)g.n[1] * m3)];
  return {w.x / sq2, -(w.y / sq2)};
}

// u_to_v in two steps, without branches around the load: u_src returns the
// slot u_to_v reads and how its value maps (0: w/sqrt2, 1: (w.x, 0),
// 2: conj(w)/sqrt2); u_map applies that map with u_to_v's arithmetic.
template <int D>
__host__ __device__ __forceinline__ int64_t u_src(int k1, int k2, int k3, const MapGeom& g,
                                                  int H1, int& mode) {
  const Cat c1 = cat_of(k1, g, 0);
  const Cat c2 = D >= 2 ? cat_of(k2, g, 1) : Cat{0, 0};
  const Cat c3 = D >= 3 ? cat_of(k3, g, 2) : Cat{0, 0};
  const bool rep = c1.c == 1 || is_rep<D>(c1, c2, c3);
  const bool vert = c1.c != 1 && rep && c2.c == 0 && c3.c == 0;
  const int m2 = (rep || k2 == 0) ? k2 : g.n[1] - k2;
  const int m3 = (rep || k3 == 0) ? k3 : g.n[2] - k3;
  mode = vert ? 1 : (rep ? 0 : 2);
  return k1 + (int64_t)H1 * (m2 + (int64_t)g.n[1] * m3);
}

template <typename T>
__host__ __device__ __forceinline__ cpx<T> u_map(cpx<T> w, int mode) {
#pragma clang fp contract(off)
  const T sq2 = (T)1.4142135623730951;
  const T x = w.x / sq2, y = w.y / sq2;
  if (mode == 1) return {w.x, (T)0};
  return {x, mode == 2 ? -y : y};
}

// u_map on the way into a pass, without its division: w / sqrt2 as w h + w l,
// the first product inside the fma, with h + l the reciprocal of the rounded
// sqrt2.  This is the rounded quotient (none of 1e7 samples differs, but a
// unit in the last place where w l is subnormal), whose rounding the sqrt2 on the way out cancels: h alone put
// M^T M of 1024 samples 5.7e-16 off instead of 4.5e-16.  h is rounded down, so
// that h and l have one sign and an infinity stays one.
template <typename T>
__host__ __device__ __forceinline__ cpx<T> u_scale(cpx<T> w, int mode) {
#pragma clang fp contract(off)
  const T h = sizeof(T) == 8 ? (T)0x1.6a09e667f3bccp-1 : (T)0x1.6a09e6p-1;
  const T l = sizeof(T) == 8 ? (T)0x1.08b2fb1366eaap-56 : (T)2.4203234416068298e-08;
  if (mode == 1) return {w.x, (T)0};
  const T x = fma(w.x, h, w.x * l), y = fma(w.y, h, w.y * l);
  return {x, mode == 2 ? -y : y};
}

// sqrt2 * v, v_to_u of a representative element (kept apart from any
// following add, as in v_to_u)
template <typename T>
__host__ __device__ __forceinline__ cpx<T> scale_sq2(cpx<T> v) {
#pragma clang fp contract(off)
  const T sq2 = (T)1.4142135623730951;
  return {sq2 * v.x, sq2 * v.y};
}

// u slot value of spectrum element (k1,k2,k3) holding v
template <int D, typename T>
__host__ __device__ __forceinline__ cpx<T> v_to_u(cpx<T> v, int k1, int k2, int k3,
                                                  const MapGeom& g) {
#pragma clang fp contract(off)
  const T sq2 = (T)1.4142135623730951;
  const Cat c1 = cat_of(k1, g, 0);
  if (c1.c == 1) return {sq2 * v.x, sq2 * v.y};
  const Cat c2 = D >= 2 ? cat_of(k2, g, 1) : Cat{0, 0};
  const Cat c3 = D >= 3 ? cat_of(k3, g, 2) : Cat{0, 0};
  if (!is_rep<D>(c1, c2, c3)) return {(T)0, (T)0};
  if (c2.c == 0 && c3.c == 0) return {v.x, (T)0};
  return {sq2 * v.x, sq2 * v.y};
}

// ---------------------------------------------------------------------------
// Deterministic block reduction (wave64 shuffles, then LDS across waves).
// The result is valid in thread 0.
// ---------------------------------------------------------------------------
template <typename Op>
__device__ __forceinline__ double block_reduce(double v, Op op) {
  __shared__ double red_smem[16];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = op(v, __shfl_down(v, off, 64));
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red_smem[w] = v;
  __syncthreads();
  double r = v;
  if (threadIdx.x == 0) {
    const int nw = (blockDim.x + 63) >> 6;
    r = red_smem[0];
    for (int i = 1; i < nw; ++i) r = op(r, red_smem[i]);
  }
  return r;
}

struct OpSum {
  __device__ double operator()(double a, double b) const { return a + b; }
};
struct OpMax {
  __device__ double operator()(double a, double b) const { return a > b ? a : b; }
};
struct OpMin {
  __device__ double operator()(double a, double b) const { return a < b ? a : b; }
};

}  // namespace csipm
