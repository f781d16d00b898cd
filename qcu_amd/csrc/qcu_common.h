// qcu_common.h -- shared device types for the MI355X (gfx950) hot path.
//
// Internal field layouts (all site-fastest so that a wavefront of 64 lanes
// reading 64 consecutive sites issues one contiguous 1 KiB (FP64) / 1 KiB
// (FP32 float4) / 1 KiB (FP16 uint4) transaction per load instruction):
//
//   FP64 spinor (one parity)  double2 [12 sc][Vh]
//   FP32 spinor               float4  [6 sc-pairs][Vh]
//   FP16 spinor               uint4   [3 x 8 halves][Vh] + float norm[Vh]
//   FP64 links (compressed)   double2 [2 p][4 mu][6 (rows 0,1)][Vh]
//   FP32 links                float4  [2][4][3][Vh]
//   FP16 links                uint4   [2][4][Vh] (halves 0..7) + uint2 [2][4][Vh]
//   clover inverse (packed)   36 reals per chiral block, 2 blocks per site:
//                             FP64 double2 [2 p][36][Vh], FP32 float4 [2][18][Vh],
//                             FP16 uint4 [2][9][Vh] + float norm[2][Vh]
//
// The half-site index is i = ((t*Lz + z)*Ly + y)*(Lx/2) + x/2 with the full
// x coordinate 2*(x/2) + ((y+z+t+parity)&1), as qcu's kernels decode it
// (src/wilson_dslash.cu:12-30).
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#define QCU_HD __host__ __device__ __forceinline__
#define QCU_D __device__ __forceinline__

namespace qcu {

template <class T>
struct cplx {
  T re, im;
};

template <class T>
QCU_HD cplx<T> mk(T r, T i) {
  cplx<T> c;
  c.re = r;
  c.im = i;
  return c;
}
template <class T>
QCU_HD cplx<T> operator+(cplx<T> a, cplx<T> b) { return mk(a.re + b.re, a.im + b.im); }
template <class T>
QCU_HD cplx<T> operator-(cplx<T> a, cplx<T> b) { return mk(a.re - b.re, a.im - b.im); }
template <class T>
QCU_HD cplx<T> operator*(cplx<T> a, cplx<T> b) {
  return mk(a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re);
}
template <class T>
QCU_HD cplx<T> operator*(T s, cplx<T> a) { return mk(s * a.re, s * a.im); }
template <class T>
QCU_HD cplx<T> conj(cplx<T> a) { return mk(a.re, -a.im); }
// i*a and -i*a
template <class T>
QCU_HD cplx<T> mul_i(cplx<T> a) { return mk(-a.im, a.re); }
template <class T>
QCU_HD cplx<T> mul_mi(cplx<T> a) { return mk(a.im, -a.re); }
// a += b*c ; a += conj(b)*c.  The fused operations are written out, so that every
// kernel rounds these sums alike, whatever is around them.
QCU_HD double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
QCU_HD float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
template <class T>
QCU_HD cplx<T> prod_(cplx<T> b, cplx<T> c) {
#pragma clang fp contract(off)
  return mk(fma_(b.re, c.re, -(b.im * c.im)), fma_(b.re, c.im, b.im * c.re));
}
template <class T>
QCU_HD cplx<T> prodj_(cplx<T> b, cplx<T> c) {
#pragma clang fp contract(off)
  return mk(fma_(b.re, c.re, b.im * c.im), fma_(b.re, c.im, -(b.im * c.re)));
}
template <class T>
QCU_HD void cmad(cplx<T> &a, cplx<T> b, cplx<T> c) {
  a = a + prod_(b, c);
}
template <class T>
QCU_HD void cmadj(cplx<T> &a, cplx<T> b, cplx<T> c) {
  a = a + prodj_(b, c);
}
// cmad / cmadj, or with CHAIN the products as chained FMAs: 2 instructions per
// component instead of 3, with two roundings of the running sum instead of one of it
// and two of the product.  For the FP16 fields, whose hop is near its vector rate
// (24^3x48 with 12 right-hand sides 356 against 310 us) and whose halves the FMAs
// take unconverted; its error is that of the stored halves either way (clover hop at
// 16^3x32 against FP64: 3.4366e-4 unchained, 3.4365e-4).  The FP32 hop is slower with
// it (380 against 395 us: longer dependent chains).
template <bool CHAIN, class T>
QCU_HD void cmad_(cplx<T> &a, cplx<T> b, cplx<T> c) {
  if (CHAIN) {
    a.re = fma_(-b.im, c.im, fma_(b.re, c.re, a.re));
    a.im = fma_(b.im, c.re, fma_(b.re, c.im, a.im));
  } else {
    cmad(a, b, c);
  }
}
template <bool CHAIN, class T>
QCU_HD void cmadj_(cplx<T> &a, cplx<T> b, cplx<T> c) {
  if (CHAIN) {
    a.re = fma_(b.im, c.im, fma_(b.re, c.re, a.re));
    a.im = fma_(-b.im, c.re, fma_(b.re, c.im, a.im));
  } else {
    cmadj(a, b, c);
  }
}
// x - k d, in one rounding per component
template <class T>
QCU_HD cplx<T> nmad(cplx<T> x, T k, cplx<T> d) {
  return mk(fma_(-k, d.re, x.re), fma_(-k, d.im, x.im));
}
template <class T>
QCU_HD T norm2(cplx<T> a) { return a.re * a.re + a.im * a.im; }

// ---------------------------------------------------------------------------
// geometry
// ---------------------------------------------------------------------------
struct Geom {
  int lxh, ly, lz, lt;  // half x extent and full y, z, t
  int vh;               // half volume
  int tbc;              // +1 periodic, -1 antiperiodic time boundary
};

struct Site {
  int xh, y, z, t, xodd;  // xodd: full x coordinate is odd
};

QCU_HD Site decode(const Geom &g, int i, int parity) {
  Site s;
  int r = i / g.lxh;
  s.xh = i - r * g.lxh;
  int r2 = r / g.ly;
  s.y = r - r2 * g.ly;
  s.t = r2 / g.lz;
  s.z = r2 - s.t * g.lz;
  s.xodd = (s.y + s.z + s.t + parity) & 1;
  return s;
}

// Site number k of the order in which the hop kernels visit the sites: with
// zslab = 0 the storage order, else slabs of zslab z planes one after the other,
// t by t within a slab (the last slab may be thinner).  i: the half-site index.
// Past the last site (lanes that fill up a wave) there is no slab to divide by: k
// there stands for the last site.
QCU_HD Site ordered_site(const Geom &g, int zslab, int k, int parity, int &i) {
  k = k < g.vh ? k : g.vh - 1;
  if (zslab == 0) {
    i = k;
    return decode(g, k, parity);
  }
  const int plane = g.lxh * g.ly;
  const int full = zslab * plane * g.lt;
  const int slab = k / full;
  const int left = g.lz - slab * zslab;
  const int row = (left < zslab ? left : zslab) * plane;  // sites of one t in this slab
  int r = k - slab * full;
  Site s;
  s.t = r / row;
  r -= s.t * row;
  const int zi = r / plane;
  r -= zi * plane;
  s.z = slab * zslab + zi;
  s.y = r / g.lxh;
  s.xh = r - s.y * g.lxh;
  s.xodd = (s.y + s.z + s.t + parity) & 1;
  i = (s.t * g.lz + s.z) * plane + r;
  return s;
}

// Loads and stores address a wavefront-uniform base (component k of a field,
// kept in scalar registers) plus a 32-bit per-lane byte offset, so that the
// compiler can use the scalar-base / 32-bit-offset form of global memory
// instructions instead of a 64-bit address per load and per component.
// NT: non-temporal, for data a kernel reads once, or writes for a later kernel to read
// (the network's activations and term fields): they need not displace the lines that
// the kernel reads again.  The global address space is stated: the compiler cannot
// know it of a base that was itself read from memory (a segment's links and clover
// blocks), and would use flat loads, which return out of order and make every wait a
// full one.
#define QCU_GLOBAL __attribute__((address_space(1)))
template <class V, bool NT = false>
QCU_D V ld_at(const void *base, size_t comp_bytes, unsigned lane_off) {
  typedef unsigned words __attribute__((ext_vector_type(sizeof(V) / 4)));
  const QCU_GLOBAL words *p = (const QCU_GLOBAL words *)((const QCU_GLOBAL char *)base + comp_bytes + lane_off);
  const words w = NT ? __builtin_nontemporal_load(p) : *p;
  V v;
  __builtin_memcpy(&v, &w, sizeof(V));
  return v;
}
template <class V, bool NT = false>
QCU_D void st_at(void *base, size_t comp_bytes, unsigned lane_off, const V &v) {
  typedef unsigned words __attribute__((ext_vector_type(sizeof(V) / 4)));
  words w;
  __builtin_memcpy(&w, &v, sizeof(V));
  QCU_GLOBAL words *p = (QCU_GLOBAL words *)((QCU_GLOBAL char *)base + comp_bytes + lane_off);
  if (NT) __builtin_nontemporal_store(w, p);
  else *p = w;
}

// ---------------------------------------------------------------------------
// precision tags
// ---------------------------------------------------------------------------
enum Prec { P64 = 0, P32 = 1, P16 = 2 };

template <int P>
struct real_of {
  typedef float type;
};
template <>
struct real_of<P64> {
  typedef double type;
};

// Spinor field of one parity (or a slice of a batch) in internal storage.
struct SpinorPtr {
  void *p;      // payload
  float *norm;  // FP16 only
  int stride;   // sites between consecutive components (>= vh)
};

template <int P>
struct SpinorIO;

template <>
struct SpinorIO<P64> {
  typedef double real;
  template <bool NT = false>
  static QCU_D void load(const SpinorPtr &f, int i, cplx<double> (&v)[12]) {
    const unsigned off = (unsigned)i * 16u;
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      double2 a = ld_at<double2, NT>(f.p, (size_t)k * f.stride * 16, off);
      v[k] = mk(a.x, a.y);
    }
  }
  template <bool NT = false>
  static QCU_D void store(const SpinorPtr &f, int i, const cplx<double> (&v)[12]) {
    const unsigned off = (unsigned)i * 16u;
#pragma unroll
    for (int k = 0; k < 12; ++k) st_at<double2, NT>(f.p, (size_t)k * f.stride * 16, off, make_double2(v[k].re, v[k].im));
  }
};

template <>
struct SpinorIO<P32> {
  typedef float real;
  template <bool NT = false>
  static QCU_D void load(const SpinorPtr &f, int i, cplx<float> (&v)[12]) {
    const unsigned off = (unsigned)i * 16u;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      float4 a = ld_at<float4, NT>(f.p, (size_t)k * f.stride * 16, off);
      v[2 * k] = mk(a.x, a.y);
      v[2 * k + 1] = mk(a.z, a.w);
    }
  }
  template <bool NT = false>
  static QCU_D void store(const SpinorPtr &f, int i, const cplx<float> (&v)[12]) {
    const unsigned off = (unsigned)i * 16u;
#pragma unroll
    for (int k = 0; k < 6; ++k)
      st_at<float4, NT>(f.p, (size_t)k * f.stride * 16, off,
                    make_float4(v[2 * k].re, v[2 * k].im, v[2 * k + 1].re, v[2 * k + 1].im));
  }
};

QCU_D float h2f(unsigned short h) { return __half2float(__ushort_as_half(h)); }
QCU_D unsigned short f2h(float f) { return __half_as_ushort(__float2half_rn(f)); }

template <>
struct SpinorIO<P16> {
  typedef float real;
  // the stored halves and their scale: an FMA takes a half operand as it is
  // (v_fma_mix_f32), so kernels that go on with products need not convert it
  static QCU_D float load_raw(const SpinorPtr &f, int i, _Float16 (&h)[24]) {
    const unsigned off = (unsigned)i * 16u;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const uint4 a = ld_at<uint4>(f.p, (size_t)k * f.stride * 16, off);
      __builtin_memcpy(&h[8 * k], &a, 16);
    }
    return ld_at<float>(f.norm, 0, (unsigned)i * 4u);
  }
  // v as load() gives it back after store()
  static QCU_D void round(cplx<float> (&v)[12]) {
    float m = 0.f;
#pragma unroll
    for (int k = 0; k < 12; ++k) m = fmaxf(m, fmaxf(fabsf(v[k].re), fabsf(v[k].im)));
    const float inv = m > 0.f ? 1.0f / m : 0.f;
#pragma unroll
    for (int k = 0; k < 12; ++k) v[k] = mk(m * h2f(f2h(v[k].re * inv)), m * h2f(f2h(v[k].im * inv)));
  }
  template <bool NT = false>
  static QCU_D void load(const SpinorPtr &f, int i, cplx<float> (&v)[12]) {
    const unsigned off = (unsigned)i * 16u;
    const float nrm = ld_at<float, NT>(f.norm, 0, (unsigned)i * 4u);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      uint4 a = ld_at<uint4, NT>(f.p, (size_t)k * f.stride * 16, off);
      unsigned w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[4 * k + q] = mk(nrm * h2f((unsigned short)(w[q] & 0xffffu)),
                          nrm * h2f((unsigned short)(w[q] >> 16)));
      }
    }
  }
  static QCU_D void store(const SpinorPtr &f, int i, const cplx<float> (&v)[12]) {
    float m = 0.f;
#pragma unroll
    for (int k = 0; k < 12; ++k) m = fmaxf(m, fmaxf(fabsf(v[k].re), fabsf(v[k].im)));
    float inv = m > 0.f ? 1.0f / m : 0.f;
    const unsigned off = (unsigned)i * 16u;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      unsigned w[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        w[q] = (unsigned)f2h(v[4 * k + q].re * inv) | ((unsigned)f2h(v[4 * k + q].im * inv) << 16);
      st_at<uint4>(f.p, (size_t)k * f.stride * 16, off, make_uint4(w[0], w[1], w[2], w[3]));
    }
    st_at<float>(f.norm, 0, (unsigned)i * 4u, m);
  }
};

// ---------------------------------------------------------------------------
// links: 6 complex (rows 0 and 1), row 2 reconstructed as conj(row0 x row1),
// the same 12-real compression qcu applies on every load (include/define.h:198-206)
// ---------------------------------------------------------------------------
struct LinkPtr {
  void *a;  // FP64 double2 / FP32 float4 / FP16 uint4 part
  void *b;  // FP16 uint2 part
  int vh;
};

template <class T>
QCU_D void recon_row2(cplx<T> (&u)[9]) {
  u[6] = conj(u[1] * u[5] - u[2] * u[4]);
  u[7] = conj(u[2] * u[3] - u[0] * u[5]);
  u[8] = conj(u[0] * u[4] - u[1] * u[3]);
}
// the same with chained FMAs
QCU_D cplx<float> cross_chain(cplx<float> a, cplx<float> b, cplx<float> c, cplx<float> d) {  // conj(a b - c d)
  const float re = fma_(c.im, d.im, fma_(-c.re, d.re, fma_(-a.im, b.im, a.re * b.re)));
  const float im = fma_(c.im, d.re, fma_(c.re, d.im, fma_(-a.im, b.re, -(a.re * b.im))));
  return mk(re, im);
}
QCU_D void recon_row2_chain(cplx<float> (&u)[9]) {
  u[6] = cross_chain(u[1], u[5], u[2], u[4]);
  u[7] = cross_chain(u[2], u[3], u[0], u[5]);
  u[8] = cross_chain(u[0], u[4], u[1], u[3]);
}

// load(L, pm, i, u): (p, mu) slab index pm = p*4 + mu
template <int P>
struct LinkIO;

template <>
struct LinkIO<P64> {
  // rows 0 and 1 only
  template <bool NT = false>
  static QCU_D void rows(const LinkPtr &L, int pm, int i, cplx<double> (&u)[9]) {
    const unsigned off = (unsigned)i * 16u;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      double2 a = ld_at<double2, NT>(L.a, ((size_t)pm * 6 + k) * L.vh * 16, off);
      u[k] = mk(a.x, a.y);
    }
  }
  template <bool NT = false>
  static QCU_D void load(const LinkPtr &L, int pm, int i, cplx<double> (&u)[9]) {
    rows<NT>(L, pm, i, u);
    recon_row2(u);
  }
};

template <>
struct LinkIO<P32> {
  template <bool NT = false>
  static QCU_D void rows(const LinkPtr &L, int pm, int i, cplx<float> (&u)[9]) {
    const unsigned off = (unsigned)i * 16u;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      float4 a = ld_at<float4, NT>(L.a, ((size_t)pm * 3 + k) * L.vh * 16, off);
      u[2 * k] = mk(a.x, a.y);
      u[2 * k + 1] = mk(a.z, a.w);
    }
  }
  template <bool NT = false>
  static QCU_D void load(const LinkPtr &L, int pm, int i, cplx<float> (&u)[9]) {
    rows<NT>(L, pm, i, u);
    recon_row2(u);
  }
};

template <>
struct LinkIO<P16> {
  template <bool NT = false>
  static QCU_D void load(const LinkPtr &L, int pm, int i, cplx<float> (&u)[9]) {
    uint4 a = ld_at<uint4, NT>(L.a, (size_t)pm * L.vh * 16, (unsigned)i * 16u);
    uint2 b = ld_at<uint2, NT>(L.b, (size_t)pm * L.vh * 8, (unsigned)i * 8u);
    unsigned w[6] = {a.x, a.y, a.z, a.w, b.x, b.y};
#pragma unroll
    for (int k = 0; k < 6; ++k)
      u[k] = mk(h2f((unsigned short)(w[k] & 0xffffu)), h2f((unsigned short)(w[k] >> 16)));
    recon_row2_chain(u);
  }
};

// ---------------------------------------------------------------------------
// packed clover inverse: per chiral block 6 real diagonal entries followed by
// the 15 complex entries of the strict lower triangle, row-major
// ((1,0),(2,0),(2,1),(3,0),...,(5,4)); 36 reals per block, 72 per site.
// ---------------------------------------------------------------------------
struct CloverPtr {
  void *p;
  float *norm;  // FP16 only
  int vh;
};

template <int P>
struct CloverIO;

template <>
struct CloverIO<P64> {
  template <bool NT = false>
  static QCU_D void load(const CloverPtr &C, int i, double (&c)[72]) {
    const unsigned off = (unsigned)i * 16u;
#pragma unroll
    for (int k = 0; k < 36; ++k) {
      double2 a = ld_at<double2, NT>(C.p, (size_t)k * C.vh * 16, off);
      c[2 * k] = a.x;
      c[2 * k + 1] = a.y;
    }
  }
};
template <>
struct CloverIO<P32> {
  template <bool NT = false>
  static QCU_D void load(const CloverPtr &C, int i, float (&c)[72]) {
    const unsigned off = (unsigned)i * 16u;
#pragma unroll
    for (int k = 0; k < 18; ++k) {
      float4 a = ld_at<float4, NT>(C.p, (size_t)k * C.vh * 16, off);
      c[4 * k] = a.x;
      c[4 * k + 1] = a.y;
      c[4 * k + 2] = a.z;
      c[4 * k + 3] = a.w;
    }
  }
};
template <>
struct CloverIO<P16> {
  // the stored halves and their scale, which the caller applies to the product
  template <bool NT = false>
  static QCU_D float load(const CloverPtr &C, int i, float (&c)[72]) {
    const unsigned off = (unsigned)i * 16u;
    _Float16 h[72];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const uint4 a = ld_at<uint4, NT>(C.p, (size_t)k * C.vh * 16, off);
      __builtin_memcpy(&h[8 * k], &a, 16);
    }
#pragma unroll
    for (int k = 0; k < 72; ++k) c[k] = (float)h[k];
    return ld_at<float>(C.norm, 0, (unsigned)i * 4u);
  }
};

// s a, never fused into what follows
template <class T>
QCU_HD cplx<T> scale_(T s, cplx<T> a) {
#pragma clang fp contract(off)
  return mk(s * a.re, s * a.im);
}

// Row of a clover block times a spinor, begun: the diagonal's product and the first
// off-diagonal one p (unless CHAIN, where that follows as chained FMAs) rounded once.
// A rounding of its own for the diagonal, the largest term, shows: clover hop in FP64
// 2.35e-16 off instead of 2.30e-16, full operator 1.40e-16 instead of 1.33e-16, FP32
// hop 1.094e-7 instead of 1.064e-7.
template <class T>
QCU_HD cplx<T> diag_plus(T d, cplx<T> x, cplx<T> p) {
  return mk(fma_(d, x.re, p.re), fma_(d, x.im, p.im));
}

// out_b = C_b * v_b for chiral block b (spins {2b, 2b+1}) from its 36 packed reals
template <bool CHAIN = false, class T>
QCU_HD void clover_apply_block(const T *cb, cplx<T> (&v)[12], int b) {
  cplx<T> o[6];
  const cplx<T> *x = v + 6 * b;
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    cplx<T> acc = scale_(cb[r], x[r]);
    const int first = CHAIN ? 6 : (r == 0 ? 1 : 0);
#pragma unroll
    for (int col = 0; col < 6; ++col) {
      if (col < r) {
        const int k = 6 + 2 * (r * (r - 1) / 2 + col);
        const cplx<T> c = mk(cb[k], cb[k + 1]);
        if (col == first)
          acc = diag_plus(cb[r], x[r], prod_(c, x[col]));
        else
          cmad_<CHAIN>(acc, c, x[col]);
      } else if (col > r) {
        const int k = 6 + 2 * (col * (col - 1) / 2 + r);
        const cplx<T> c = mk(cb[k], cb[k + 1]);
        if (col == first)
          acc = diag_plus(cb[r], x[r], prodj_(c, x[col]));
        else
          cmadj_<CHAIN>(acc, c, x[col]);
      }
    }
    o[r] = acc;
  }
#pragma unroll
  for (int r = 0; r < 6; ++r) v[6 * b + r] = o[r];
}

// out = C * v for one site (both chiral blocks)
template <bool CHAIN, class T>
QCU_HD void clover_apply_site(const T (&c)[72], cplx<T> (&v)[12]) {
  clover_apply_block<CHAIN>(c, v, 0);
  clover_apply_block<CHAIN>(c + 36, v, 1);
}

// load one chiral block (36 reals) of a packed FP64 / FP32 clover field
template <bool NT = false>
QCU_D void clover_load_block(const CloverPtr &C, int i, int b, double (&c)[36]) {
  const unsigned off = (unsigned)i * 16u;
#pragma unroll
  for (int k = 0; k < 18; ++k) {
    double2 a = ld_at<double2, NT>(C.p, (size_t)(18 * b + k) * C.vh * 16, off);
    c[2 * k] = a.x;
    c[2 * k + 1] = a.y;
  }
}
template <bool NT = false>
QCU_D void clover_load_block(const CloverPtr &C, int i, int b, float (&c)[36]) {
  const unsigned off = (unsigned)i * 16u;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    float4 a = ld_at<float4, NT>(C.p, (size_t)(9 * b + k) * C.vh * 16, off);
    c[4 * k] = a.x;
    c[4 * k + 1] = a.y;
    c[4 * k + 2] = a.z;
    c[4 * k + 3] = a.w;
  }
}

// XCD-aware block remap: hardware places workgroup b on XCD b % 8; give each
// XCD a contiguous range of logical blocks so neighbouring t-slices share L2.
QCU_D int remap_block(int b, int n, int on) {
  if (!on) return b;
  int q = n >> 3, r = n & 7;
  int k = b & 7, j = b >> 3;
  return k * q + (k < r ? k : r) + j;
}

}  // namespace qcu
