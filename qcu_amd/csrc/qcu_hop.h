// qcu_hop.h -- device code shared by the hop kernels: spin projection and
// reconstruction, colour transport, neighbour indices, and the pieces of the
// kernels that give each of the eight directions a wave of its own.
#pragma once
#include "qcu_batch.h"
#include "qcu_common.h"
#include "qcu_reduce.h"

namespace qcu {

// spin projection of psi(neighbour) for direction MU, FWD = 1: (1 - g_mu), 0: (1 + g_mu)
template <int MU, int FWD, class T>
QCU_D void project(const cplx<T> (&s)[12], cplx<T> (&h0)[3], cplx<T> (&h1)[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const cplx<T> s0 = s[c], s1 = s[3 + c], s2 = s[6 + c], s3 = s[9 + c];
    if (MU == 0) {
      h0[c] = FWD ? s0 + mul_mi(s3) : s0 + mul_i(s3);
      h1[c] = FWD ? s1 + mul_mi(s2) : s1 + mul_i(s2);
    } else if (MU == 1) {
      h0[c] = FWD ? s0 + s3 : s0 - s3;
      h1[c] = FWD ? s1 - s2 : s1 + s2;
    } else if (MU == 2) {
      h0[c] = FWD ? s0 + mul_mi(s2) : s0 + mul_i(s2);
      h1[c] = FWD ? s1 + mul_i(s3) : s1 + mul_mi(s3);
    } else {
      h0[c] = FWD ? s0 - s2 : s0 + s2;
      h1[c] = FWD ? s1 - s3 : s1 + s3;
    }
  }
}

// the same from the stored halves of an FP16 spinor, scaled by its norm: a
// component is norm s_a +- norm s_b in two mixed FMAs, without conversions
template <int MU, int FWD>
QCU_D void project_raw(const _Float16 (&s)[24], float nrm, cplx<float> (&h0)[3], cplx<float> (&h1)[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    // base spin a, partner b, factor: +-1 (f = 0) or +-i (f = 1)
    auto comb = [&](int a, int b, int f, int sgn) {
      const int ka = 2 * (3 * a + c), kb = 2 * (3 * b + c);
      const float re = nrm * (float)s[ka], im = nrm * (float)s[ka + 1];
      const float n = sgn > 0 ? nrm : -nrm;
      if (f == 0) return mk(fma_(n, (float)s[kb], re), fma_(n, (float)s[kb + 1], im));
      return mk(fma_(-n, (float)s[kb + 1], re), fma_(n, (float)s[kb], im));
    };
    const int w = FWD ? -1 : 1;  // sign of the gamma term
    if (MU == 0) {
      h0[c] = comb(0, 3, 1, w);
      h1[c] = comb(1, 2, 1, w);
    } else if (MU == 1) {
      h0[c] = comb(0, 3, 0, -w);
      h1[c] = comb(1, 2, 0, w);
    } else if (MU == 2) {
      h0[c] = comb(0, 2, 1, w);
      h1[c] = comb(1, 3, 1, -w);
    } else {
      h0[c] = comb(0, 2, 0, w);
      h1[c] = comb(1, 3, 0, w);
    }
  }
}

// add the reconstructed 4-spinor of the transported half spinor (a0, a1)
template <int MU, int FWD, class T>
QCU_D void accumulate(cplx<T> (&d)[12], const cplx<T> (&a0)[3], const cplx<T> (&a1)[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    d[c] = d[c] + a0[c];
    d[3 + c] = d[3 + c] + a1[c];
    if (MU == 0) {
      d[6 + c] = FWD ? d[6 + c] + mul_i(a1[c]) : d[6 + c] + mul_mi(a1[c]);
      d[9 + c] = FWD ? d[9 + c] + mul_i(a0[c]) : d[9 + c] + mul_mi(a0[c]);
    } else if (MU == 1) {
      d[6 + c] = FWD ? d[6 + c] - a1[c] : d[6 + c] + a1[c];
      d[9 + c] = FWD ? d[9 + c] + a0[c] : d[9 + c] - a0[c];
    } else if (MU == 2) {
      d[6 + c] = FWD ? d[6 + c] + mul_i(a0[c]) : d[6 + c] + mul_mi(a0[c]);
      d[9 + c] = FWD ? d[9 + c] + mul_mi(a1[c]) : d[9 + c] + mul_i(a1[c]);
    } else {
      d[6 + c] = FWD ? d[6 + c] - a0[c] : d[6 + c] + a0[c];
      d[9 + c] = FWD ? d[9 + c] - a1[c] : d[9 + c] + a1[c];
    }
  }
}

// a = U h (FWD) or U^dag h
template <int FWD, bool CHAIN, class T>
QCU_D void transport(const cplx<T> (&u)[9], const cplx<T> (&h)[3], cplx<T> (&a)[3]) {
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    cplx<T> acc = mk<T>(0, 0);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if (FWD)
        cmad_<CHAIN>(acc, u[r * 3 + c], h[c]);
      else
        cmadj_<CHAIN>(acc, u[c * 3 + r], h[c]);
    }
    a[r] = acc;
  }
}

// Where the spinors of a hop live.  Reading the caller's fields directly (192
// contiguous bytes per lane, whose lines the twelve loads of a direction share)
// costs the hop 3 % more than the internal layout; staging them through it cost
// two more passes (70 + 100 us beside a 430 us clover hop at 32^3x64) and, as the
// staging was allocated per call, 10 ms of hipMalloc and hipFree.
enum HopIO {
  IO_INT = 0,  // internal layout (batch vectors)
  IO_EXT = 1,  // the caller's FP64 fields [Vh][4][3], one lattice and one right-hand side
};

template <int P, int IO>
QCU_D void load_spinor(const SpinorPtr &f, int i, cplx<typename real_of<P>::type> (&v)[12]) {
  if (IO == IO_EXT) {
    const double2 *src = (const double2 *)f.p + (size_t)i * 12;
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      const double2 a = src[k];
      v[k] = mk<typename real_of<P>::type>(a.x, a.y);
    }
  } else {
    SpinorIO<P>::load(f, i, v);
  }
}

template <int P, int IO>
QCU_D void store_spinor(const SpinorPtr &f, int i, const cplx<typename real_of<P>::type> (&v)[12]) {
  if (IO == IO_EXT) {
    double2 *dst = (double2 *)f.p + (size_t)i * 12;
#pragma unroll
    for (int k = 0; k < 12; ++k) dst[k] = make_double2(v[k].re, v[k].im);
  } else {
    SpinorIO<P>::store(f, i, v);
  }
}

// the transported half spinor (a0, a1) of one direction
template <int P, int IO, int MU, int FWD, bool NT = false>
QCU_D void hop_half(cplx<typename real_of<P>::type> (&a0)[3], cplx<typename real_of<P>::type> (&a1)[3],
                    const LinkPtr &U, int pm, int li, const SpinorPtr &in, int si, typename real_of<P>::type ph) {
  typedef typename real_of<P>::type T;
  cplx<T> h0[3], h1[3];
  if constexpr (P == P16) {
    _Float16 s[24];
    const float nrm = SpinorIO<P16>::load_raw(in, si, s);
    project_raw<MU, FWD>(s, nrm, h0, h1);
  } else {
    cplx<T> s[12];
    load_spinor<P, IO>(in, si, s);
    project<MU, FWD>(s, h0, h1);
  }
  cplx<T> u[9];
  LinkIO<P>::template load<NT>(U, pm, li, u);
  transport<FWD, P == P16>(u, h0, a0);
  transport<FWD, P == P16>(u, h1, a1);
  if (MU == 3) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      a0[c] = ph * a0[c];
      a1[c] = ph * a1[c];
    }
  }
}

template <int P, int IO, int MU, int FWD, bool NT>
QCU_D void hop_dir(cplx<typename real_of<P>::type> (&d)[12], const LinkPtr &U, int pm, int li,
                   const SpinorPtr &in, int si, typename real_of<P>::type ph) {
  cplx<typename real_of<P>::type> a0[3], a1[3];
  hop_half<P, IO, MU, FWD, NT>(a0, a1, U, pm, li, in, si, ph);
  accumulate<MU, FWD>(d, a0, a1);
}

// index of the neighbour of site i (half index) in direction MU, forward or
// backward, and the sign of a hop across the time boundary.  Branch-free; a
// site with odd full x has its x-1 neighbour at the same half index.
template <int MU, int FWD>
QCU_D int neighbour(const Geom &g, const Site &s, int i, int &sign) {
  const int sy = g.lxh, sz = g.lxh * g.ly, st = sz * g.lz;
  sign = 1;
  if (MU == 0) {
    if (FWD) return i + s.xodd - s.xodd * (int)(s.xh == g.lxh - 1) * g.lxh;
    const int xe = 1 - s.xodd;
    return i - xe + xe * (int)(s.xh == 0) * g.lxh;
  }
  if (MU == 1) return FWD ? i + sy - (int)(s.y == g.ly - 1) * g.ly * sy : i - sy + (int)(s.y == 0) * g.ly * sy;
  if (MU == 2) return FWD ? i + sz - (int)(s.z == g.lz - 1) * g.lz * sz : i - sz + (int)(s.z == 0) * g.lz * sz;
  const int edge = FWD ? (int)(s.t == g.lt - 1) : (int)(s.t == 0);
  sign = 1 - 2 * ((int)(g.tbc < 0) & edge);
  return FWD ? i + st - edge * g.lt * st : i - st + edge * g.lt * st;
}

// ---- eight waves per 64 sites (k_hop_split in dslash.hip, iterate.hip) ------
constexpr int kSplitSites = 64;

// components 2w, 2w + 1 of a spinor
template <int P, int IO>
QCU_D void load_pair(const SpinorPtr &f, int i, int w, cplx<typename real_of<P>::type> (&v)[2]) {
  typedef typename real_of<P>::type T;
  if (P == P64) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int k = 2 * w + q;
      const double2 a = IO == IO_EXT ? ((const double2 *)f.p)[(size_t)i * 12 + k]
                                     : ld_at<double2>(f.p, (size_t)k * f.stride * 16, (unsigned)i * 16u);
      v[q] = mk<T>((T)a.x, (T)a.y);
    }
  } else if (P == P32) {
    const float4 a = ld_at<float4>(f.p, (size_t)w * f.stride * 16, (unsigned)i * 16u);
    v[0] = mk<T>(a.x, a.y);
    v[1] = mk<T>(a.z, a.w);
  } else {
    const float nrm = ld_at<float>(f.norm, 0, (unsigned)i * 4u);
    const uint2 a = ld_at<uint2>((char *)f.p + 8 * (w & 1), (size_t)(w >> 1) * f.stride * 16, (unsigned)i * 16u);
    v[0] = mk<T>(nrm * h2f((unsigned short)(a.x & 0xffffu)), nrm * h2f((unsigned short)(a.x >> 16)));
    v[1] = mk<T>(nrm * h2f((unsigned short)(a.y & 0xffffu)), nrm * h2f((unsigned short)(a.y >> 16)));
  }
}

// m: the largest component of the whole spinor (FP16 only)
template <int P, int IO>
QCU_D void store_pair(const SpinorPtr &f, int i, int w, const cplx<typename real_of<P>::type> (&v)[2], float m) {
  if (P == P64) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int k = 2 * w + q;
      const double2 a = make_double2(v[q].re, v[q].im);
      if (IO == IO_EXT)
        ((double2 *)f.p)[(size_t)i * 12 + k] = a;
      else
        st_at<double2>(f.p, (size_t)k * f.stride * 16, (unsigned)i * 16u, a);
    }
  } else if (P == P32) {
    st_at<float4>(f.p, (size_t)w * f.stride * 16, (unsigned)i * 16u,
                  make_float4(v[0].re, v[0].im, v[1].re, v[1].im));
  } else {
    const float inv = m > 0.f ? 1.0f / m : 0.f;
    unsigned h[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) h[q] = (unsigned)f2h(v[q].re * inv) | ((unsigned)f2h(v[q].im * inv) << 16);
    st_at<uint2>((char *)f.p + 8 * (w & 1), (size_t)(w >> 1) * f.stride * 16, (unsigned)i * 16u,
                 make_uint2(h[0], h[1]));
    if (w == 0) st_at<float>(f.norm, 0, (unsigned)i * 4u, m);
  }
}

// reals 2q, 2q + 1 of chiral block b of a packed clover field, as stored
template <int P>
struct CloverWord;
template <>
struct CloverWord<P64> {
  typedef double2 raw;
  static QCU_D raw load(const CloverPtr &C, unsigned off, int n) {
    return ld_at<double2>(C.p, (size_t)n * C.vh * 16, off);
  }
  static QCU_D cplx<double> value(raw a) { return mk(a.x, a.y); }
};
template <>
struct CloverWord<P32> {
  typedef float2 raw;
  static QCU_D raw load(const CloverPtr &C, unsigned off, int n) {
    return ld_at<float2>((char *)C.p + 8 * (n & 1), (size_t)(n >> 1) * C.vh * 16, off);
  }
  static QCU_D cplx<float> value(raw a) { return mk(a.x, a.y); }
};
template <>
struct CloverWord<P16> {
  typedef unsigned raw;
  static QCU_D raw load(const CloverPtr &C, unsigned off, int n) {
    return ld_at<unsigned>((char *)C.p + 4 * (n & 3), (size_t)(n >> 2) * C.vh * 16, off);
  }
  static QCU_D cplx<float> value(raw a) {
    return mk(h2f((unsigned short)(a & 0xffffu)), h2f((unsigned short)(a >> 16)));
  }
};

// rows 2j, 2j + 1 of a chiral block: the word of both diagonals and the 9
// off-diagonal entries (their common one once), loaded ahead of their use
template <int P>
struct CloverRows {
  typedef typename real_of<P>::type T;
  typename CloverWord<P>::raw dg, e[2][5];
  float nrm;

  // entry of column c in row 2j + q: its word
  static QCU_D int word(int b, int j, int q, int k) {
    const int r = 2 * j + q;
    const int c = k < r ? k : k + 1;  // k counts the 5 columns other than r
    const int hi = c < r ? r : c, lo = c < r ? c : r;
    return 18 * b + 3 + hi * (hi - 1) / 2 + lo;
  }
  QCU_D void load(const CloverPtr &C, int i, int b, int j) {
    const unsigned off = (unsigned)i * 16u;
    nrm = P == P16 ? ld_at<float>(C.norm, 0, (unsigned)i * 4u) : 1.f;
    dg = CloverWord<P>::load(C, off, 18 * b + j);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int k = 0; k < 5; ++k) e[q][k] = CloverWord<P>::load(C, off, word(b, j, q, k));
  }
  // row 2j + q times the block's six components x (in LDS, one lane per site),
  // in the order of clover_apply_block
  QCU_D cplx<T> row(int j, int q, const cplx<T> (*x)[kSplitSites], int lane) const {
    const int r = 2 * j + q;
    const cplx<T> d = CloverWord<P>::value(dg);
    const T diag = q ? d.im : d.re;
    const cplx<T> v = x[r][lane];
    cplx<T> acc = scale_(diag, v);
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const cplx<T> c = CloverWord<P>::value(e[q][k]);
      if (k == 0 && P != P16) {
        const bool low = q == 1 || j > 0;  // column 0; row 0 begins with the adjoint of column 1
        acc = diag_plus(diag, v, prod_(mk(c.re, low ? c.im : -c.im), x[low ? 0 : 1][lane]));
      } else if (k < r)
        cmad_<P == P16>(acc, c, x[k][lane]);
      else
        cmadj_<P == P16>(acc, c, x[k + 1][lane]);
    }
    return P == P16 ? scale_((T)nrm, acc) : acc;
  }
};

// component k of the sum over the eight directions' half spinors
template <class T>
QCU_D cplx<T> hop_sum(const cplx<T> (*half)[6][kSplitSites], int k, int lane) {
  cplx<T> acc = mk<T>(0, 0);
  if (k < 6) {
#pragma unroll
    for (int d = 0; d < 8; ++d) acc = acc + half[d][k][lane];
    return acc;
  }
  // the lower spins take the upper ones' colour c with the factors of accumulate()
  const bool s3 = k >= 9;
  const int c = s3 ? k - 9 : k - 6;
  const int k01 = (s3 ? 0 : 3) + c, k23 = (s3 ? 3 : 0) + c;
  acc = acc + mul_mi(half[0][k01][lane]);
  acc = acc + mul_i(half[1][k01][lane]);
  const cplx<T> b1 = half[2][k01][lane], f1 = half[3][k01][lane];
  acc = s3 ? acc - b1 : acc + b1;
  acc = s3 ? acc + f1 : acc - f1;
  const cplx<T> b2 = half[4][k23][lane], f2 = half[5][k23][lane];
  acc = s3 ? acc + mul_i(b2) : acc + mul_mi(b2);
  acc = s3 ? acc + mul_mi(f2) : acc + mul_i(f2);
  acc = acc + half[6][k23][lane];
  acc = acc - half[7][k23][lane];
  return acc;
}

// Partials of 64 sites whose per-lane sums sit in sh[k][w][lane], w < 6 the waves
// that formed them: added in wave order, then over the sites of each system.
// Called by every wave; wave k writes value k.
template <int NR>
QCU_D void split_partials(double (*sh)[6][kSplitSites], double *partials, int blk, int t0, int nrhs, int pcap, int w,
                          int lane) {
  __syncthreads();
  if (w >= NR) return;
  double sum = 0;
#pragma unroll
  for (int j = 0; j < 6; ++j) sum += sh[w][j][lane];
  if (nrhs == 1) {
    sum = wave_sum(sum);
    if (lane == 0) partials[(size_t)blk * NR + w] = sum;
  } else {
    sh[w][0][lane] = sum;  // this wave's own slots
    __builtin_amdgcn_wave_barrier();
    if (lane < nrhs) {
      const int j0 = ((lane - t0 % nrhs) % nrhs + nrhs) % nrhs;
      double acc = 0;
      for (int j = j0; j < kSplitSites; j += nrhs) acc += sh[w][0][j];
      partials[((size_t)lane * pcap + blk) * NR + w] = acc;
    }
  }
}

}  // namespace qcu
