// clover.hip -- clover term A = 1 - coeff/8 sum_{mu<nu} T_munu (Q_munu - Q_munu^dag)
// per site of one parity, and its inverse, stored as two packed Hermitian 6x6
// chiral blocks (spins {0,1} and {2,3}).
//
// Leaves and sign table follow src/clover_dslash.cu:5-837 (T_munu = -i sigma_munu
// in the DeGrand-Rossi basis; the reference hard-codes coeff = kappa*csw = 1 at
// :826-835).  The reference inverts the full 12x12 matrix by Gauss-Jordan
// without pivoting (src/clover_dslash.cu:839-855); A is block diagonal, so the
// two 6x6 blocks are inverted here, with partial pivoting, in FP64, once per
// gauge field instead of on every call.
#include "qcu_internal.h"

namespace qcu {

typedef cplx<double> cd;

// s += x y and s += conj(x) y as four chained FMAs (x y - z w + s is contracted
// to a product, an FMA and an addition instead)
QCU_D void fma3(cd &s, const cd &x, const cd &y) {
  s.re = fma(x.re, y.re, s.re);
  s.im = fma(x.re, y.im, s.im);
  s.re = fma(-x.im, y.im, s.re);
  s.im = fma(x.im, y.re, s.im);
}

// c = a b, a b^dag, a^dag b
template <int ADJ_A, int ADJ_B>
QCU_D void mul3(const cd (&a)[9], const cd (&b)[9], cd (&c)[9]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      cd s = mk(0.0, 0.0);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const cd x = ADJ_A ? conj(a[k * 3 + i]) : a[i * 3 + k];
        const cd y = ADJ_B ? conj(b[j * 3 + k]) : b[k * 3 + j];
        fma3(s, x, y);
      }
      c[i * 3 + j] = s;
    }
}

struct Pt {
  int x, y, z, t;
};

// p + d in direction mu (wavefront-uniform), periodic; d = +1 or -1.  Without
// branches: the whole field computation is then one basic block, and the
// scheduling fences in leaves() hold.
QCU_D int wrap(int v, int n) {
  v = v < 0 ? n - 1 : v;
  return v == n ? 0 : v;
}
QCU_D Pt step(const Geom &g, Pt p, int mu, int d) {
  p.x = wrap(p.x + d * (int)(mu == 0), 2 * g.lxh);
  p.y = wrap(p.y + d * (int)(mu == 1), g.ly);
  p.z = wrap(p.z + d * (int)(mu == 2), g.lz);
  p.t = wrap(p.t + d * (int)(mu == 3), g.lt);
  return p;
}

QCU_D void link_at(const LinkPtr &U, const Geom &g, int mu, const Pt &p, cd (&u)[9]) {
  const int par = (p.x + p.y + p.z + p.t) & 1;
  const int i = ((p.t * g.lz + p.z) * g.ly + p.y) * g.lxh + (p.x >> 1);
  const double2 *src = (const double2 *)U.a + (size_t)(par * 4 + mu) * 6 * U.vh + i;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const double2 a = src[(size_t)k * U.vh];
    u[k] = mk(a.x, a.y);
  }
  recon_row2(u);
}

// A point of the schedule: m is formed before it and nothing moves across.
// (The scheduling fence alone holds back loads, but products whose results are
// needed later would still be formed later, with their operands kept.)
QCU_D void done_here(cd (&m)[9]) {
#pragma unroll
  for (int k = 0; k < 9; ++k) asm volatile("" : "+v"(m[k].re), "+v"(m[k].im));
  __builtin_amdgcn_sched_barrier(0);
}

// Q_munu - Q_munu^dag at p, Q the four leaves of the (mu, nu) plane, each
// counter-clockwise.  The second leaf of each pair is taken as its adjoint
// (Q - Q^dag only changes its sign with that), so that the pair shares a factor:
//   leaf 1 - leaf 4^dag = U_mu(x) [ U_nu(x+mu) U_mu(x+nu)^dag U_nu(x)^dag
//                                  - U_nu(x+mu-nu)^dag U_mu(x-nu)^dag U_nu(x-nu) ]
//   leaf 2 - leaf 3^dag = [ U_nu(x) U_mu(x-mu+nu)^dag U_nu(x-mu)^dag
//                           - U_nu(x-nu)^dag U_mu(x-mu-nu)^dag U_nu(x-mu-nu) ] U_mu(x-mu)
// 10 matrix products instead of 12.
QCU_D void leaves(const LinkPtr &U, const Geom &g, Pt p, int mu, int nu, cd (&Q)[9]) {
  const Pt pm = step(g, p, mu, 1), pn = step(g, p, nu, 1);
  const Pt mm = step(g, p, mu, -1), mn = step(g, p, nu, -1);
  // one bracket's matrices at a time, instead of every link loaded first
  cd a[9], b[9], c[9], s[9];
  link_at(U, g, nu, pm, a);
  link_at(U, g, mu, pn, b);
  mul3<0, 1>(a, b, c);
  done_here(c);
  link_at(U, g, nu, p, a);
  mul3<0, 1>(c, a, s);
  done_here(s);
  link_at(U, g, nu, step(g, pm, nu, -1), a);
  link_at(U, g, mu, mn, b);
  // U_nu(x+mu-nu)^dag U_mu(x-nu)^dag = (U_mu(x-nu) U_nu(x+mu-nu))^dag
  mul3<0, 0>(b, a, c);
  done_here(c);
  link_at(U, g, nu, mn, a);
  mul3<1, 0>(c, a, b);
#pragma unroll
  for (int k = 0; k < 9; ++k) s[k] = s[k] - b[k];
  done_here(s);
  link_at(U, g, mu, p, a);
  mul3<0, 0>(a, s, Q);
  done_here(Q);
  // the second pair; two of its links were read before and are read again
  // (from the vector cache) rather than kept in registers meanwhile
  asm volatile("" : "+v"(p.t));
  link_at(U, g, mu, step(g, mm, nu, 1), a);
  link_at(U, g, nu, mm, b);
  mul3<0, 0>(b, a, c);  // U_nu(x-mu) U_mu(x-mu+nu)
  done_here(c);
  link_at(U, g, nu, p, a);
  mul3<0, 1>(a, c, s);
  done_here(s);
  const Pt mmn = step(g, mm, nu, -1);
  link_at(U, g, mu, mmn, a);
  link_at(U, g, nu, step(g, p, nu, -1), b);
  mul3<0, 0>(a, b, c);  // U_mu(x-mu-nu) U_nu(x-nu)
  done_here(c);
  link_at(U, g, nu, mmn, a);
  mul3<1, 0>(c, a, b);
#pragma unroll
  for (int k = 0; k < 9; ++k) s[k] = s[k] - b[k];
  done_here(s);
  link_at(U, g, mu, mm, a);
  mul3<0, 0>(s, a, c);
#pragma unroll
  for (int k = 0; k < 9; ++k) Q[k] = Q[k] + c[k];
}

// in-place Gauss-Jordan with partial pivoting on a 6x6 complex block; every
// index is static (the pivot row is brought up by conditional swaps), so the
// block stays in registers.  Returns 1 if a pivot vanishes or is not a number.
// The products, small against the entries near 1 that they change, are formed
// first and added with one rounding.
QCU_D void swap_if(bool c, cd &a, cd &b) {
  const cd t = a;
  a = mk(c ? b.re : a.re, c ? b.im : a.im);
  b = mk(c ? t.re : b.re, c ? t.im : b.im);
}

QCU_D int invert6(cd (&m)[36]) {
  int bad = 0;
  int piv[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    piv[k] = k;
    double best = norm2(m[k * 7]);
#pragma unroll
    for (int r = k + 1; r < 6; ++r) {
      const double v = norm2(m[r * 6 + k]);
      const bool c = v > best;
      best = c ? v : best;
      piv[k] = c ? r : piv[k];
    }
    if (!(best > 0)) bad = 1;
#pragma unroll
    for (int r = k + 1; r < 6; ++r)
#pragma unroll
      for (int j = 0; j < 6; ++j) swap_if(piv[k] == r, m[k * 6 + j], m[r * 6 + j]);
    const cd pv = m[k * 7];
    const double den = norm2(pv);
    const cd ip = mk(pv.re / den, -pv.im / den);
    m[k * 7] = mk(1.0, 0.0);
#pragma unroll
    for (int j = 0; j < 6; ++j) m[k * 6 + j] = m[k * 6 + j] * ip;
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      if (r == k) continue;
      const cd f = mk(-m[r * 6 + k].re, -m[r * 6 + k].im);
      m[r * 6 + k] = mk(0.0, 0.0);
#pragma unroll
      for (int j = 0; j < 6; ++j) m[r * 6 + j] = m[r * 6 + j] + f * m[k * 6 + j];
    }
  }
  // the row exchanges of A are column exchanges of its inverse, undone last first
#pragma unroll
  for (int k = 5; k >= 0; --k)
#pragma unroll
    for (int r = k + 1; r < 6; ++r)
#pragma unroll
      for (int j = 0; j < 6; ++j) swap_if(piv[k] == r, m[j * 6 + k], m[j * 6 + r]);
  return bad;
}

// 6 diagonal reals, then the strict lower triangle row by row
QCU_D void pack6(const cd (&m)[36], double (&buf)[36]) {
#pragma unroll
  for (int r = 0; r < 6; ++r) buf[r] = m[r * 7].re;
#pragma unroll
  for (int r = 1; r < 6; ++r)
#pragma unroll
    for (int c = 0; c < r; ++c) {
      const int k = 6 + 2 * (r * (r - 1) / 2 + c);
      buf[k] = m[r * 6 + c].re;
      buf[k + 1] = m[r * 6 + c].im;
    }
}

QCU_D void store6(void *dst, int vh, int i, int b, const double (&buf)[36]) {
#pragma unroll
  for (int q = 0; q < 18; ++q)
    st_at<double2>(dst, (size_t)(18 * b + q) * vh * 16, (unsigned)i * 16u, make_double2(buf[2 * q], buf[2 * q + 1]));
}

struct CloverKArgs {
  LinkPtr U;
  Geom g;
  double coeff;
  CloverOut out[2];  // per parity
  int *bad;  // host memory: set to 1 by a plain store
};

// The term is built in two launches, each over both parities (neighbouring
// blocks alternate parity, so that both find each other's links in the XCD's L2).
//
// k_clover_field: one thread per (site, plane) forms H = -i (Q - Q^dag), a
// Hermitian 3x3 of 9 reals, and leaves it in the memory of the packed A.
// k_clover: one thread per (site, chiral block) assembles its 6x6 block, inverts
// it and writes it in every precision the lattice keeps.
//
// Both keep their matrices in registers (every index static).  At 24^3x48 with
// all precisions: 0.41 ms (about 40 % of the FP64 vector rate; 166 registers, 3
// waves per SIMD) and 0.28 ms (its reads and 1588 bytes of stores per site, 4.7
// TB/s).  One thread per site for everything needed 7 matrices and both blocks
// with run-time indices, that is scratch memory: 6.7 ms and 0.2 ms of
// conversions.  One launch that hands H over through LDS holds the larger
// kernel's registers throughout, so 6 waves per CU: 1.18 ms.
constexpr int kCloverSites = 64;

__global__ void __launch_bounds__(384) k_clover_field(CloverKArgs a) {
  const Geom &g = a.g;
  const int blk = remap_block(blockIdx.x, gridDim.x, 1);
  const int parity = blk & 1;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // the plane
  const int i = (blk >> 1) * kCloverSites + (threadIdx.x & 63);
  if (i >= g.vh) return;
  const int mu = w < 3 ? 0 : (w < 5 ? 1 : 2);
  const int nu = w < 3 ? w + 1 : (w < 5 ? w - 1 : 3);
  const Site s = decode(g, i, parity);
  const Pt p = {2 * s.xh + s.xodd, s.y, s.z, s.t};
  cd Q[9];
  leaves(a.U, g, p, mu, nu, Q);
  // diagonal 2 Im Q_rr, below it -i (Q_rc - conj(Q_cr)); in 5 of the 36 16-byte
  // words that A takes at the same site, so that A may replace it site by site
  double h[10];
  h[9] = 0;
#pragma unroll
  for (int r = 0; r < 3; ++r) h[r] = 2 * Q[4 * r].im;
#pragma unroll
  for (int r = 1; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < r; ++c) {
      const int k = 3 + 2 * (r + c - 1);
      h[k] = Q[r * 3 + c].im + Q[c * 3 + r].im;
      h[k + 1] = Q[c * 3 + r].re - Q[r * 3 + c].re;
    }
#pragma unroll
  for (int k = 0; k < 5; ++k)
    st_at<double2>(a.out[parity].clov, (size_t)(5 * w + k) * g.vh * 16, (unsigned)i * 16u,
                   make_double2(h[2 * k], h[2 * k + 1]));
}

// With H_k of planes XY, XZ, XT, YZ, YT, ZT and s = +1 for block 0, -1 for block 1:
//   block = 1 - coeff/8 [[D, E^dag], [E, -D]],  D = H_0 - s H_5,
//   E = i H_1 + H_3 - s H_2 + s i H_4
// (the sign table of src/clover_dslash.cu:161-172, :288-300, :416-428, :548-560,
// :680-692, :812-824).  Waves 0 and 1 of a block take blocks 0 and 1 of 64 sites.
__global__ void __launch_bounds__(2 * kCloverSites) k_clover(CloverKArgs a) {
  __shared__ double shmax[2][kCloverSites];
  const Geom &g = a.g;
  const int blk = remap_block(blockIdx.x, gridDim.x, 1);
  const int parity = blk & 1;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = (blk >> 1) * kCloverSites + lane;
  const bool in = i < g.vh;
  const CloverOut &o = a.out[parity];
  cd m[36];
  if (in) {
    const double sc = -0.125 * a.coeff;
    const double s = w == 0 ? 1.0 : -1.0;
    double h[6][10];
#pragma unroll
    for (int k = 0; k < 30; ++k) {
      const double2 v = ld_at<double2>(o.clov, (size_t)k * g.vh * 16, (unsigned)i * 16u);
      h[k / 5][2 * (k % 5)] = v.x;
      h[k / 5][2 * (k % 5) + 1] = v.y;
    }
    auto H = [&](int pl, int r, int c) {  // an entry on or below the diagonal
      if (r == c) return mk(h[pl][r], 0.0);
      const int k = 3 + 2 * (r + c - 1);
      return mk(h[pl][k], h[pl][k + 1]);
    };
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c <= r; ++c) {
        const cd d = sc * (H(0, r, c) - s * H(5, r, c));
        const double one = r == c ? 1.0 : 0.0;
        m[r * 6 + c] = mk(one + d.re, d.im);
        m[(r + 3) * 6 + c + 3] = mk(one - d.re, -d.im);
        // E = F + i G with Hermitian F and G, so both triangles from one read
        const cd f = sc * (H(3, r, c) - s * H(2, r, c)), e = sc * (H(1, r, c) + s * H(4, r, c));
        m[(r + 3) * 6 + c] = mk(f.re - e.im, f.im + e.re);
        if (r != c) {
          m[c * 6 + r] = conj(m[r * 6 + c]);
          m[(c + 3) * 6 + r + 3] = conj(m[(r + 3) * 6 + c + 3]);
          m[(c + 3) * 6 + r] = mk(f.re + e.im, e.re - f.im);
        }
      }
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) m[c * 6 + r + 3] = conj(m[(r + 3) * 6 + c]);
  }
  __syncthreads();  // both waves have read H, which A now replaces
  double buf[36];
  double mx = 0;
  if (in) {
    pack6(m, buf);
    store6(o.clov, g.vh, i, w, buf);
    if (invert6(m)) *(volatile int *)a.bad = 1;
    pack6(m, buf);
    store6(o.cinv64, g.vh, i, w, buf);
    if (o.cinv32) {
#pragma unroll
      for (int k = 0; k < 9; ++k)
        st_at<float4>(o.cinv32, (size_t)(9 * w + k) * g.vh * 16, (unsigned)i * 16u,
                      make_float4((float)buf[4 * k], (float)buf[4 * k + 1], (float)buf[4 * k + 2],
                                  (float)buf[4 * k + 3]));
    }
#pragma unroll
    for (int k = 0; k < 36; ++k) mx = fmax(mx, fabs(buf[k]));
    shmax[w][lane] = mx;
  }
  if (!o.cinv16) return;  // uniform: the same for both waves
  __syncthreads();
  if (in) {
    // one FP16 scale per site, shared by its two blocks
    mx = fmax(mx, shmax[1 - w][lane]);
    const double inv = mx > 0 ? 1.0 / mx : 0.0;
    unsigned h[18];
#pragma unroll
    for (int k = 0; k < 18; ++k)
      h[k] = (unsigned)f2h((float)(buf[2 * k] * inv)) | ((unsigned)f2h((float)(buf[2 * k + 1] * inv)) << 16);
    // 16-byte words 0..3 and the first half of word 4 hold block 0, the rest block 1
    const unsigned off = (unsigned)i * 16u;
    st_at<uint2>((char *)o.cinv16 + 8 * w, (size_t)4 * g.vh * 16, off,
                 w == 0 ? make_uint2(h[16], h[17]) : make_uint2(h[0], h[1]));
#pragma unroll
    for (int k = 0; k < 4; ++k)
      st_at<uint4>(o.cinv16, (size_t)(5 * w + k) * g.vh * 16, off,
                   w == 0 ? make_uint4(h[4 * k], h[4 * k + 1], h[4 * k + 2], h[4 * k + 3])
                          : make_uint4(h[4 * k + 2], h[4 * k + 3], h[4 * k + 4], h[4 * k + 5]));
    if (w == 0) o.cinv16n[i] = (float)mx;
  }
}

int clover_build(const LinkPtr &U64, const Geom &g, double coeff, const CloverOut (&out)[2], int *bad,
                 hipStream_t s) {
  CloverKArgs a;
  a.U = U64;
  a.g = g;
  a.coeff = coeff;
  a.out[0] = out[0];
  a.out[1] = out[1];
  a.bad = bad;
  const int nb = 2 * ((g.vh + kCloverSites - 1) / kCloverSites);
  hipLaunchKernelGGL(k_clover_field, dim3(nb), dim3(6 * kCloverSites), 0, s, a);
  hipLaunchKernelGGL(k_clover, dim3(nb), dim3(2 * kCloverSites), 0, s, a);
  QCU_HIP(hipGetLastError());
  return 0;
}

}  // namespace qcu
