// iterate.hip -- BiCGSTAB iterations of small batches (FP64 and FP32, no
// preconditioner) in five launches instead of ten.
//
// On a lattice of a few thousand sites every kernel lasts as long as its launch,
// its first loads and its chain of dependent steps (4 to 5 us), whatever it
// computes, so an iteration costs what its launches cost (8^4 FP64: 10 launches,
// 47 us; these five 32 us).  Here
//   * the finishing kernels are gone: every block of the kernel that needs a
//     scalar sums the block partials itself (all blocks in the same order, so all
//     get the same value) while its first vector loads are in flight;
//   * p = r + beta (p - omega v) and s = r - alpha v are formed where the hop loads
//     them, eight times per site instead of once, and each block also stores them
//     for its own odd sites.
//   1  p, hop to the even sites      [rho, beta]
//   2  v = Mhat p, <r~, v>
//   3  s, hop to the even sites      [alpha]
//   4  t = Mhat s, <t, s>, |t|^2
//   5  x, r, <r~, r>, |r|^2          [omega]
// A kernel reads the states of one buffer and one of its blocks per segment writes
// the updated ones to the other, as it writes p to the other of two vectors, so
// that no block reads what another one replaces.
#include "qcu_hop.h"
#include "qcu_internal.h"
#include "qcu_state.h"

namespace qcu {

struct ItArgs {
  SpinorPtr out;               // hop output (even sites)
  SpinorPtr r, v, p, own;      // own: where the block's p or s goes
  SpinorPtr x, rt, s, t;       // kernel 5
  const SegDesc *segs;
  int nseg;
  const SysState *in;
  SysState *st;
  const double *part;          // partials to finish
  double *part_out;
  int kind;                    // FK_ALPHA, FK_OMEGA, FK_RHO; FK_NONE: take the states as they are
};

// the states of this block's systems after epilogue `kind` on the totals of their
// block partials, in LDS; the first block of the segment writes them out
template <int NR>
QCU_D void finish_local(SysState *ls, const ItArgs &a, const SegPart &sd, int blk, int t0, int w, int lane,
                        int nwaves) {
  const int blk0 = blk - t0 / kSplitSites, nb = (sd.nthr + kSplitSites - 1) / kSplitSites;
  for (int r = w; r < sd.nrhs; r += nwaves) {
    const SysState *in = a.in + sd.sys0 + r;
    const bool run = a.kind != FK_NONE && in->done == 0;
    // the partials load beside the state (those of a stopped system are not used)
    const double *part = a.part + ((size_t)r * sd.pcap + blk0) * NR;
    double tot[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) tot[k] = 0;
    if (a.kind != FK_NONE) {
      for (int b = lane; b < nb; b += 64)
#pragma unroll
        for (int k = 0; k < NR; ++k) tot[k] += part[(size_t)b * NR + k];
#pragma unroll
      for (int k = 0; k < NR; ++k) tot[k] = wave_sum(tot[k]);
    }
    // the state goes through LDS, a word per lane
    constexpr int kWords = sizeof(SysState) / 8;
    char *l = (char *)(ls + r);
    if (lane < kWords) __builtin_memcpy(l + 8 * lane, (const char *)in + 8 * lane, 8);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane == 0 && run) {
      if (NR == 2) fin_alpha(ls + r, tot[0], tot[1]);
      if (NR == 3 && a.kind == FK_OMEGA) fin_omega(ls + r, tot[0], tot[1], tot[NR - 1]);
      if (NR == 3 && a.kind == FK_RHO) fin_rho(ls + r, tot[0], tot[1], tot[NR - 1]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (t0 == 0 && lane < kWords) __builtin_memcpy((char *)(a.st + sd.sys0 + r) + 8 * lane, l + 8 * lane, 8);
  }
  __syncthreads();
}

template <class T>
QCU_D cplx<T> sc(const double (&c)[2]) {
  return mk<T>((T)c[0], (T)c[1]);
}

// kernels 1 (KIND 0: p) and 3 (KIND 1: s)
template <int P, int CLOVER, int KIND>
__global__ void __launch_bounds__(8 * kSplitSites) k_it_even(ItArgs a) {
  typedef typename real_of<P>::type T;
  __shared__ cplx<T> half[8][6][kSplitSites];
  __shared__ SysState ls[kMaxRhs];
  const int blk = blockIdx.x;
  const BlockSeg bs = find_seg(a.segs, a.nseg, blk, kSplitSites);
  if (bs.seg < 0) return;  // uniform
  const SegPart sd = seg_part<P>(a.segs, bs.seg, 0);
  const Geom g = sd.g;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = bs.t0 + lane;
  const int k = n / sd.nrhs, rhs = n - k * sd.nrhs;
  const bool valid = n < sd.nthr;
  int i;
  const Site s = ordered_site(g, sd.zslab, k, 0, i);
  const int t = i * sd.nrhs + rhs;
  const SpinorPtr rv = seg_view(a.r, P, sd.voff, sd.nthr), vv = seg_view(a.v, P, sd.voff, sd.nthr),
                  pv = seg_view(a.p, P, sd.voff, sd.nthr);
  // this wave's neighbour and link, loaded before the scalars are known
  int j = 0, sg = 1, pm = 0, li = 0;
#define QCU_IT_DIR(MU)                      \
  case 2 * MU:                              \
    j = neighbour<MU, 0>(g, s, i, sg);      \
    pm = 4 + MU;                            \
    li = j;                                 \
    break;                                  \
  case 2 * MU + 1:                          \
    j = neighbour<MU, 1>(g, s, i, sg);      \
    pm = MU;                                \
    li = i;                                 \
    break;
  switch (w) {
    QCU_IT_DIR(0)
    QCU_IT_DIR(1)
    QCU_IT_DIR(2)
    QCU_IT_DIR(3)
  }
#undef QCU_IT_DIR
  cplx<T> rr[12], v[12], pp[12], u[9], ro[2], vo[2], po[2];
  const bool mine = valid && w < 6;  // this wave's pair of components of the result
  if (valid) {
    const int sj = j * sd.nrhs + rhs;
    SpinorIO<P>::load(rv, sj, rr);
    SpinorIO<P>::load(vv, sj, v);
    if (KIND == 0) SpinorIO<P>::load(pv, sj, pp);
    LinkIO<P>::rows(sd.U, pm, li, u);
  }
  finish_local<KIND == 0 ? 3 : 2>(ls, a, sd, blk, bs.t0, w, lane, 8);
  const bool active = valid && ls[rhs].done == 0;
  const cplx<T> c0 = sc<T>(KIND == 0 ? ls[rhs].beta : ls[rhs].alpha), c1 = sc<T>(ls[rhs].omega);
  auto comb = [&](cplx<T> r, cplx<T> v, cplx<T> p) { return KIND == 0 ? r + c0 * (p - c1 * v) : r - c0 * v; };
  const int cb = w / 3, cj = w - 3 * cb;
  CloverRows<P> cr;
  if (active) {
#pragma unroll
    for (int q = 0; q < 12; ++q) rr[q] = comb(rr[q], v[q], pp[q]);
    recon_row2(u);
    cplx<T> h0[3], h1[3], a0[3], a1[3];
#define QCU_IT_DIR(D, MU, FWD)       \
  case D:                            \
    project<MU, FWD>(rr, h0, h1);    \
    transport<FWD, false>(u, h0, a0); \
    transport<FWD, false>(u, h1, a1); \
    break;
    switch (w) {
      QCU_IT_DIR(0, 0, 0)
      QCU_IT_DIR(1, 0, 1)
      QCU_IT_DIR(2, 1, 0)
      QCU_IT_DIR(3, 1, 1)
      QCU_IT_DIR(4, 2, 0)
      QCU_IT_DIR(5, 2, 1)
      QCU_IT_DIR(6, 3, 0)
      QCU_IT_DIR(7, 3, 1)
    }
#undef QCU_IT_DIR
    const T ph = (T)sg;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      half[w][c][lane] = ph * a0[c];
      half[w][3 + c][lane] = ph * a1[c];
    }
    if (CLOVER && w < 6) cr.load(sd.Cinv, i, cb, cj);
  }
  if (mine) {  // in flight over the barrier
    load_pair<P, IO_INT>(rv, t, w, ro);
    load_pair<P, IO_INT>(vv, t, w, vo);
    if (KIND == 0) load_pair<P, IO_INT>(pv, t, w, po);
  }
  __syncthreads();
  const bool store = active && w < 6;
  cplx<T> d[2];
  if (store) {
#pragma unroll
    for (int q = 0; q < 2; ++q) d[q] = hop_sum(half, 2 * w + q, lane);
  }
  if (CLOVER) {
    cplx<T>(*b)[kSplitSites] = half[0];
    __syncthreads();
    if (store) {
#pragma unroll
      for (int q = 0; q < 2; ++q) b[2 * w + q][lane] = d[q];
    }
    __syncthreads();
    if (store) {
#pragma unroll
      for (int q = 0; q < 2; ++q) d[q] = cr.row(cj, q, b + 6 * cb, lane);
    }
  }
  if (store) store_pair<P, IO_INT>(seg_view(a.out, P, sd.voff, sd.nthr), t, w, d, 0.f);
  if (mine) {
    const SpinorPtr own = seg_view(a.own, P, sd.voff, sd.nthr);
    if (active) {
#pragma unroll
      for (int q = 0; q < 2; ++q) ro[q] = comb(ro[q], vo[q], po[q]);
      store_pair<P, IO_INT>(own, t, w, ro, 0.f);
    } else if (KIND == 0) {
      store_pair<P, IO_INT>(own, t, w, po, 0.f);  // a stopped system's p moves along unchanged
    }
  }
}

// kernel 5: x += alpha p + omega s, r = s - omega t, <r~, r> and |r|^2; six waves,
// one per pair of components.  x has the precision of the other vectors.
template <int P>
__global__ void __launch_bounds__(6 * kSplitSites) k_it_xr(ItArgs a) {
  typedef typename real_of<P>::type T;
  __shared__ double sh[3][6][kSplitSites];
  __shared__ SysState ls[kMaxRhs];
  const int blk = blockIdx.x;
  const BlockSeg bs = find_seg(a.segs, a.nseg, blk, kSplitSites);
  if (bs.seg < 0) return;  // uniform
  const SegPart sd = seg_part<P>(a.segs, bs.seg, 1);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = bs.t0 + lane;
  const int rhs = n % sd.nrhs;
  const bool valid = n < sd.nthr;
  auto view = [&](const SpinorPtr &f) { return seg_view(f, P, sd.voff, sd.nthr); };
  cplx<T> x[2], p[2], s[2], t[2], rt[2];
  if (valid) {
    load_pair<P, IO_INT>(view(a.s), n, w, s);
    load_pair<P, IO_INT>(view(a.t), n, w, t);
    load_pair<P, IO_INT>(view(a.p), n, w, p);
    load_pair<P, IO_INT>(view(a.x), n, w, x);
    load_pair<P, IO_INT>(view(a.rt), n, w, rt);
  }
  finish_local<3>(ls, a, sd, blk, bs.t0, w, lane, 6);
  double acc[3] = {0, 0, 0};
  if (valid && ls[rhs].done == 0) {
    const cplx<T> al = sc<T>(ls[rhs].alpha), om = sc<T>(ls[rhs].omega);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      x[q] = x[q] + al * p[q] + om * s[q];
      s[q] = s[q] - om * t[q];
      acc[0] += (double)rt[q].re * s[q].re + (double)rt[q].im * s[q].im;
      acc[1] += (double)rt[q].re * s[q].im - (double)rt[q].im * s[q].re;
      acc[2] += (double)s[q].re * s[q].re + (double)s[q].im * s[q].im;
    }
    store_pair<P, IO_INT>(view(a.x), n, w, x, 0.f);
    store_pair<P, IO_INT>(view(a.r), n, w, s, 0.f);
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) sh[k][w][lane] = acc[k];
  split_partials<3>(sh, a.part_out, blk, bs.t0, sd.nrhs, sd.pcap, w, lane);
}

// the last iteration's rho: one block per segment
__global__ void __launch_bounds__(512) k_it_end(ItArgs a) {
  __shared__ SysState ls[kMaxRhs];
  const int seg = blockIdx.x;
  const SegPart sd = seg_part<P64>(a.segs, seg, 0);
  int blk0 = 0;
  for (int s = 0; s < seg; ++s) blk0 += (a.segs[s].nthr + kSplitSites - 1) / kSplitSites;
  finish_local<3>(ls, a, sd, blk0, 0, threadIdx.x >> 6, threadIdx.x & 63, 8);
}

template <int P, int CLOVER>
static int iterations(const BatchOp &op, const SplitIter &v, int n, hipStream_t s) {
  ItArgs a{};
  a.segs = op.dev_segs;
  a.nseg = (int)op.segs.size();
  a.r = v.r;
  a.v = v.v;
  a.rt = v.rt;
  a.s = v.s;
  a.t = v.t;
  a.x = v.x;
  int nb = 0;
  for (const SegDesc &d : op.segs) nb += (d.nthr + kSplitSites - 1) / kSplitSites;
  int cur = 0, pc = 0;  // the current state buffer and p
  auto states = [&](int kind, int part) {
    a.kind = kind;
    a.part = v.part[part];
    a.in = v.st[cur];
    a.st = v.st[1 - cur];
    cur = 1 - cur;
  };
  for (int it = 0; it < n; ++it) {
    states(it ? FK_RHO : FK_NONE, 0);
    a.out = v.tmp;
    a.p = v.p[pc];
    a.own = v.p[1 - pc];
    pc = 1 - pc;
    hipLaunchKernelGGL((k_it_even<P, CLOVER, 0>), dim3(nb), dim3(8 * kSplitSites), 0, s, a);
    QCU_HIP(hipGetLastError());
    QCU_TRY(hop_split_red(op, P, v.v, v.tmp, v.p[pc], RED_DOT_Y_OUT, v.rt, v.st[cur], v.part[0], s));
    states(FK_ALPHA, 0);
    a.own = v.s;
    hipLaunchKernelGGL((k_it_even<P, CLOVER, 1>), dim3(nb), dim3(8 * kSplitSites), 0, s, a);
    QCU_HIP(hipGetLastError());
    SpinorPtr none{};
    QCU_TRY(hop_split_red(op, P, v.t, v.tmp, v.s, RED_OUT_X, none, v.st[cur], v.part[1], s));
    states(FK_OMEGA, 1);
    a.p = v.p[pc];
    a.part_out = v.part[0];
    hipLaunchKernelGGL(k_it_xr<P>, dim3(nb), dim3(6 * kSplitSites), 0, s, a);
    QCU_HIP(hipGetLastError());
  }
  a.kind = FK_RHO;
  a.part = v.part[0];
  a.in = v.st[cur];
  a.st = v.st[0];
  hipLaunchKernelGGL(k_it_end, dim3((unsigned)op.segs.size()), dim3(512), 0, s, a);
  QCU_HIP(hipGetLastError());
  return 0;
}

int split_iterations(const BatchOp &op, int prec, const SplitIter &v, int n, hipStream_t s) {
  QCU_CHECK(n > 0 && n % 2 == 0, QCU_ERR_ARG, "split iterations come in pairs");
  QCU_CHECK(prec == P64 || prec == P32, QCU_ERR_ARG, "split iterations run in FP64 or FP32");
  if (prec == P64) return op.has_clover ? iterations<P64, 1>(op, v, n, s) : iterations<P64, 0>(op, v, n, s);
  return op.has_clover ? iterations<P32, 1>(op, v, n, s) : iterations<P32, 0>(op, v, n, s);
}

}  // namespace qcu
