// dslash.hip -- even-odd Wilson / clover hopping term for gfx950.
//
// out_p(x) = sum_mu (1 - g_mu) U_mu(x) psi(x+mu) + (1 + g_mu) U_mu(x-mu)^dag psi(x-mu)
// on the sites of output parity p, psi on parity 1-p: the operator of
// src/wilson_dslash.cu:9-245 with the spin projectors of the DeGrand-Rossi
// basis written out as half-spinor (two 3-vectors) products, the 12-real link
// reconstruction of include/define.h:198-206, periodic wrap in every direction
// (the single-GPU case of include/lattice_dslash.h:11-197) and an optional -1
// phase on the hops that cross the time boundary.
//
// One thread per output site, site-fastest SoA loads (coalesced 16-byte lanes),
// eight directions fused, optional epilogues: packed clover inverse (two
// Hermitian 6x6 blocks, src/clover_dslash.cu:857-882 restricted to its
// non-zero chiral blocks), x - k2 * (...) for the even-odd Schur operator
// (src/bistabcg.cu:85-96), and fused FP64 grid reductions feeding the BiCGSTAB
// scalar epilogues.  The stencil is HBM bound (about 0.5 flop per byte), so
// no matrix cores are involved.
#include "qcu_hop.h"
#include "qcu_internal.h"
#include "qcu_solver.h"
#include "qcu_state.h"

namespace qcu {

struct HopKArgs {
  SpinorPtr out, in, x, y;  // batch vectors
  const SegDesc *segs;
  int nseg;
  int parity;
  int remap;
  const SysState *st;  // per-system states, or null
  double *partials;
};

// G: scheduling groups.  0 lets the compiler hoist every load of the eight
// directions (most memory-level parallelism, most registers); 1 and 2 fence the
// instruction schedule after every direction / every pair of directions, which
// caps the live registers and raises occupancy (the FP64 kernel needs this).
#define QCU_GROUP_FENCE(G, k)                                                      \
  do {                                                                             \
    if ((G) == 1 || ((G) == 2 && ((k) & 1))) __builtin_amdgcn_sched_barrier(0);    \
  } while (0)

// parity and block of a launch: with EPI_MAT one launch covers both parities,
// in alternate blocks
template <int EPI>
QCU_D int hop_block(const HopKArgs &a, int &parity) {
  const int b = remap_block(blockIdx.x, gridDim.x, a.remap);
  parity = EPI == EPI_MAT ? (b & 1) : a.parity;
  return EPI == EPI_MAT ? b >> 1 : b;
}

// the fields of a launch for one segment (and parity): EPI_MAT works on full
// external fields
template <int P, int IO, int EPI>
QCU_D SpinorPtr hop_field(const SpinorPtr &f, const SegPart &sd, int parity) {
  if (IO == IO_INT) return seg_view(f, P, sd.voff, sd.nthr);
  SpinorPtr v = f;
  if (EPI == EPI_MAT) v.p = (char *)f.p + (size_t)parity * sd.g.vh * 192;
  return v;
}

template <int P, int IO, int CLOVER, int EPI, int RED, int G, bool NT>
__global__ void __launch_bounds__(256) k_hop(HopKArgs a) {
  typedef typename real_of<P>::type T;
  int p;
  const int blk = hop_block<EPI>(a, p);
  const BlockSeg bs = find_seg(a.segs, a.nseg, blk, blockDim.x);
  if (bs.seg < 0) return;  // uniform: a block past the last segment
  const SegPart sd = seg_part<P>(a.segs, bs.seg, p);
  const Geom g = sd.g;
  const int nrhs = IO == IO_EXT ? 1 : sd.nrhs;
  const int n = bs.t0 + threadIdx.x;
  const int k = n / nrhs, rhs = n - k * nrhs;
  bool active = n < sd.nthr;
  // a solver state, when given, stops the work of its system once it has stopped
  if (a.st && active && a.st[sd.sys0 + rhs].done) active = false;
  cplx<T> d[12];
  double red[3] = {0, 0, 0};
  if (active) {
    const int q = 1 - p;
    const SpinorPtr in = hop_field<P, IO, EPI>(a.in, sd, q);
    const LinkPtr U = sd.U;
    int i;
    const Site s = ordered_site(g, sd.zslab, k, p, i);
    const int t = i * nrhs + rhs;
#pragma unroll
    for (int k = 0; k < 12; ++k) d[k] = mk<T>(0, 0);
    int j, sg;
    // branch-free index arithmetic keeps the body one basic block, so the
    // scheduling fences below bound the live registers
    j = neighbour<0, 0>(g, s, i, sg);
    hop_dir<P, IO, 0, 0, NT>(d, U, q * 4 + 0, j, in, j * nrhs + rhs, (T)1);
    QCU_GROUP_FENCE(G, 0);
    j = neighbour<0, 1>(g, s, i, sg);
    hop_dir<P, IO, 0, 1, NT>(d, U, p * 4 + 0, i, in, j * nrhs + rhs, (T)1);
    QCU_GROUP_FENCE(G, 1);
    j = neighbour<1, 0>(g, s, i, sg);
    hop_dir<P, IO, 1, 0, NT>(d, U, q * 4 + 1, j, in, j * nrhs + rhs, (T)1);
    QCU_GROUP_FENCE(G, 2);
    j = neighbour<1, 1>(g, s, i, sg);
    hop_dir<P, IO, 1, 1, NT>(d, U, p * 4 + 1, i, in, j * nrhs + rhs, (T)1);
    QCU_GROUP_FENCE(G, 3);
    j = neighbour<2, 0>(g, s, i, sg);
    hop_dir<P, IO, 2, 0, NT>(d, U, q * 4 + 2, j, in, j * nrhs + rhs, (T)1);
    QCU_GROUP_FENCE(G, 4);
    j = neighbour<2, 1>(g, s, i, sg);
    hop_dir<P, IO, 2, 1, NT>(d, U, p * 4 + 2, i, in, j * nrhs + rhs, (T)1);
    QCU_GROUP_FENCE(G, 5);
    j = neighbour<3, 0>(g, s, i, sg);
    hop_dir<P, IO, 3, 0, NT>(d, U, q * 4 + 3, j, in, j * nrhs + rhs, (T)sg);
    QCU_GROUP_FENCE(G, 6);
    j = neighbour<3, 1>(g, s, i, sg);
    hop_dir<P, IO, 3, 1, NT>(d, U, p * 4 + 3, i, in, j * nrhs + rhs, (T)sg);
    QCU_GROUP_FENCE(G, 7);
    if (EPI == EPI_MAT) {
      // A x - kappa d
      cplx<T> x[12];
      load_spinor<P, IO>(hop_field<P, IO, EPI>(a.in, sd, p), t, x);
      if (CLOVER) {
        T c[36];
        clover_load_block<NT>(sd.A, i, 0, c);
        clover_apply_block(c, x, 0);
        QCU_GROUP_FENCE(G, 1);
        clover_load_block<NT>(sd.A, i, 1, c);
        clover_apply_block(c, x, 1);
      }
      const T kap = (T)sd.kappa;
#pragma unroll
      for (int k = 0; k < 12; ++k) d[k] = nmad(x[k], kap, d[k]);
    } else if (CLOVER) {
      const CloverPtr C = sd.Cinv;
      if constexpr (P == P16) {
        T c[72];
        const float nrm = CloverIO<P>::template load<NT>(C, i, c);
        clover_apply_site<true>(c, d);
#pragma unroll
        for (int k = 0; k < 12; ++k) d[k] = scale_(nrm, d[k]);
      } else {
        // one chiral block at a time bounds the live registers
        T c[36];
        clover_load_block<NT>(C, i, 0, c);
        clover_apply_block(c, d, 0);
        QCU_GROUP_FENCE(G, 1);
        clover_load_block<NT>(C, i, 1, c);
        clover_apply_block(c, d, 1);
      }
    }
    if (EPI == EPI_XPAY) {
      cplx<T> x[12];
      SpinorIO<P>::load(seg_view(a.x, P, sd.voff, sd.nthr), t, x);
      const T k2 = (T)(sd.kappa * sd.kappa);
#pragma unroll
      for (int k = 0; k < 12; ++k) d[k] = nmad(x[k], k2, d[k]);
      if (RED == RED_OUT_X) {
        // <out, x> and |out|^2
#pragma unroll
        for (int k = 0; k < 12; ++k) {
          red[0] += (double)d[k].re * (double)x[k].re + (double)d[k].im * (double)x[k].im;
          red[1] += (double)d[k].re * (double)x[k].im - (double)d[k].im * (double)x[k].re;
          red[2] += (double)d[k].re * (double)d[k].re + (double)d[k].im * (double)d[k].im;
        }
      }
    }
    if (RED == RED_RES) {
      cplx<T> y[12];
      SpinorIO<P>::load(seg_view(a.y, P, sd.voff, sd.nthr), t, y);
#pragma unroll
      for (int k = 0; k < 12; ++k) {
        d[k] = y[k] - d[k];
        red[0] += (double)norm2(d[k]);
      }
    }
    if (RED == RED_DOT_Y_OUT) {
      cplx<T> y[12];
      SpinorIO<P>::load(seg_view(a.y, P, sd.voff, sd.nthr), t, y);
#pragma unroll
      for (int k = 0; k < 12; ++k) {
        red[0] += (double)y[k].re * (double)d[k].re + (double)y[k].im * (double)d[k].im;
        red[1] += (double)y[k].re * (double)d[k].im - (double)y[k].im * (double)d[k].re;
      }
    }
    store_spinor<P, IO>(hop_field<P, IO, EPI>(a.out, sd, p), t, d);
  }
  if (RED == RED_DOT_Y_OUT) {
    double v[2] = {red[0], red[1]};
    block_partial_rhs<2>(v, a.partials, blk, bs.t0, nrhs, sd.pcap);
  } else if (RED == RED_OUT_X) {
    block_partial_rhs<3>(red, a.partials, blk, bs.t0, nrhs, sd.pcap);
  } else if (RED == RED_RES) {
    double v[1] = {red[0]};
    block_partial_rhs<1>(v, a.partials, blk, bs.t0, nrhs, sd.pcap);
  }
}

// ---- eight waves per 64 sites ----------------------------------------------
// The same operator with one wave per direction: a lattice too small to fill the
// chip with one thread per site (8^4: 32 waves for 256 CUs) is bound by the
// latency of the eight hops one after the other.  Each of the 8 waves of a block
// transports its direction's half spinor for the block's 64 sites into LDS; then
// wave w < 6 forms components 2w and 2w + 1 of the result (every sum in the
// order of k_hop, so the results are the same bit for bit), applies rows of the
// clover block and the epilogue, and stores its pair of components.
template <int P, int IO, int CLOVER, int EPI, int RED>
__global__ void __launch_bounds__(8 * kSplitSites) k_hop_split(HopKArgs a) {
  typedef typename real_of<P>::type T;
  __shared__ cplx<T> half[8][6][kSplitSites];
  int p;
  const int blk = hop_block<EPI>(a, p);
  const BlockSeg bs = find_seg(a.segs, a.nseg, blk, kSplitSites);
  if (bs.seg < 0) return;  // uniform
  const SegPart sd = seg_part<P>(a.segs, bs.seg, p);
  const Geom g = sd.g;
  const int nrhs = IO == IO_EXT ? 1 : sd.nrhs;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = bs.t0 + lane;
  const int k = n / nrhs, rhs = n - k * nrhs;
  bool active = n < sd.nthr;
  int i;
  const Site s = ordered_site(g, sd.zslab, k, p, i);
  const int t = i * nrhs + rhs;
  if (a.st && active && a.st[sd.sys0 + rhs].done) active = false;
  const bool mine = active && w < 6;  // this wave's pair of components
  const int cb = w / 3, cj = w - 3 * cb;  // its chiral block and rows 2 cj, 2 cj + 1 of it
  CloverRows<P> cr;
  if (active) {
    const int q = 1 - p;
    const SpinorPtr in = hop_field<P, IO, EPI>(a.in, sd, q);
    const LinkPtr U = sd.U;
    cplx<T> a0[3], a1[3];
    int j, sg;
#define QCU_SPLIT_DIR(MU)                                                                 \
  case 2 * MU:                                                                            \
    j = neighbour<MU, 0>(g, s, i, sg);                                                    \
    hop_half<P, IO, MU, 0>(a0, a1, U, q * 4 + MU, j, in, j * nrhs + rhs, (T)sg);          \
    break;                                                                                \
  case 2 * MU + 1:                                                                        \
    j = neighbour<MU, 1>(g, s, i, sg);                                                    \
    hop_half<P, IO, MU, 1>(a0, a1, U, p * 4 + MU, i, in, j * nrhs + rhs, (T)sg);          \
    break;
    switch (w) {
      QCU_SPLIT_DIR(0)
      QCU_SPLIT_DIR(1)
      QCU_SPLIT_DIR(2)
      QCU_SPLIT_DIR(3)
    }
#undef QCU_SPLIT_DIR
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      half[w][c][lane] = a0[c];
      half[w][3 + c][lane] = a1[c];
    }
  }
  // in flight over the barriers and the sum
  cplx<T> d[2] = {mk<T>(0, 0), mk<T>(0, 0)}, x[2] = {mk<T>(0, 0), mk<T>(0, 0)}, y[2];
  if (mine) {
    if (CLOVER) cr.load(EPI == EPI_MAT ? sd.A : sd.Cinv, i, cb, cj);
    if (EPI == EPI_MAT) load_pair<P, IO>(hop_field<P, IO, EPI>(a.in, sd, p), t, w, x);
    if (EPI == EPI_XPAY) load_pair<P, IO_INT>(seg_view(a.x, P, sd.voff, sd.nthr), t, w, x);
    if (RED == RED_DOT_Y_OUT || RED == RED_RES) load_pair<P, IO_INT>(seg_view(a.y, P, sd.voff, sd.nthr), t, w, y);
  }
  __syncthreads();
  if (mine) {
#pragma unroll
    for (int q = 0; q < 2; ++q) d[q] = hop_sum(half, 2 * w + q, lane);
  }
  if (CLOVER) {
    // the clover term acts on the sum (its inverse), or on x (EPI_MAT)
    cplx<T>(*v)[kSplitSites] = half[0];  // 12 components over the first two directions' slots
    __syncthreads();
    if (mine) {
#pragma unroll
      for (int q = 0; q < 2; ++q) v[2 * w + q][lane] = EPI == EPI_MAT ? x[q] : d[q];
    }
    __syncthreads();
    if (mine) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const cplx<T> y = cr.row(cj, q, v + 6 * cb, lane);
        if (EPI == EPI_MAT)
          x[q] = y;
        else
          d[q] = y;
      }
    }
  }
  double red[3] = {0, 0, 0};
  if (mine) {
    if (EPI == EPI_MAT) {
      const T kap = (T)sd.kappa;
#pragma unroll
      for (int q = 0; q < 2; ++q) d[q] = nmad(x[q], kap, d[q]);
    }
    if (EPI == EPI_XPAY) {
      const T k2 = (T)(sd.kappa * sd.kappa);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        d[q] = nmad(x[q], k2, d[q]);
        if (RED == RED_OUT_X) {
          red[0] += (double)d[q].re * (double)x[q].re + (double)d[q].im * (double)x[q].im;
          red[1] += (double)d[q].re * (double)x[q].im - (double)d[q].im * (double)x[q].re;
          red[2] += (double)d[q].re * (double)d[q].re + (double)d[q].im * (double)d[q].im;
        }
      }
    }
    if (RED == RED_RES) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        d[q] = y[q] - d[q];
        red[0] += (double)norm2(d[q]);
      }
    }
    if (RED == RED_DOT_Y_OUT) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        red[0] += (double)y[q].re * (double)d[q].re + (double)y[q].im * (double)d[q].im;
        red[1] += (double)y[q].re * (double)d[q].im - (double)y[q].im * (double)d[q].re;
      }
    }
  }
  float m = 0.f;
  if (P == P16) {  // the site's scale over all 12 components
    __shared__ float mx[6][kSplitSites];
    if (w < 6)
      mx[w][lane] = fmaxf(fmaxf(fabsf((float)d[0].re), fabsf((float)d[0].im)),
                          fmaxf(fabsf((float)d[1].re), fabsf((float)d[1].im)));
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 6; ++k) m = fmaxf(m, mx[k][lane]);
  }
  if (mine) store_pair<P, IO>(hop_field<P, IO, EPI>(a.out, sd, p), t, w, d, m);
  if (RED != RED_NONE) {
    // the six waves' sums per site, added in order, then the sites of each system
    constexpr int NR = RED == RED_RES ? 1 : (RED == RED_DOT_Y_OUT ? 2 : 3);
    __shared__ double sh[NR][6][kSplitSites];
    if (w < 6) {
#pragma unroll
      for (int k = 0; k < NR; ++k) sh[k][w][lane] = red[k];
    }
    split_partials<NR>(sh, a.partials, blk, bs.t0, nrhs, sd.pcap, w, lane);
  }
}

static int total_blocks(const std::vector<SegDesc> &segs, int bsz) {
  int nb = 0;
  for (const SegDesc &d : segs) nb += (d.nthr + bsz - 1) / bsz;
  return nb;
}

template <int P, int IO, int CLOVER, int EPI, int RED, bool NT>
static void launch_group(const HopKArgs &a, int nb, const LaunchCfg &cfg, hipStream_t s) {
  const dim3 n(nb), b(cfg.block);
  switch (cfg.group) {
    case 1: hipLaunchKernelGGL((k_hop<P, IO, CLOVER, EPI, RED, 1, NT>), n, b, 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_hop<P, IO, CLOVER, EPI, RED, 2, NT>), n, b, 0, s, a); break;
    default: hipLaunchKernelGGL((k_hop<P, IO, CLOVER, EPI, RED, 0, NT>), n, b, 0, s, a); break;
  }
}

template <int P, int IO, int CLOVER, int EPI, int RED>
static int launch(const HopKArgs &a, int nb, bool split, bool nt, const LaunchCfg &cfg, hipStream_t s) {
  if (split) {
    hipLaunchKernelGGL((k_hop_split<P, IO, CLOVER, EPI, RED>), dim3(nb), dim3(8 * kSplitSites), 0, s, a);
  } else if (nt) {
    launch_group<P, IO, CLOVER, EPI, RED, true>(a, nb, cfg, s);
  } else {
    launch_group<P, IO, CLOVER, EPI, RED, false>(a, nb, cfg, s);
  }
  QCU_HIP(hipGetLastError());
  return 0;
}

template <int P>
static int dispatch(const HopKArgs &a, int nb, int clover, int epi, int red, bool split, bool nt,
                    const LaunchCfg &cfg, hipStream_t s) {
  constexpr int I = IO_INT;
  if (epi == EPI_PLAIN) {
    return clover ? launch<P, I, 1, EPI_PLAIN, RED_NONE>(a, nb, split, nt, cfg, s)
                  : launch<P, I, 0, EPI_PLAIN, RED_NONE>(a, nb, split, nt, cfg, s);
  }
  if (red == RED_NONE)
    return clover ? launch<P, I, 1, EPI_XPAY, RED_NONE>(a, nb, split, nt, cfg, s)
                  : launch<P, I, 0, EPI_XPAY, RED_NONE>(a, nb, split, nt, cfg, s);
  if constexpr (P == P64) {
    if (red == RED_RES)
      return clover ? launch<P, I, 1, EPI_XPAY, RED_RES>(a, nb, split, nt, cfg, s)
                    : launch<P, I, 0, EPI_XPAY, RED_RES>(a, nb, split, nt, cfg, s);
  }
  if (red == RED_DOT_Y_OUT)
    return clover ? launch<P, I, 1, EPI_XPAY, RED_DOT_Y_OUT>(a, nb, split, nt, cfg, s)
                  : launch<P, I, 0, EPI_XPAY, RED_DOT_Y_OUT>(a, nb, split, nt, cfg, s);
  return clover ? launch<P, I, 1, EPI_XPAY, RED_OUT_X>(a, nb, split, nt, cfg, s)
                : launch<P, I, 0, EPI_XPAY, RED_OUT_X>(a, nb, split, nt, cfg, s);
}

static int check_cfg(const LaunchCfg &cfg) {
  QCU_CHECK(cfg.block >= 64 && cfg.block <= 256 && cfg.block % 64 == 0, QCU_ERR_ARG,
            "block size must be a multiple of 64 in [64, 256]");
  return 0;
}

// Eight waves per 64 sites up to 32 768 virtual sites, where one thread per site
// gives the chip less than one wave per two SIMDs.  Hop in us, split against one
// thread per site: 8^4 Wilson FP64 4.9 / 6.9, FP32 4.3 / 6.5; 16^4 (32 768 sites)
// Wilson FP64 8.8 / 11.3, FP32 6.3 / 8.4, FP16 6.2 / 7.7, clover FP64 13.1 / 13.8,
// FP16 8.6 / 8.6; 16^3x24 (49 152) Wilson FP64 13.6 / 13.1, clover 18.3 / 16.6.
constexpr long long kSplitMax = 32768;
bool hop_is_split(const BatchOp &op, const LaunchCfg &cfg) { return cfg.automatic && op.nvsites <= kSplitMax; }

// Links and clover blocks are read once per launch.  Where they do not stay in
// the 256 MB Infinity Cache from one launch to the next, non-temporal loads leave
// more of the caches to the spinors, each of which is read eight times.  Clover
// hop with xpay in us, plain against non-temporal: 32^3x64 FP64 457 / 431, FP32
// 213 / 199, FP16 111 / 103; 24^3x48 FP64 142 / 131, FP32 65 / 60; but where the
// fields fit, 24^3x48 FP16 33.7 / 36.0, Wilson FP32 43.6 / 46.2.
static bool use_nt(const BatchOp &op, int prec, bool clover) {
  const double real = prec == P64 ? 8 : (prec == P32 ? 4 : 2);
  double bytes = 0;
  for (const SegDesc &d : op.segs) bytes += (double)d.g.vh * real * (8 * 12 + (clover ? 72 : 0) + 2 * 24 * d.nrhs);
  return bytes > 256e6;
}

int hop_split_red(const BatchOp &op, int prec, SpinorPtr out, SpinorPtr in, SpinorPtr x, int red, SpinorPtr y,
                  SysState *st, double *partials, hipStream_t s) {
  QCU_CHECK(prec == P64 || prec == P32, QCU_ERR_ARG, "split iterations run in FP64 or FP32");
  HopKArgs a{};
  a.out = out;
  a.in = in;
  a.x = x;
  a.y = y;
  a.segs = op.dev_segs;
  a.nseg = (int)op.segs.size();
  a.parity = 1;
  a.remap = 1;
  a.st = st;
  a.partials = partials;
  const int nb = total_blocks(op.segs, kSplitSites);
  const LaunchCfg cfg;
  return prec == P64 ? dispatch<P64>(a, nb, op.has_clover, EPI_XPAY, red, true, false, cfg, s)
                     : dispatch<P32>(a, nb, op.has_clover, EPI_XPAY, red, true, false, cfg, s);
}

int hop_ext(const BatchOp &op, void *out, const void *in, int parity, int mat, bool use_clover, hipStream_t s,
            const SysState *gate) {
  QCU_CHECK(op.segs.size() == 1 && op.nsys == 1, QCU_ERR_ARG, "external fields: one lattice, one right-hand side");
  LaunchCfg cfg = tuned_cfg(op, P64);
  QCU_TRY(check_cfg(cfg));
  HopKArgs a{};
  a.out.p = out;
  a.in.p = const_cast<void *>(in);
  a.segs = op.dev_segs;
  a.nseg = 1;
  a.parity = parity;
  a.remap = cfg.remap;
  a.st = gate;
  const int clover = use_clover && op.has_clover;
  const bool split = hop_is_split(op, cfg), nt = use_nt(op, P64, clover);
  const int nb = total_blocks(op.segs, split ? kSplitSites : cfg.block) * (mat ? 2 : 1);
  if (mat)
    return clover ? launch<P64, IO_EXT, 1, EPI_MAT, RED_NONE>(a, nb, split, nt, cfg, s)
                  : launch<P64, IO_EXT, 0, EPI_MAT, RED_NONE>(a, nb, split, nt, cfg, s);
  return clover ? launch<P64, IO_EXT, 1, EPI_PLAIN, RED_NONE>(a, nb, split, nt, cfg, s)
                : launch<P64, IO_EXT, 0, EPI_PLAIN, RED_NONE>(a, nb, split, nt, cfg, s);
}

int hop(const BatchOp &op, int prec, SpinorPtr out, SpinorPtr in, int parity, int epi, SpinorPtr x, int red,
        SpinorPtr y, SysState *st, double *partials, const LaunchCfg &cfg, hipStream_t s, bool use_clover) {
  QCU_CHECK(parity == 0 || parity == 1, QCU_ERR_ARG, "parity must be 0 or 1");
  QCU_CHECK(prec >= P64 && prec <= P16, QCU_ERR_ARG, "unknown precision");
  QCU_TRY(check_cfg(cfg));
  QCU_CHECK(red == RED_NONE || (epi == EPI_XPAY && st && partials), QCU_ERR_ARG,
            "fused reductions need the xpay epilogue and solver state");
  QCU_CHECK(red != RED_RES || prec == P64, QCU_ERR_ARG, "residuals are formed in FP64");
  HopKArgs a;
  a.out = out;
  a.in = in;
  a.x = x;
  a.y = y;
  a.segs = op.dev_segs;
  a.nseg = (int)op.segs.size();
  a.parity = parity;
  a.remap = cfg.remap;
  a.st = red == RED_RES ? nullptr : st;  // residuals of every system, stopped or not
  a.partials = partials;
  const int clover = use_clover && op.has_clover;
  const bool split = hop_is_split(op, cfg), nt = use_nt(op, prec, clover);
  const int bsz = split ? kSplitSites : cfg.block;
  const int nb = total_blocks(op.segs, bsz);
  int rc;
  switch (prec) {
    case P64: rc = dispatch<P64>(a, nb, clover, epi, red, split, nt, cfg, s); break;
    case P32: rc = dispatch<P32>(a, nb, clover, epi, red, split, nt, cfg, s); break;
    default: rc = dispatch<P16>(a, nb, clover, epi, red, split, nt, cfg, s); break;
  }
  if (rc || red == RED_NONE) return rc;
  if (red == RED_RES) return finish(op, partials, bsz, 1, FK_STORE_TMP, st, nullptr, s);
  return red == RED_DOT_Y_OUT ? finish(op, partials, bsz, 2, FK_ALPHA, st, nullptr, s)
                              : finish(op, partials, bsz, 3, FK_OMEGA, st, nullptr, s);
}

}  // namespace qcu
