// layout.hip -- external (PyQuda) <-> internal field layouts.
//
// External layouts (the C ABI, python/PyQuda/pyquda/field.py:72-78):
//   gauge  complex128 [4 mu][2 p][Vh][3][3]
//   spinor complex128 [Vh][4][3]  (one parity)
// The reference converts in place through a temporary and cuBLAS copies
// (src/lattice_cuda.cu:41-211); here the caller's buffers are only read (or
// only written), and the internal copies stay resident.
#include "qcu_hash.h"
#include "qcu_internal.h"

namespace qcu {

// ---- content hash of an external gauge field -------------------------------
// A 64-bit summary of every bit of the field, position-dependent, used by the
// reference-named entry points to keep converted links and the clover term
// while the caller's gauge is unchanged.  Each complex entry k is mixed with k
// (qcu_hash.h) and the mixed words are added modulo 2^64; addition commutes, so
// the result does not depend on the block order, and a load of the field forms it
// on the way.
QCU_D unsigned long long hash_entry(double2 v, long k) {
  return hash_mix((unsigned long long)__double_as_longlong(v.x), (unsigned long long)__double_as_longlong(v.y),
                  (unsigned long long)k);
}

// sum of h over the 256 threads of a block, in thread 0
QCU_D unsigned long long block_hash(unsigned long long h) {
  __shared__ unsigned long long sh[256];
  sh[threadIdx.x] = h;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  return sh[0];
}

constexpr int kHashBlocks = 1024;

__global__ void __launch_bounds__(256) k_gauge_hash(const double2 *ext, long n, unsigned long long *part) {
  unsigned long long h = 0;
  for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x)
    h += hash_entry(ext[k], k);
  h = block_hash(h);
  if (threadIdx.x == 0) part[blockIdx.x] = h;
}

// gate: a state whose done says whether the hash is another one than known
__global__ void __launch_bounds__(256) k_hash_sum(const unsigned long long *part, int n, unsigned long long *out,
                                                  unsigned long long known, SysState *gate) {
  unsigned long long h = 0;
  for (int k = threadIdx.x; k < n; k += blockDim.x) h += part[k];
  h = block_hash(h);
  if (threadIdx.x == 0) {
    *out = h;
    if (gate) gate->done = h != known;
  }
}

static int hash_sum(const void *part, long n, unsigned long long *out, unsigned long long known, SysState *gate,
                    hipStream_t s) {
  hipLaunchKernelGGL(k_hash_sum, dim3(1), dim3(256), 0, s, (const unsigned long long *)part, (int)n, out, known, gate);
  QCU_HIP(hipGetLastError());
  return 0;
}

int gauge_hash(const void *ext, const Geom &g, void *scratch, unsigned long long *out, unsigned long long known,
               SysState *gate, hipStream_t s) {
  const long n = 36L * 2 * g.vh;  // complex entries: [4][2][Vh][3][3]
  hipLaunchKernelGGL(k_gauge_hash, dim3(kHashBlocks), dim3(256), 0, s, (const double2 *)ext, n,
                     (unsigned long long *)scratch);
  QCU_HIP(hipGetLastError());
  return hash_sum(scratch, kHashBlocks, out, known, gate, s);
}

static long gauge_blocks(const Geom &g) { return (8L * g.vh + 255) / 256; }

size_t gauge_hash_scratch_bytes(const Geom &g) {
  const long nb = gauge_blocks(g);
  return (nb > kHashBlocks ? nb : kHashBlocks) * sizeof(unsigned long long);
}

// Links in every precision the lattice keeps, from one read of the field.
// 256 consecutive links (36 KiB) are staged through LDS with whole-line loads,
// then each thread takes rows 0 and 1 of its own link (a stride of 36 banks
// between lanes: no conflicts for 16-byte reads) and writes them
// component-planar.  HBM bound: 144 bytes read and 168 written per link with
// all three precisions.
template <int M, bool HASH>  // M bit k: precision k; HASH: partial content hashes as well
__global__ void __launch_bounds__(256) k_gauge_in(const double2 *ext, Geom g, GaugeOut o) {
  __shared__ double2 sh[256 * 9];
  const int vh = g.vh;
  const long total = 8L * vh;
  const long n0 = (long)blockIdx.x * 256;
  const int m = (int)(total - n0 < 256 ? total - n0 : 256) * 9;  // entries of this block
  unsigned long long h = 0;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const int k = q * 256 + threadIdx.x;
    if (k < m) {
      const double2 v = ext[n0 * 9 + k];
      sh[k] = v;
      if (HASH) h += hash_entry(v, n0 * 9 + k);
    }
  }
  if (HASH) {
    h = block_hash(h);
    if (threadIdx.x == 0) o.hash[blockIdx.x] = h;
  }
  __syncthreads();
  const long n = n0 + threadIdx.x;
  if (n >= total) return;
  const int pm = (int)(n / vh), i = (int)(n - (long)pm * vh);
  const int mu = pm >> 1, p = pm & 1;  // external order [mu][p]
  const int slab = p * 4 + mu;         // internal order [p][mu]
  double2 u[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) u[k] = sh[threadIdx.x * 9 + k];
  if (M & 1) {
    double2 *dst = (double2 *)o.u64 + (size_t)slab * 6 * vh + i;
#pragma unroll
    for (int k = 0; k < 6; ++k) dst[(size_t)k * vh] = u[k];
  }
  if (M & 2) {
    float4 *dst = (float4 *)o.u32 + (size_t)slab * 3 * vh + i;
#pragma unroll
    for (int k = 0; k < 3; ++k)
      dst[(size_t)k * vh] = make_float4((float)u[2 * k].x, (float)u[2 * k].y, (float)u[2 * k + 1].x,
                                        (float)u[2 * k + 1].y);
  }
  if (M & 4) {
    unsigned w[6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
      w[k] = (unsigned)f2h((float)u[k].x) | ((unsigned)f2h((float)u[k].y) << 16);
    ((uint4 *)o.u16a)[(size_t)slab * vh + i] = make_uint4(w[0], w[1], w[2], w[3]);
    ((uint2 *)o.u16b)[(size_t)slab * vh + i] = make_uint2(w[4], w[5]);
  }
}

int gauge_ext_to_internal(const void *ext, const Geom &g, int mask, const GaugeOut &o, hipStream_t s) {
  const dim3 nb((unsigned)gauge_blocks(g)), bs(256);
  const double2 *e = (const double2 *)ext;
  if (o.hash) {
    QCU_CHECK(mask == 1, QCU_ERR_ARG, "bad precision mask");
    hipLaunchKernelGGL((k_gauge_in<1, true>), nb, bs, 0, s, e, g, o);
    QCU_HIP(hipGetLastError());
    return hash_sum(o.hash, nb.x, o.hash_out, 0, nullptr, s);
  }
  switch (mask) {
    case 1: hipLaunchKernelGGL((k_gauge_in<1, false>), nb, bs, 0, s, e, g, o); break;
    case 3: hipLaunchKernelGGL((k_gauge_in<3, false>), nb, bs, 0, s, e, g, o); break;
    case 5: hipLaunchKernelGGL((k_gauge_in<5, false>), nb, bs, 0, s, e, g, o); break;
    case 7: hipLaunchKernelGGL((k_gauge_in<7, false>), nb, bs, 0, s, e, g, o); break;
    default: set_error(QCU_ERR_ARG, "bad precision mask"); return QCU_ERR_ARG;
  }
  QCU_HIP(hipGetLastError());
  return 0;
}

// external one-parity field [Vh][4][3] <-> system (segment seg, rhs r) of a batch vector,
// FP32 or FP16
template <int P>
__global__ void k_spinor_in(const double2 *ext, int vh, int nrhs, int rhs, SpinorPtr dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  typedef typename real_of<P>::type T;
  cplx<T> v[12];
  const double2 *src = ext + (size_t)i * 12;
#pragma unroll
  for (int k = 0; k < 12; ++k) {
    double2 a = src[k];
    v[k] = mk<T>((T)a.x, (T)a.y);
  }
  SpinorIO<P>::store(dst, i * nrhs + rhs, v);
}

template <int P>
__global__ void k_spinor_out(SpinorPtr src, int vh, int nrhs, int rhs, double2 *ext) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= vh) return;
  typedef typename real_of<P>::type T;
  cplx<T> v[12];
  SpinorIO<P>::load(src, i * nrhs + rhs, v);
  double2 *dst = ext + (size_t)i * 12;
#pragma unroll
  for (int k = 0; k < 12; ++k) dst[k] = make_double2((double)v[k].re, (double)v[k].im);
}

int spinor_ext_to_batch(const void *ext, const BatchOp &op, int seg, int rhs, SpinorPtr dst, int prec,
                        hipStream_t s) {
  QCU_CHECK(seg >= 0 && seg < (int)op.segs.size(), QCU_ERR_ARG, "bad segment");
  const SegDesc &d = op.segs[seg];
  QCU_CHECK(rhs >= 0 && rhs < d.nrhs, QCU_ERR_ARG, "bad right-hand side");
  const SpinorPtr v = seg_view(dst, prec, d.voff, d.nthr);
  const int vh = d.g.vh, bs = 256, nb = (vh + bs - 1) / bs;
  const double2 *e = (const double2 *)ext;
  switch (prec) {
    case P32: hipLaunchKernelGGL(k_spinor_in<P32>, dim3(nb), dim3(bs), 0, s, e, vh, d.nrhs, rhs, v); break;
    case P16: hipLaunchKernelGGL(k_spinor_in<P16>, dim3(nb), dim3(bs), 0, s, e, vh, d.nrhs, rhs, v); break;
    default: set_error(QCU_ERR_ARG, "bad precision"); return QCU_ERR_ARG;
  }
  QCU_HIP(hipGetLastError());
  return 0;
}

int spinor_batch_to_ext(SpinorPtr src, const BatchOp &op, int seg, int rhs, void *ext, int prec, hipStream_t s) {
  QCU_CHECK(seg >= 0 && seg < (int)op.segs.size(), QCU_ERR_ARG, "bad segment");
  const SegDesc &d = op.segs[seg];
  QCU_CHECK(rhs >= 0 && rhs < d.nrhs, QCU_ERR_ARG, "bad right-hand side");
  const SpinorPtr v = seg_view(src, prec, d.voff, d.nthr);
  const int vh = d.g.vh, bs = 256, nb = (vh + bs - 1) / bs;
  double2 *e = (double2 *)ext;
  switch (prec) {
    case P32: hipLaunchKernelGGL(k_spinor_out<P32>, dim3(nb), dim3(bs), 0, s, v, vh, d.nrhs, rhs, e); break;
    case P16: hipLaunchKernelGGL(k_spinor_out<P16>, dim3(nb), dim3(bs), 0, s, v, vh, d.nrhs, rhs, e); break;
    default: set_error(QCU_ERR_ARG, "bad precision"); return QCU_ERR_ARG;
  }
  QCU_HIP(hipGetLastError());
  return 0;
}

// All right-hand sides of a segment and both parities (blockIdx.y) in one launch:
// thread = virtual site, so that the batch vector is accessed whole lines at a
// time (one launch per right-hand side touched 16 bytes in every nrhs * 16:
// 12 right-hand sides at 24^3x48 193 us each to load, 126 us to store).
struct ExtFields {
  double2 *f[kMaxRhs];
};

__global__ void __launch_bounds__(256) k_systems_in(ExtFields ext, int vh, int nrhs, SpinorPtr even, SpinorPtr odd) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= vh * nrhs) return;
  const int i = t / nrhs, r = t - i * nrhs, p = blockIdx.y;
  const double2 *src = ext.f[r] + ((size_t)p * vh + i) * 12;
  cplx<double> v[12];
#pragma unroll
  for (int k = 0; k < 12; ++k) {
    const double2 a = ld_at<double2>(src, 0, 16u * k);
    v[k] = mk(a.x, a.y);
  }
  SpinorIO<P64>::store(p ? odd : even, t, v);
}

__global__ void __launch_bounds__(256) k_systems_out(ExtFields ext, int vh, int nrhs, SpinorPtr even, SpinorPtr odd) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= vh * nrhs) return;
  const int i = t / nrhs, r = t - i * nrhs, p = blockIdx.y;
  double2 *dst = ext.f[r] + ((size_t)p * vh + i) * 12;
  cplx<double> v[12];
  SpinorIO<P64>::load(p ? odd : even, t, v);
#pragma unroll
  for (int k = 0; k < 12; ++k) st_at<double2>(dst, 0, 16u * k, make_double2(v[k].re, v[k].im));
}

static int move_systems(bool in, void *const *ext, const BatchOp &op, SpinorPtr even, SpinorPtr odd, hipStream_t s) {
  for (const SegDesc &d : op.segs) {
    ExtFields e{};
    for (int r = 0; r < d.nrhs; ++r) e.f[r] = (double2 *)ext[d.sys0 + r];
    const SpinorPtr ev = seg_view(even, P64, d.voff, d.nthr), od = seg_view(odd, P64, d.voff, d.nthr);
    const dim3 nb((unsigned)((d.nthr + 255) / 256), 2);
    if (in)
      hipLaunchKernelGGL(k_systems_in, nb, dim3(256), 0, s, e, d.g.vh, d.nrhs, ev, od);
    else
      hipLaunchKernelGGL(k_systems_out, nb, dim3(256), 0, s, e, d.g.vh, d.nrhs, ev, od);
    QCU_HIP(hipGetLastError());
  }
  return 0;
}

int systems_to_batch(const void *const *ext, const BatchOp &op, SpinorPtr even, SpinorPtr odd, hipStream_t s) {
  return move_systems(true, const_cast<void *const *>(ext), op, even, odd, s);
}

int batch_to_systems(SpinorPtr even, SpinorPtr odd, const BatchOp &op, void *const *ext, hipStream_t s) {
  return move_systems(false, ext, op, even, odd, s);
}

}  // namespace qcu
