"""A row of a clover block: the diagonal's product and the first off-diagonal one are
added with one rounding, in FP32 and FP64 and in either kernel's form of the sum."""
import host_code

PROGRAM = r"""
using namespace qcu;
static unsigned long long seed = 11;
static double uniform() {
  seed = seed * 6364136223846793005ull + 1442695040888963407ull;
  return (double)(seed >> 11) * 0x1p-52 - 1;
}
// a b + c rounded once (FP64 holds the products of FP32 and, but for a last rounding
// far below FP32's, their sums)
static float once(float a, float b, float c) { return (float)((double)a * b + c); }
static double once(double a, double b, double c) { return std::fma(a, b, c); }
template <class T>
static int check() {
  for (int pass = 0; pass < 2000; ++pass)
    for (int r = 0; r < 6; ++r) {
      // a block of the diagonal and the first off-diagonal entry of row r
      T cb[36] = {};
      const int col = r ? 0 : 1, k = r ? 6 + r * (r - 1) : 6;
      cb[r] = (T)uniform();
      cb[k] = (T)uniform();
      cb[k + 1] = (T)uniform();
      cplx<T> v[12];
      for (auto &e : v) e = mk((T)uniform(), (T)uniform());
      const cplx<T> d = v[r], x = v[col];
      const T im = r ? cb[k + 1] : -cb[k + 1];
      const T pre = once(cb[k], x.re, -(im * x.im)), pim = once(cb[k], x.im, im * x.re);
      clover_apply_block(cb, v, 0);
      if (v[r].re != once(cb[r], d.re, pre) || v[r].im != once(cb[r], d.im, pim))
        return printf("row %d, %d bytes: %.17g %.17g\n", r, (int)sizeof(T), (double)v[r].re, (double)v[r].im), 1;
    }
  return 0;
}
int main() { return check<float>() || check<double>(); }
"""


def test_row_begins_with_one_rounding(tmp_path):
    host_code.run(tmp_path, "#pragma clang fp contract(off)\n" + PROGRAM, ["qcu_common.h"])
