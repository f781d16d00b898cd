"""The content hash that decides whether resident links still are the caller's:
every change a program makes to a gauge field in place has to change it."""
import host_code

# exit 1 with a line per kind of change that some field does not show
PROGRAM = r"""
using namespace qcu;
typedef unsigned long long u64;
static u64 seed = 7;
static double uniform() {
  seed = seed * 6364136223846793005ull + 1442695040888963407ull;
  return ((seed >> 11) + 1) * 0x1p-53;
}
static u64 bits(double x) { u64 b; memcpy(&b, &x, 8); return b; }
typedef std::vector<double> Field;  // [4][2][Vh][3][3] complex
static u64 hash(const Field &f) {
  u64 h = 0;
  for (size_t k = 0; k < f.size() / 2; ++k) h += hash_mix(bits(f[2 * k]), bits(f[2 * k + 1]), k);
  return h;
}
int main() {
  const int vh = 32, n = 8 * vh * 9;
  Field U(2 * n);
  int missed[10] = {};
  const char *names[10] = {"an entry negated",  "a real part negated", "an entry conjugated", "a link negated",
                           "a direction negated", "the field negated",  "two entries exchanged", "parts exchanged",
                           "one bit",            "two bits of an entry"};
  for (int pass = 0; pass < 2; ++pass) {
    // random links, and the unit links of a free field
    for (int k = 0; k < n; ++k) {
      U[2 * k] = pass ? (k % 9 % 4 == 0) : 2 * uniform() - 1;
      U[2 * k + 1] = pass ? 0.0 : 2 * uniform() - 1;
    }
    const u64 h = hash(U);
    auto is = [&](int what, const Field &f) { missed[what] += hash(f) == h; };
    auto neg = [&](int from, int to, int step = 1) {
      Field f = U;
      for (int k = 2 * from; k < 2 * to; k += step) f[k] = -f[k];
      return f;
    };
    for (int k = 0; k < n; ++k) {
      is(0, neg(k, k + 1));
      is(1, neg(k, k + 1, 2));
      Field f = U;
      f[2 * k + 1] = -f[2 * k + 1];
      is(2, f);
      if (k % 9 == 0) is(3, neg(k, k + 9));
      f = U;
      std::swap(f[2 * k], f[2 * ((k + 1) % n)]);
      std::swap(f[2 * k + 1], f[2 * ((k + 1) % n) + 1]);
      if (f != U) is(6, f);
      f = U;
      std::swap(f[2 * k], f[2 * k + 1]);
      if (f != U) is(7, f);
    }
    for (int mu = 0; mu < 4; ++mu) is(4, neg(mu * 2 * vh * 9, (mu + 1) * 2 * vh * 9));
    is(5, neg(0, n));
    // single entries, bit by bit and in pairs
    for (int k = 0; k < n; k += 97) {
      const u64 a = bits(U[2 * k]), b = bits(U[2 * k + 1]), e = hash_mix(a, b, k);
      for (int i = 0; i < 128; ++i) {
        const u64 ai = i < 64 ? a ^ (1ull << i) : a, bi = i < 64 ? b : b ^ (1ull << (i - 64));
        missed[8] += hash_mix(ai, bi, k) == e;
        for (int j = 0; j < i; ++j) {
          const u64 aj = j < 64 ? ai ^ (1ull << j) : ai, bj = j < 64 ? bi : bi ^ (1ull << (j - 64));
          missed[9] += hash_mix(aj, bj, k) == e;
        }
      }
    }
  }
  int bad = 0;
  for (int k = 0; k < 10; ++k)
    if (missed[k]) bad = printf("%s: %d not seen\n", names[k], missed[k]);
  return bad ? 1 : 0;
}
"""


def test_changes_in_place_change_the_hash(tmp_path):
    host_code.run(tmp_path, PROGRAM, ["qcu_hash.h"])
