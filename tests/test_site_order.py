"""The hop kernels' site order on the host: every site once, and a valid site for the
lanes past the last one, whatever the slabs."""
import host_code

PROGRAM = r"""
using namespace qcu;
int main() {
  // slabs that divide Lz, slabs with a thinner last one, half volumes that do and do
  // not fill blocks of 256
  const int shapes[][4] = {{18, 50, 24, 2}, {18, 54, 24, 2}, {32, 32, 22, 4}, {4, 2, 6, 6}, {2, 2, 2, 2}, {8, 8, 8, 8}};
  for (auto &L : shapes) {
    Geom g{};
    g.lxh = L[0] / 2;
    g.ly = L[1];
    g.lz = L[2];
    g.lt = L[3];
    g.vh = g.lxh * g.ly * g.lz * g.lt;
    const int lanes = (g.vh + 255) / 256 * 256;
    for (int zslab = 0; zslab < g.lz; ++zslab)
      for (int parity = 0; parity < 2; ++parity) {
        std::vector<int> seen(g.vh, 0);
        for (int k = 0; k < lanes; ++k) {
          int i = -1;
          const Site s = ordered_site(g, zslab, k, parity, i);
          const Site d = decode(g, i, parity);
          if (i < 0 || i >= g.vh || d.xh != s.xh || d.y != s.y || d.z != s.z || d.t != s.t || d.xodd != s.xodd)
            return printf("%dx%dx%dx%d slabs of %d: site %d at k = %d\n", L[0], L[1], L[2], L[3], zslab, i, k), 1;
          if (k < g.vh && seen[i]++) return printf("site %d twice\n", i), 1;
        }
      }
  }
  return 0;
}
"""


def test_every_site_once_and_lanes_past_the_end(tmp_path):
    host_code.run(tmp_path, PROGRAM, ["qcu_common.h"])
