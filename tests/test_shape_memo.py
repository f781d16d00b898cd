"""The remembered launch shapes on the host: every shape comes back as it was put, for
its generation only, and threads never see half of one."""
import host_code

PROGRAM = r"""
#include <thread>
using namespace qcu;
int main() {
  ShapeMemo m;
  LaunchCfg c;
  for (int prec = 0; prec < 3; ++prec)
    if (m.get(prec, 1, &c)) return printf("a shape before the first\n"), 1;
  unsigned long long gen = 0;
  for (int block = 64; block <= 256; block += 64)
    for (int remap = 0; remap < 2; ++remap)
      for (int group = 0; group < 3; ++group)
        for (int automatic = 0; automatic < 2; ++automatic)
          for (int prec = 0; prec < 3; ++prec) {
            LaunchCfg p;
            p.block = block;
            p.remap = remap;
            p.group = group;
            p.automatic = automatic;
            m.put(prec, ++gen, p);
            if (m.get(prec, gen + 1, &c) || !m.get(prec, gen, &c) || c.block != block || c.remap != remap ||
                c.group != group || c.automatic != (bool)automatic)
              return printf("%d %d %d %d\n", block, remap, group, automatic), 1;
          }
  // two threads look shapes up while the generation moves: block and group belong together
  std::atomic<unsigned long long> now{1};
  std::atomic<int> bad{0};
  m.clear();
  auto look = [&]() {
    for (int k = 0; k < 2000000; ++k) {
      const unsigned long long g = now.load();
      LaunchCfg p;
      if (!m.get(0, g, &p)) {
        p.block = g & 1 ? 64 : 256;
        p.group = g & 1 ? 0 : 2;
        m.put(0, g, p);
      }
      if (p.block != (g & 1 ? 64 : 256) || p.group != (g & 1 ? 0 : 2)) bad = 1;
      if (k % 64 == 0) ++now;
    }
  };
  std::thread a(look), b(look);
  a.join();
  b.join();
  return bad;
}
"""


def test_shapes_come_back_whole(tmp_path):
    host_code.run(tmp_path, PROGRAM, ["qcu_internal.h"])
