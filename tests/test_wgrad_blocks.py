"""How many blocks share a weight gradient's sites: no FP32 sum of a wave is longer than
with 1024 blocks per term at any size, and no block is without work where fewer do."""
import host_code

PROGRAM = r"""
using namespace qcu;
int main() {
  // half volumes up to 32^3x64, all of the small ones
  for (int vh = 8; vh <= 1 << 20; vh += vh < 40000 ? 1 : 997)
    for (int lds = 0; lds < 2; ++lds) {
      const int n = wgrad_blocks(vh, lds);
      const long long groups = (2LL * vh + 3) / 4, per = lds ? 8 : 4;  // groups of 4 sites, per step of a block
      auto longest = [&](long long blocks) { return (groups + per * blocks - 1) / (per * blocks); };
      if (n < 8 || n > kWgBlocks || n % 8 || longest(n) > longest(1024) || per * (n - 8) >= groups)
        return printf("half volume %d, lds %d: %d blocks\n", vh, lds, n), 1;
    }
  return 0;
}
"""


def test_no_sum_is_longer_than_with_all_blocks(tmp_path):
    host_code.run(tmp_path, PROGRAM, ["qcu_net.h"])
