"""Weight gradients on lattices that take different numbers of blocks per term
(8, 88 and 128), and after the weights change between two calls (the transposed
operands are packed once per weight version), against the oracle."""
import numpy as np
import pytest

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

CHAN = (1, 8, 8, 8, 1)


@pytest.mark.parametrize("L", [(4, 2, 2, 2), (8, 8, 8, 6), (16, 16, 16, 16)])
def test_backward_across_block_counts(orc, L):
    """bounds of the network tests: weight gradient 1e-4, input gradient 2e-5"""
    from qcu_amd.lattice import Lattice, LearnedPreconditioner
    U = orc.gauge_random(L, 0.3, 1500)
    lat = Lattice(L, 0.124, 0.0, -1)
    lat.load_gauge(dev(U))
    net = LearnedPreconditioner(lat, CHAN, seed=3, init_scale=0.3)
    x = orc.gauss((1, 2, orc.vol(L) // 2, 4, 3), 1501)
    g = orc.gauss((1, 2, orc.vol(L) // 2, 4, 3), 1502)
    for scale in (1.0, -0.5):
        W = scale * net.get_weights()
        net.set_weights(W)
        _, acts = orc.net_forward(x, W, CHAN, U, L, -1)
        gin_ref, gw_ref = orc.net_backward(g, W, CHAN, U, L, acts, -1)
        gw, gin = net.backward(dev(x), dev(g))
        e = rel(gw, gw_ref), rel(host(gin).ravel(), np.asarray(gin_ref).ravel())
        log(f"L={L} scale {scale}: weight gradient {e[0]:.1e}, input gradient {e[1]:.1e}")
        assert e[0] < 1e-4 and e[1] < 2e-5
    net.close()
    lat.close()
