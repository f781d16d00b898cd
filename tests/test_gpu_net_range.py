"""The preconditioner's composed steps over the range of its weights: layers whose
outputs are all within FP32 give the same network whatever the size of the weights."""
import numpy as np
import pytest

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

TOL = 2e-5  # FP32 network against the oracle, as in the other network tests
L, CHAN = (8, 4, 4, 8), (1, 8, 8, 8, 1)


def _network(orc, seed):
    from qcu_amd.lattice import Lattice, LearnedPreconditioner
    U = orc.gauge_random(L, 0.3, seed)
    lat = Lattice(L, 0.124, 0.0, -1)
    lat.load_gauge(dev(U))
    net = LearnedPreconditioner(lat, CHAN, seed=seed)
    rng = np.random.default_rng(seed)
    W = (0.2 * (rng.standard_normal(net.nweights) + 1j * rng.standard_normal(net.nweights))).astype(np.complex64)
    xo = orc.gauss((orc.vol(L) // 2, 4, 3), seed + 1)
    return U, lat, net, W.astype(np.complex128), xo


def _reference(orc, U, W, xo):
    full = np.zeros((1, 2) + xo.shape, complex)
    full[0, 1] = xo
    return orc.net_forward(full, W, CHAN, U, L, -1)[0].reshape(2, -1)[1]


@pytest.mark.parametrize("a,b", [(2.0 ** 33, 2.0 ** -100), (2.0 ** -33, 2.0 ** 83), (2.0 ** 45, 2.0 ** -120),
                                 (2.0 ** -40, 2.0 ** 100)])
def test_all_layers_scaled(orc, a, b):
    """weights times a, input times b: the output times a^4 b, by powers of two"""
    U, lat, net, W, xo = _network(orc, 720)
    net.set_weights(a * W)
    got = host(net.apply_odd(dev(b * xo))).ravel() / a ** 4 / b
    e = rel(got, _reference(orc, U, W, xo))
    log(f"a={a:g} b={b:g}: {e:.1e}")
    assert e < TOL
    net.close()
    lat.close()


@pytest.mark.parametrize("f", [2.0 ** -60, 2.0 ** -100, 2.0 ** -120])
@pytest.mark.parametrize("layer", [1, 3])
def test_hop_terms_far_below_the_site_term(orc, f, layer):
    """one layer's hop weights times f"""
    U, lat, net, W, xo = _network(orc, 730)
    n = [9 * CHAN[k] * CHAN[k + 1] * 16 for k in range(4)]
    at = sum(n[:layer])
    W[at:at + n[layer] * 8 // 9] *= f  # terms 0..7 are the hops
    net.set_weights(W)
    e = rel(host(net.apply_odd(dev(xo))).ravel(), _reference(orc, U, W, xo))
    log(f"layer {layer}: hop weights times {f:g}: {e:.1e}")
    assert e < TOL
    net.close()
    lat.close()
