"""The preconditioner's composed steps: the second layer on its odd sites and the
third and last layers as one (1-8-8-8-1), and the second layer on both parities
(deeper networks), at half volumes around the 32-site chunks and with the layers'
weights far apart in size."""
import numpy as np
import pytest

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

TOL = 2e-5  # FP32 network against the oracle, as in the other network tests


def _check(orc, L, chan, tb, seed, a=1.0, scale=1.0):
    from qcu_amd.lattice import Lattice, LearnedPreconditioner
    U = orc.gauge_random(L, 0.3, seed)
    lat = Lattice(L, 0.124, 0.0, tb)
    lat.load_gauge(dev(U))
    net = LearnedPreconditioner(lat, chan, seed=seed)
    rng = np.random.default_rng(seed)
    W = (0.2 * (rng.standard_normal(net.nweights) + 1j * rng.standard_normal(net.nweights))).astype(np.complex64)
    W = W.astype(np.complex128)
    Ws = W.copy()
    if a != 1.0:  # the third layer times a, the last over a: the same network
        n = [9 * chan[k] * chan[k + 1] * 16 for k in range(len(chan) - 1)]
        Ws[n[0] + n[1]:n[0] + n[1] + n[2]] *= a
        Ws[-n[-1]:] /= a
    net.set_weights(Ws)
    xo = orc.gauss((orc.vol(L) // 2, 4, 3), seed + 1)
    full = np.zeros((1, 2) + xo.shape, complex)
    full[0, 1] = xo
    ref, _ = orc.net_forward(full, W, chan, U, L, tb)
    got = host(net.apply_odd(dev(xo * scale))).ravel() / scale
    e = rel(got, ref.reshape(2, -1)[1])
    log(f"L={L} chan={chan} tb={tb} a={a:g} scale={scale:g}: {e:.1e}")
    assert e < TOL
    net.close()
    lat.close()


# half volumes 8, 48, 96 and 360: less than one chunk, one and a half, three, eleven and a quarter
@pytest.mark.parametrize("tb", [1, -1])
@pytest.mark.parametrize("L", [(2, 2, 2, 2), (4, 2, 2, 6), (4, 2, 4, 6), (2, 10, 6, 6)])
@pytest.mark.parametrize("chan", [(1, 8, 8, 8, 1), (1, 8, 8, 8, 8, 1), (1, 8, 8, 4, 1)])
def test_apply_odd_sizes(orc, chan, L, tb):
    _check(orc, L, chan, tb, 700 + L[1])


@pytest.mark.parametrize("a,scale", [(1e-12, 1.0), (1e12, 1.0), (1e6, 1e-15)])
def test_apply_odd_last_layers_scaled(orc, a, scale):
    _check(orc, (8, 4, 4, 8), (1, 8, 8, 8, 1), -1, 710, a, scale)
