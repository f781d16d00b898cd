"""Loading a gauge field at lattice sizes that end inside a block: links and the
packed clover term (and its inverse) in every precision, against the oracle."""
import numpy as np
import pytest

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

# half volumes 8 (less than one block), 96 (one and a half), 360 (five and five
# eighths) and 64 (exactly one); extents of 2 wrap onto one neighbour
SIZES = [(2, 2, 2, 2), (4, 2, 4, 6), (2, 10, 6, 6), (4, 4, 2, 4)]


@pytest.mark.parametrize("L", SIZES)
def test_links_and_clover_in_every_precision(orc, L):
    """tolerances as in the hop tests: FP64 1e-12, FP32 2e-6, FP16 5e-3 of the result"""
    from qcu_amd.lattice import Lattice
    kappa, csw = 0.124, 1.0
    U = orc.gauge_random(L, 0.3, 900 + L[1])
    psi = orc.gauss((2, orc.vol(L) // 2, 4, 3), 901)
    lat = Lattice(L, kappa, csw, -1)
    lat.load_gauge(dev(U))
    for prec, tol in ((0, 1e-12), (1, 2e-6), (2, 5e-3)):
        for parity in (0, 1):
            inp = np.ascontiguousarray(psi[1 - parity])
            out = host(lat.dslash(dev(inp), parity, clover=True, prec=prec))
            err = rel(out, orc.clover_dslash(inp, U, L, parity, kappa * csw, -1))
            log(f"L={L} prec={prec} parity={parity}: clover hop {err:.2e}")
            assert err < tol
    # the clover term itself
    err = rel(host(lat.mat(dev(psi))), orc.mat_full(psi, U, L, kappa, csw, -1))
    log(f"L={L}: full operator {err:.2e}")
    assert err < 1e-13


def test_reload_replaces_every_precision(orc):
    """a second load on the same handle replaces the links and the clover term"""
    from qcu_amd.lattice import Lattice
    L, kappa, csw = (4, 6, 4, 6), 0.124, 1.0
    psi = orc.gauss((orc.vol(L) // 2, 4, 3), 911)
    lat = Lattice(L, kappa, csw, -1)
    for seed in (912, 913):
        U = orc.gauge_random(L, 0.3, seed)
        lat.load_gauge(dev(U))
        for prec, tol in ((0, 1e-12), (1, 2e-6), (2, 5e-3)):
            err = rel(host(lat.dslash(dev(psi), 1, clover=True, prec=prec)),
                      orc.clover_dslash(psi, U, L, 1, kappa * csw, -1))
            assert err < tol, (seed, prec, err)
