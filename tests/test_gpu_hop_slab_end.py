"""Slabs that divide Lz exactly with a last block of 64 sites that is not full, in the
kernels with eight waves per 64 sites, against the oracle."""
import numpy as np
import pytest

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

L, KAPPA = (18, 50, 24, 2), 0.124  # FP64: slabs of 8 planes; 21 600 half sites, 337.5 blocks


@pytest.mark.parametrize("csw", [0.0, 1.0])
def test_exact_slabs(orc, csw):
    """FP64 hops 1e-12, the full operator 1e-13, the solve's true residual 1e-10"""
    from qcu_amd.lattice import Lattice
    U = orc.gauge_random(L, 0.3, 1430)
    lat = Lattice(L, KAPPA, csw, -1)
    lat.load_gauge(dev(U))
    psi = orc.gauss((2, orc.vol(L) // 2, 4, 3), 1431)
    for parity in (0, 1):
        inp = np.ascontiguousarray(psi[1 - parity])
        out = host(lat.dslash(dev(inp), parity, clover=csw != 0))
        ref = orc.clover_dslash(inp, U, L, parity, KAPPA * csw, -1) if csw else orc.hop(inp, U, L, parity, -1)
        log(f"csw={csw} parity={parity}: {rel(out, ref):.1e}")
        assert rel(out, ref) < 1e-12
    assert rel(host(lat.mat(dev(psi))), orc.mat_full(psi, U, L, KAPPA, csw, -1)) < 1e-13
    x, res = lat.solve(dev(psi), tol=1e-10)
    tr = orc.true_residual(host(x), psi, U, L, KAPPA, csw, -1)
    log(f"csw={csw}: {res.iters} iterations, true residual {tr:.1e}")
    assert res.converged and tr <= 1e-10
    lat.close()
