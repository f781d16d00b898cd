"""The hop's site order in z slabs (lattices whose time slice outgrows an XCD's
L2), with a thinner last slab, against the oracle, and batches whose segments
are found through the block table."""
import numpy as np
import pytest

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

KAPPA = 0.124


# FP64 slices of 2.2 and 2.4 MB: slabs of 8, 8, 6 and of 9, 9, 6 planes
@pytest.mark.parametrize("L", [(32, 32, 22, 4), (18, 54, 24, 2)])
@pytest.mark.parametrize("csw", [0.0, 1.0])
def test_slabs_match_oracle(orc, L, csw):
    """FP64 1e-12, as every FP64 hop; the full operator 1e-13"""
    from qcu_amd.lattice import Lattice
    U = orc.gauge_random(L, 0.3, 1400)
    lat = Lattice(L, KAPPA, csw, -1)
    lat.load_gauge(dev(U))
    psi = orc.gauss((2, orc.vol(L) // 2, 4, 3), 1401)
    for parity in (0, 1):
        inp = np.ascontiguousarray(psi[1 - parity])
        out = host(lat.dslash(dev(inp), parity, clover=csw != 0))
        ref = orc.clover_dslash(inp, U, L, parity, KAPPA * csw, -1) if csw else orc.hop(inp, U, L, parity, -1)
        log(f"L={L} csw={csw} parity={parity}: {rel(out, ref):.1e}")
        assert rel(out, ref) < 1e-12
    assert rel(host(lat.mat(dev(psi))), orc.mat_full(psi, U, L, KAPPA, csw, -1)) < 1e-13
    lat.close()


@pytest.mark.parametrize("prec", [0, 1, 2])
def test_batch_slabs_and_segments(orc, prec):
    """12 right-hand sides in slabs (16x16x16x4 in FP64: planes of 295 KB, slabs of
    3 and a last one of 1; FP32: 6, 6, 4) next to small lattices: every system's
    oracle residual meets the tolerance"""
    from qcu_amd.lattice import Batch, Lattice
    shapes, nrhs = [(4, 4, 4, 4), (16, 16, 16, 4), (6, 4, 2, 8), (10, 6, 4, 4)], [1, 12, 3, 2]
    lats, Us, bs = [], [], []
    for k, (L, n) in enumerate(zip(shapes, nrhs)):
        U = orc.gauge_random(L, 0.3, 1410 + k)
        lat = Lattice(L, KAPPA, 1.0, -1)
        lat.load_gauge(dev(U))
        lats.append(lat)
        Us.append(U)
        bs += [orc.gauss((2, orc.vol(L) // 2, 4, 3), 1420 + 20 * k + r) for r in range(n)]
    batch = Batch(lats, nrhs)
    xs, infos = batch.solve([dev(b) for b in bs], tol=1e-10, prec=prec, reliable_delta=0.1)
    at = [k for k, n in enumerate(nrhs) for _ in range(n)]
    worst = max(orc.true_residual(host(x), b, Us[k], shapes[k], KAPPA, 1.0, -1) for x, b, k in zip(xs, bs, at))
    log(f"batch prec={prec}: worst oracle residual {worst:.1e}")
    assert all(r.converged for r in infos) and worst <= 1e-10
    batch.close()
