"""The number of iterations launched between two host checks does not change a
single system's iterates: a system that asks for a reliable update or has stopped
is skipped by every kernel until the host has looked."""
import numpy as np
import pytest

from gpu_util import dev, host, log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(4, 4, 4, 6), (16, 16, 10, 28)])
@pytest.mark.parametrize("prec,csw", [(0, 0.0), (0, 1.0), (1, 1.0), (2, 1.0)])
def test_solution_does_not_depend_on_the_chunk(orc, L, prec, csw):
    """equal bit for bit: the same kernels in the same order, (4,4,4,6) in five launches
    per iteration (FP64, FP32), the larger lattice in the general ones"""
    from qcu_amd.lattice import Lattice
    U = orc.gauge_random(L, 0.3, 1700)
    lat = Lattice(L, 0.124, csw, -1)
    lat.load_gauge(dev(U))
    b = dev(orc.gauss((2, orc.vol(L) // 2, 4, 3), 1701))
    ref, info = lat.solve(b, tol=1e-10, prec=prec, reliable_delta=0.05)
    ref = host(ref)
    assert info.converged
    for chunk in (2, 6, 8):
        for graph in (True, False):
            x, r = lat.solve(b, tol=1e-10, prec=prec, reliable_delta=0.05, chunk=chunk, use_graph=graph)
            assert r.iters == info.iters and r.reliable_updates == info.reliable_updates
            assert np.array_equal(host(x), ref), (chunk, graph)
    log(f"L={L} prec={prec}: {info.iters} iterations, {info.reliable_updates} updates at every chunk length")
    lat.close()


def test_scaled_sources_in_one_batch(orc):
    """systems whose residuals differ by 1e8, and one of zero source, keep their own pace"""
    from qcu_amd.lattice import Batch, Lattice
    L = (4, 6, 4, 6)
    U = orc.gauge_random(L, 0.3, 1710)
    lat = Lattice(L, 0.124, 1.0, -1)
    lat.load_gauge(dev(U))
    bs = [s * orc.gauss((2, orc.vol(L) // 2, 4, 3), 1711 + k) for k, s in enumerate((1e-8, 1.0, 0.0, 1e8))]
    for prec in (0, 1, 2):
        batch = Batch([lat], [4])
        xs, infos = batch.solve([dev(b) for b in bs], tol=1e-10, prec=prec, reliable_delta=0.05)
        for x, b, r in zip(xs, bs, infos):
            if not b.any():
                assert not host(x).any()
                continue
            assert r.converged and orc.true_residual(host(x), b, U, L, 0.124, 1.0, -1) <= 1e-10
        batch.close()
    lat.close()
