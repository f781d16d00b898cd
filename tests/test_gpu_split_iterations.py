"""BiCGSTAB iterations in five launches (small batches, FP64 and FP32) against the
general ones (a pinned launch shape) and the oracle: partial blocks, several
right-hand sides, systems that stop at different iterations, odd chunks."""
import numpy as np
import pytest

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

KAPPA = 0.124


def _systems(orc, csw):
    """half volumes 48, 360 and 512 with 2, 5 and 1 right-hand sides; the sources differ
    in size by 1e12, so that their systems reach a given absolute target apart"""
    from qcu_amd.lattice import Lattice
    shapes, nrhs = [(4, 2, 2, 6), (2, 10, 6, 6), (4, 4, 8, 8)], [2, 5, 1]
    lats, Us, bs = [], [], []
    for k, (L, n) in enumerate(zip(shapes, nrhs)):
        U = orc.gauge_random(L, 0.3, 1600 + k)
        lat = Lattice(L, KAPPA, csw, -1)
        lat.load_gauge(dev(U))
        lats.append(lat)
        Us.append(U)
        bs += [10.0 ** (6 * (r % 3) - 6) * orc.gauss((2, orc.vol(L) // 2, 4, 3), 1610 + 10 * k + r) for r in range(n)]
    return shapes, nrhs, lats, Us, bs


@pytest.mark.parametrize("csw", [0.0, 1.0])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("chunk", [2, 8, 3])
def test_batch_of_small_lattices(orc, csw, prec, chunk):
    from qcu_amd.lattice import Batch
    shapes, nrhs, lats, Us, bs = _systems(orc, csw)
    batch = Batch(lats, nrhs)
    run = lambda **kw: batch.solve([dev(b) for b in bs], tol=1e-10, prec=prec, reliable_delta=0.1,  # noqa: E731
                                   chunk=chunk, **kw)
    xs, infos = run()
    ys, _ = run(use_graph=False)
    at = [k for k, n in enumerate(nrhs) for _ in range(n)]
    worst = max(orc.true_residual(host(x), b, Us[k], shapes[k], KAPPA, csw, -1) for x, b, k in zip(xs, bs, at))
    log(f"csw={csw} prec={prec} chunk={chunk}: iterations {[r.iters for r in infos]}, worst residual {worst:.1e}")
    assert all(r.converged for r in infos) and worst <= 1e-10
    # graph and eager runs are the same bit for bit
    assert all(np.array_equal(host(x), host(y)) for x, y in zip(xs, ys))
    # the general iterations: FP64 rounding apart, the same recurrence
    batch.set_launch_shape(prec, 128, 1, 0)
    zs, others = run()
    assert all(r.converged for r in others)
    if prec == 0:
        assert [r.iters for r in infos] == [r.iters for r in others]
        # two solutions of residual 1e-10 from one recurrence
        assert max(rel(host(x), host(z)) for x, z in zip(xs, zs)) < 1e-9
    batch.close()


def test_max_iter_not_a_multiple_of_the_chunk(orc):
    """an odd remainder of iterations runs the general kernels on the same vectors"""
    from qcu_amd.lattice import Lattice
    L = (4, 4, 4, 6)
    U = orc.gauge_random(L, 0.3, 1650)
    lat = Lattice(L, KAPPA, 0.0, -1)
    lat.load_gauge(dev(U))
    b = orc.gauss((2, orc.vol(L) // 2, 4, 3), 1651)
    ref = None
    for max_iter in (7, 8, 11):
        x, r = lat.solve(dev(b), tol=1e-12, prec=0, max_iter=max_iter, chunk=4)
        res = orc.true_residual(host(x), b, U, L, KAPPA, 0.0, -1)
        log(f"max_iter {max_iter}: {r.iters} iterations, residual {res:.1e}")
        assert r.iters <= max_iter
        assert ref is None or res < ref  # more iterations from the same start
        ref = res
    lat.close()
