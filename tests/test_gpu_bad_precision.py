"""A precision that does not exist is refused by every call that looks up a launch
shape for it, and leaves the handles as they were."""
import pytest

from gpu_util import dev, host, log

pytestmark = pytest.mark.gpu

ERR_ARG = 1


def test_bad_precision_is_refused(orc):
    from qcu_amd._lib import QcuError
    from qcu_amd.lattice import Batch, Lattice
    L, kappa = (4, 4, 4, 6), 0.124
    U = orc.gauge_random(L, 0.3, 330)
    lat = Lattice(L, kappa, 0.0, -1)
    lat.load_gauge(dev(U))
    batch = Batch([lat], [2])
    bs = [orc.gauss((2, orc.vol(L) // 2, 4, 3), 331 + k) for k in range(2)]

    def solves():
        x, r = lat.solve(dev(bs[0]), tol=1e-10)
        xs, rs = batch.solve([dev(b) for b in bs], tol=1e-10)
        assert r.converged and all(q.converged for q in rs)
        worst = max(orc.true_residual(host(y), b, U, L, kappa, 0.0, -1) for y, b in zip([x] + xs, bs[:1] + bs))
        assert worst <= 1e-10
        return worst

    solves()
    shapes = [lat.launch_shape(p) for p in range(3)]
    for prec in (3, -1, 4, 1000, -2 ** 31, 2 ** 31 - 1):
        for name, call in (("launch_shape", lambda: lat.launch_shape(prec)),
                           ("bench_hop", lambda: lat.bench_hop(prec, iters=1)),
                           ("batch bench_hop", lambda: batch.bench_hop(prec, iters=1)),
                           ("tune", lambda: lat.tune(prec)),
                           ("set_launch_shape", lambda: lat.set_launch_shape(prec, 64, 1, 0))):
            with pytest.raises(QcuError) as e:
                call()
            assert e.value.code == ERR_ARG, (name, prec)
    assert [lat.launch_shape(p) for p in range(3)] == shapes
    log(f"after the refused calls: worst residual {solves():.1e}")
    batch.close()
    lat.close()
