"""Solves while another thread tunes lattices of the same size: the launch shapes
change between any two of a solve's launches, and every solve still converges."""
import threading

import pytest

from gpu_util import dev, host, log

pytestmark = pytest.mark.gpu

KAPPA = 0.124


def _lattice(L, U, csw):
    from qcu_amd.lattice import Lattice
    lat = Lattice(L, KAPPA, csw, -1)
    lat.load_gauge(dev(U))
    return lat


def _beside(work, other):
    """runs other() over and over in a second thread while work() runs"""
    stop, failed = threading.Event(), []

    def loop():
        try:
            while not stop.is_set():
                other()
        except Exception as e:  # noqa: BLE001
            failed.append(e)

    t = threading.Thread(target=loop)
    t.start()
    try:
        work()
    finally:
        stop.set()
        t.join()
    assert not failed, failed


@pytest.mark.parametrize("csw", [0.0, 1.0])
def test_solves_beside_tuning(orc, csw):
    L = (4, 4, 6, 10)  # used nowhere else: tuning leaves its shapes behind
    U = orc.gauge_random(L, 0.3, 1800)
    lat, same = _lattice(L, U, csw), _lattice(L, U, csw)
    b = orc.gauss((2, orc.vol(L) // 2, 4, 3), 1801)
    bd = dev(b)

    def other():
        for prec in (0, 1):
            same.set_launch_shape(prec, 128, 1, 0)
            same.tune(prec)

    def work():
        worst = 0.0
        for k in range(60):
            x, r = lat.solve(bd, tol=1e-10, prec=k % 2, reliable_delta=0.1, use_graph=k % 3 != 0)
            tr = orc.true_residual(host(x), b, U, L, KAPPA, csw, -1)
            worst = max(worst, tr)
            assert r.converged and tr <= 1e-10, k
        log(f"csw={csw}: worst residual of 60 solves beside tuning {worst:.1e}")

    _beside(work, other)
    lat.close()
    same.close()


def test_network_and_lattice_threads_beside_tuning(orc):
    """a network's handle in one thread, its lattice's in another, shapes changing"""
    import numpy as np
    from qcu_amd.lattice import FP32, FP64, LearnedPreconditioner
    L, csw = (4, 6, 4, 10), 1.0
    U = orc.gauge_random(L, 0.3, 1810)
    lat, same = _lattice(L, U, csw), _lattice(L, U, csw)
    net = LearnedPreconditioner(lat, (1, 4, 1), seed=1811)
    src = dev(orc.gauss((orc.vol(L) // 2, 4, 3), 1812))
    psi = orc.gauss((orc.vol(L) // 2, 4, 3), 1813)
    pd, ref = dev(psi), orc.clover_dslash(psi, U, L, 0, KAPPA * csw, -1)
    want = net.loss_grad(src)

    def other():
        for prec in (FP64, FP32):
            for shape in ((64, 1, 0), (256, 0, 2), (128, 1, 1)):
                same.set_launch_shape(prec, *shape)
        loss, grad = net.loss_grad(src)
        assert abs(loss - want[0]) <= 1e-6 * abs(want[0])
        assert np.linalg.norm(grad - want[1]) <= 1e-4 * np.linalg.norm(want[1])

    def work():
        for k in range(200):
            out = host(lat.dslash(pd, 0, clover=True, prec=k % 2))
            assert np.linalg.norm(out - ref) <= (2e-6 if k % 2 else 1e-12) * np.linalg.norm(ref), k

    _beside(work, other)
    net.close()
    lat.close()
    same.close()
