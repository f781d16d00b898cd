"""The hop kernels against each other and the oracle: eight waves per 64 sites
(small lattices, no shape pinned) against one thread per site (a pinned shape),
and the FP64 operators that read and write the caller's fields directly."""
import ctypes as C

import numpy as np
import pytest
import torch

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

KAPPA, CSW = 0.124, 1.0


def _lattice(orc, L, csw, seed):
    from qcu_amd.lattice import Lattice
    U = orc.gauge_random(L, 0.3, seed)
    lat = Lattice(L, KAPPA, csw, -1)
    lat.load_gauge(dev(U))
    return lat, U


# half volumes 8 and 360 (partial blocks), 64 (one block), 32 768 (the largest of
# the split kernel) and 33 280 (the first beyond it); shapes used nowhere else, so
# that no other test has pinned a launch shape for them
@pytest.mark.parametrize("L", [(2, 2, 2, 2), (2, 10, 6, 6), (2, 4, 4, 4), (16, 16, 8, 32), (16, 16, 10, 26)])
@pytest.mark.parametrize("csw", [0.0, CSW])
def test_split_kernel_equals_one_thread_per_site(orc, L, csw):
    """both sum every component in the same order: equal bit for bit"""
    lat, U = _lattice(orc, L, csw, 1300)
    psi = orc.gauss((orc.vol(L) // 2, 4, 3), 1301)
    x = dev(psi)
    auto = {(p, c, q): host(lat.dslash(x, parity=q, clover=c, prec=p)) for p in (0, 1, 2)
            for c in ((False, True) if csw else (False,)) for q in (0, 1)}
    full = dev(orc.gauss((2, orc.vol(L) // 2, 4, 3), 1302))
    mat = host(lat.mat(full))
    err = rel(auto[(0, csw != 0, 1)], orc.clover_dslash(psi, U, L, 1, KAPPA * csw, -1) if csw
              else orc.hop(psi, U, L, 1, -1))
    log(f"L={L} csw={csw}: hop {err:.1e} from the oracle")
    assert err < 1e-12
    for p in (0, 1, 2):
        lat.set_launch_shape(p, 128, 1, 2)
    for (p, c, q), ref in auto.items():
        assert np.array_equal(host(lat.dslash(x, parity=q, clover=c, prec=p)), ref), (p, c, q)
    assert np.array_equal(host(lat.mat(full)), mat)
    lat.close()


@pytest.mark.parametrize("L", [(4, 2, 6, 4), (16, 16, 10, 28)])
def test_output_over_input(orc, L):
    """calls whose output is, or partly overlaps, their input"""
    lat, U = _lattice(orc, L, CSW, 1310)
    n = orc.vol(L) // 2 * 12
    psi = dev(orc.gauss((2, n), 1311))
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    lib = lat._lib
    for name, args in (("qcuDslash", (1, 1, 0)), ("qcuDslash", (0, 0, 1)), ("qcuDslashNoAlloc", (1, 1, 0))):
        ref = torch.empty(n, dtype=torch.complex128, device="cuda")
        assert getattr(lib, name)(lat.h, p(ref), p(psi[0]), *args) == 0
        for shift in (0, 7):
            buf = torch.zeros(n + 16, dtype=torch.complex128, device="cuda")
            buf[:n] = psi[0]
            torch.cuda.synchronize()
            assert getattr(lib, name)(lat.h, p(buf[shift:]), p(buf), *args) == 0
            assert torch.equal(buf[shift:shift + n], ref), (name, args, shift)
    ref = lat.mat(psi.reshape(2, -1))
    buf = psi.clone()
    torch.cuda.synchronize()
    assert lib.qcuMatFull(lat.h, p(buf), p(buf)) == 0
    assert torch.equal(buf.reshape(-1), ref.reshape(-1))
    lat.close()
