"""The reference-named hops on a resident gauge: the operator runs ahead of the
check of the field's contents, so every call has to give what a first call gives
- after a change of the first or the last link only, in place, and with the
output laid over the gauge itself."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

# 8 * half volume links in blocks of 256: less than one block, remainders, exactly one
SIZES = [(2, 2, 2, 2), (4, 2, 4, 6), (2, 10, 6, 6), (4, 4, 2, 2)]


@pytest.mark.parametrize("L", SIZES)
def test_resident_gauge(orc, L):
    """tolerance 1e-12 of the FP64 Wilson hop, as in the hop tests"""
    from qcu_amd import pyqcu
    vh = orc.vol(L) // 2
    U, V = orc.gauge_random(L, 0.3, 70), orc.gauge_random(L, 0.3, 71)
    psi = orc.gauss((vh, 4, 3), 72)
    param = pyqcu.QcuParam()
    param.lattice_size = list(L)
    buf = dev(U).reshape(-1).clone()
    inp, out = dev(psi), torch.zeros_like(dev(psi))

    def check(what, res, links, x=psi):
        err = rel(host(res), orc.hop(x, links.reshape(U.shape), L, 0, 1))
        log(f"L={L} {what}: {err:.1e}")
        assert err < 1e-12

    flat = np.ascontiguousarray(U).reshape(-1).copy()
    for what, sel in (("load", None), ("resident", None), ("first link", slice(0, 9)), ("last link", slice(-9, None))):
        if sel is not None:
            flat[sel] = V.reshape(-1)[sel]
            buf.copy_(dev(flat))
        out.zero_()
        pyqcu.dslashQcu(out, inp, buf, param, 0)
        check(what, out, flat)
    pyqcu.dslashQcu(inp, inp, buf, param, 0)
    check("in place", inp, flat)
    over = buf[:psi.size].view(psi.shape)
    psi2 = orc.gauss((vh, 4, 3), 73)
    pyqcu.dslashQcu(over, dev(psi2), buf, param, 0)
    check("over the gauge", over, flat, psi2)
    buf.copy_(dev(flat))
    pyqcu.dslashQcu(out, dev(psi2), buf, param, 0)
    check("restored", out, flat, psi2)
