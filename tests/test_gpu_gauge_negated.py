"""The reference-named hops after entries of the resident gauge changed their sign in
place: the call has to see it.  The links stay in SU(3) (two rows or two columns of a
link change sign together)."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("clover", [False, True])
def test_negated_links_are_seen(orc, clover):
    """tolerance 1e-12 of the FP64 hops, as in the hop tests"""
    from qcu_amd import pyqcu
    L = (4, 4, 2, 6)
    vh = orc.vol(L) // 2
    U = orc.gauge_random(L, 0.3, 75)
    psi = orc.gauss((vh, 4, 3), 76)
    param = pyqcu.QcuParam()
    param.lattice_size = list(L)
    buf, inp, out = dev(U), dev(psi), torch.zeros_like(dev(psi))
    links = U.reshape(4, 2, L[3], -1, 3, 3).copy()
    changes = {"nothing": np.s_[:0], "rows, last time slice": np.s_[3, :, -1, :, :2],
               "rows of a link": np.s_[1, 0, 2, 3, 1:], "columns of a link": np.s_[0, 1, 1, 2, :, :2],
               "columns, a direction": np.s_[2, ..., 1:]}
    for what, sel in changes.items():
        links[sel] *= -1
        buf.copy_(dev(links.reshape(U.shape)))
        (pyqcu.dslashCloverQcu if clover else pyqcu.dslashQcu)(out, inp, buf, param, 1)
        ref = links.reshape(U.shape)
        ref = orc.clover_dslash(psi, ref, L, 1, 1.0, 1) if clover else orc.hop(psi, ref, L, 1, 1)
        err = rel(host(out), ref)
        log(f"clover={clover} {what}: {err:.1e}")
        assert err < 1e-12
