"""A reference-named hop whose gauge changed to one without a clover inverse reports
the error and leaves its output as it was."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

ERR_STATE = 7


# half volumes 48 (eight waves per 64 sites) and 33 280 (one thread per site)
@pytest.mark.parametrize("L", [(4, 4, 2, 6), (16, 16, 10, 26)])
def test_output_is_untouched(orc, L):
    from qcu_amd import pyqcu
    from qcu_amd._lib import QcuError
    vh = orc.vol(L) // 2
    U = orc.gauge_random(L, 0.05, 85)
    psi = orc.gauss((vh, 4, 3), 86)
    param = pyqcu.QcuParam()
    param.lattice_size = list(L)
    buf, inp = dev(U), dev(psi)
    mark = dev(orc.gauss((vh, 4, 3), 87))
    out = mark.clone()
    torch.cuda.synchronize()
    pyqcu.dslashCloverQcu(out, inp, buf, param, 1)
    want = out.clone()
    assert rel(host(out), orc.clover_dslash(psi, U, L, 1, 1.0, 1)) < 1e-12
    bad = U.copy()
    bad[2, 1, 5, 1, 1] = np.nan
    for what in ("known pointer", "after the failure"):
        buf.copy_(dev(bad))
        out.copy_(mark)
        torch.cuda.synchronize()
        with pytest.raises(QcuError) as e:
            pyqcu.dslashCloverQcu(out, inp, buf, param, 1)
        assert e.value.code == ERR_STATE
        assert torch.equal(out, mark), what
    # and with the good field back, the same result as at first
    buf.copy_(dev(U))
    torch.cuda.synchronize()
    for _ in range(2):
        out.copy_(mark)
        pyqcu.dslashCloverQcu(out, inp, buf, param, 1)
        assert torch.equal(out, want)
    log(f"L={L}: output untouched by the failed reload")
