"""Inputs still being written on the default stream when a call is made: the library
works on streams of its own and waits for that work first."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host, log, rel

pytestmark = pytest.mark.gpu

L, KAPPA, CSW = (8, 4, 4, 8), 0.124, 1.0


def _late(dst, src, a):
    """dst <- src behind some 50 ms of work on the default stream"""
    for _ in range(8):
        a = (a @ a).mul_(1e-4)
    dst.copy_(src)


@pytest.mark.parametrize("call", ["dslash", "dslash_fp32", "mat", "legacy", "load_gauge", "forward"])
def test_call_waits_for_pending_inputs(orc, call):
    """the same result as with the input in place (bitwise: the kernels are deterministic)"""
    from qcu_amd import pyqcu
    from qcu_amd.lattice import FP32, FP64, Lattice, LearnedPreconditioner
    vh = orc.vol(L) // 2
    U = dev(orc.gauge_random(L, 0.3, 400))
    lat = Lattice(L, KAPPA, CSW, -1)
    lat.load_gauge(U)
    net = LearnedPreconditioner(lat, (1, 4, 1), seed=1) if call == "forward" else None
    param = pyqcu.QcuParam()
    param.lattice_size = list(L)
    half, full = dev(orc.gauss((vh, 4, 3), 401)), dev(orc.gauss((2, vh, 4, 3), 402))
    src = U if call == "load_gauge" else full if call in ("mat", "forward") else half
    if call == "forward":
        src = src.reshape(1, 2, vh, 4, 3).contiguous()

    def run(x):
        if call == "dslash":
            return lat.dslash(x, 0, clover=True, prec=FP64)
        if call == "dslash_fp32":
            return lat.dslash(x, 0, clover=True, prec=FP32)
        if call == "mat":
            return lat.mat(x)
        if call == "legacy":
            out = torch.zeros_like(half)
            torch.cuda.synchronize()
            pyqcu.dslashQcu(out, x, U, param, 0)
            return out
        if call == "load_gauge":
            lat.load_gauge(x)
            return lat.dslash(half, 0, clover=True, prec=FP64)
        return net.forward(x)

    want = host(run(src))
    a = torch.randn(6144, 6144, device="cuda")
    x = torch.zeros_like(src)
    if call == "load_gauge":
        x.copy_(U.flip(0))
    torch.cuda.synchronize()
    if call != "legacy":  # (the wait inside run would hide the pending copy)
        _late(x, src, a)
        got = host(run(x))
    else:
        out = torch.zeros_like(half)
        torch.cuda.synchronize()
        _late(x, src, a)
        pyqcu.dslashQcu(out, x, U, param, 0)
        got = host(out)
    log(f"{call}: rel {rel(got, want):.1e}")
    assert np.array_equal(got, want)
