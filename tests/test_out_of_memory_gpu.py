"""A call that is refused for want of device memory leaves the next one alone,
and a GEMM launch whose optional workspace cannot grow takes its other kernel:
the same bits, no error.  The sizes asked for are thousands of times the memory
of the device, so nothing is allocated and nothing launched.
"""
import numpy as np
import pytest

from tests._cases import C, F, rel_l2, rng
from tests.test_gemm_bf16_pipe_gpu import _capture, _operands, say

pytestmark = pytest.mark.gpu

ENOMEM = -3


def test_next_call_after_a_refused_one(gpu, port):
    import ctypes
    from chimera_amd._lib import lib
    from chimera_amd.device import DeviceArray
    L = lib()
    say("case: refused allocation and refused workspace, then a transform")
    r = rng(5)
    kx = 2 * np.pi * np.fft.fftfreq(64, 0.04)
    v, In = C(r, 64, 9, 2), F(r, 8, 8, 2)
    z = np.zeros((64, 8, 2), complex, order="F")
    ref = port.fb_scl_in(z.copy(order="F"), v, -3.7, kx, In)
    p = ctypes.c_void_p(0)
    assert L.chimera_malloc(ctypes.byref(p), 1 << 46) == ENOMEM
    assert rel_l2(gpu.fb_scl_in(z.copy(order="F"), v, -3.7, kx, In), ref) < 1e-12
    # the transform's own workspace: 8192 x 2^24 x 8 x 3 complex values
    a = DeviceArray((64,), np.complex128)
    assert L.chimera_fb_forward(a.ptr, a.ptr, 0.0, a.ptr, a.ptr, None, 8192, 16, 8, 1 << 24, 3, 0, None) == ENOMEM
    assert rel_l2(gpu.fb_scl_in(z.copy(order="F"), v, -3.7, kx, In), ref) < 1e-12


def test_split_workspace_held_by_a_graph(gpu):
    """While a captured graph lives, the room for split matrices does not grow:
    the launch splits them in the kernel."""
    from chimera_amd._lib import check, lib
    from chimera_amd.batch import Context
    say("case: large mixed operator beside a live graph")
    out, run = _operands(1030, 544, 1, 32)
    run()
    ref = out.numpy()
    with Context() as ctx:
        o1, f1 = _operands(4100, 300, 1, 31)
        f1()
        g = _capture(f1)
        out2, run2 = _operands(1030, 544, 1, 32)
        run2()
        assert np.array_equal(out2.numpy(), ref)
        check("chimera_graph_destroy", lib().chimera_graph_destroy(g))
    ctx.close()
