"""The split-BF16 GEMMs of large launches (matrices split once per call) at the
edges of their tiles: x and column remainders in 128-, 64- and 32-column tiles,
K no multiple of the 32-deep stage, both kinds of segments and one and two
accumulators (rot, grad, div, graddiv), against the FP64 oracle; and the same
bits from call to call.

Bar 2e-6, that of the other tile tests: 6e-8 sqrt(2 K) for FP32 sums of two
segments of K <= 544 products, with operands exact in FP32.
"""
import numpy as np
import pytest

from tests._cases import C, F, rel_l2, rng
from tests.test_gemm_tiles_gpu import OPS, TOL32, _c8, say

pytestmark = pytest.mark.gpu


# 8190 x 160: 128-column tiles with 32 columns left, two x of the last tile
# missing; 4100 x 300: K remainder 12; 1030 x 544: 64-column tiles; 520 x 520:
# 32-column tiles, K remainder 8; 190 x 1024: three x tiles, fewer than XCDs;
# 830 x 544: 13, five more than XCDs
@pytest.mark.timeout(900)
@pytest.mark.parametrize("nkx,nkr,nko,name", [(8190, 160, 1, "div"), (8190, 160, 1, "rot"), (4100, 300, 1, "grad"),
                                              (4100, 300, 1, "graddiv"), (1030, 544, 1, "div"),
                                              (1030, 544, 1, "grad"), (520, 520, 2, "graddiv"),
                                              (520, 520, 2, "rot"), (190, 1024, 2, "rot"),
                                              (190, 1024, 2, "div"), (830, 544, 1, "rot"),
                                              (830, 544, 1, "graddiv")])
def test_edges(gpu, port, nkx, nkr, nko, name):
    say(f"case: fb_{name} nkx={nkx} nkr={nkr} nko={nko}")
    r = rng(9000 + nkx + nkr)
    f4 = lambda a: np.asfortranarray(a.astype(np.float32 if a.dtype == float else np.complex64).astype(a.dtype))  # noqa: E731
    kx = 2 * np.pi * np.fft.fftfreq(nkx, 1.0)
    Dp, Dm = f4(F(r, nkr, nkr, nko + 2)), f4(F(r, nkr, nkr, nko + 2))
    v, s = f4(C(r, nkx, nkr, nko + 1, 3)), f4(C(r, nkx, nkr, nko + 1))
    if name == "graddiv":
        out, inp = v, v
        ref = port.fb_graddiv(v.copy(order="F"), Dp, Dm, kx)
    else:
        out = np.zeros((nkx, nkr, nko + 1) + (() if name == "div" else (3,)), complex, order="F")
        inp = s if name == "grad" else v
        ref = getattr(port, "fb_" + name)(out.copy(order="F"), inp, Dp, Dm, kx)
    first = _c8(OPS[name], out.copy(order="F"), inp, Dp, Dm, kx, nko)
    e = rel_l2(first, ref)
    say(f"  mixed {e:.2e}")
    assert e < TOL32
    for _ in range(3):
        assert np.array_equal(_c8(OPS[name], out.copy(order="F"), inp, Dp, Dm, kx, nko), first)


def _operands(nkx, nkr, nko, seed):
    """Device operands of one large mixed divergence and a function that runs it."""
    from chimera_amd.device import DeviceArray, call
    r = rng(seed)
    d = lambda a, t: DeviceArray.from_numpy(a, t)                                    # noqa: E731
    a = [d(C(r, nkx, nkr, nko + 1, 3), np.complex64), d(F(r, nkr, nkr, nko + 2), np.float32),
         d(F(r, nkr, nkr, nko + 2), np.float32), DeviceArray.from_numpy(2 * np.pi * np.fft.fftfreq(nkx, 1.0))]
    out = DeviceArray((nkx, nkr, nko + 1), np.complex64)
    return out, lambda: call("chimera_fb_op_c8", OPS["div"], out.ptr, *(x.ptr for x in a), nkx, nkr, nko)


def _capture(run):
    import ctypes
    from chimera_amd._lib import DEVICE_LOCK, check, lib
    with DEVICE_LOCK:
        check("chimera_capture_begin", lib().chimera_capture_begin())
        try:
            run()
        except Exception:
            lib().chimera_capture_abort()
            raise
        h = ctypes.c_void_p(0)
        check("chimera_capture_end", lib().chimera_capture_end(ctypes.byref(h)))
    return h.value


def test_split_captured_after_one_pass(gpu):
    """A step whose second operator needs more room for its matrices than the
    first is recorded after one eager pass, and every replay gives its bits."""
    from chimera_amd._lib import check, lib
    from chimera_amd.batch import Context
    say("case: two large mixed operators, one eager pass, capture, replays")
    with Context() as ctx:
        (o1, f1), (o2, f2) = _operands(4100, 300, 1, 31), _operands(1030, 544, 1, 32)
        f1(), f2()
        ref = o1.numpy(), o2.numpy()
        g = _capture(lambda: (f1(), f2()))
        for _ in range(3):
            o1.write(0, np.zeros(o1.size, np.complex64))
            o2.write(0, np.zeros(o2.size, np.complex64))
            check("chimera_graph_launch", lib().chimera_graph_launch(g))
            ctx.synchronize()
            assert np.array_equal(o1.numpy(), ref[0]) and np.array_equal(o2.numpy(), ref[1])
        check("chimera_graph_destroy", lib().chimera_graph_destroy(g))
    ctx.close()
