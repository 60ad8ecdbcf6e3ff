"""The x transforms at every length that has its own passes: powers of two from
1 to 8192 (one thread per line up to 32 points, several lines per wave up to
512, one block per line beyond, three passes from 512) and one or two other
lengths for each convolution length 64..8192, with a line count that leaves the
last block partly empty, forward, backward and there and back with the filter,
in complex128 and complex64.  At 1024 x 1200 lines the phase has its own launch.

Tolerances (relative L2 against the FP64 oracle): complex128 1e-12, the bar of
the other transform tests; complex64 2e-6: three roundings of 6e-8 a pass, at
most 2 x 3 passes and two chirps, and as much again for the Hankel product.
"""
import sys

import numpy as np
import pytest

from tests._cases import C, F, rel_l2, rng

pytestmark = pytest.mark.gpu

LENGTHS = [2 ** k for k in range(14)] + [3, 31, 33, 63, 100, 129, 255, 300, 513, 1025, 1999, 4095]


def case(nkx, nr, nkr, M):
    print(f"case: transforms nkx={nkx} nr={nr} nkr={nkr} M={M}", flush=True)
    sys.stdout.flush()
    r = rng(4100 + nkx)
    c8 = lambda a: np.asfortranarray(a.astype(np.complex64).astype(complex))         # noqa: E731
    f4 = lambda a: np.asfortranarray(a.astype(np.float32).astype(float))             # noqa: E731
    kx = 2 * np.pi * np.fft.fftfreq(nkx, 0.04)
    return (c8(C(r, nkx, nr + 1, M)), f4(F(r, nr, nkr, M)), c8(C(r, nkx, nkr, M, 6)), c8(C(r, nkx, nkr, M, 3)),
            f4(F(r, nkr, nr, M)), kx)


@pytest.mark.parametrize("nkx,nr,nkr,M", [(n, 5, 3, 1) for n in LENGTHS] + [(1024, 3, 600, 2)])
def test_lines(gpu, port, nkx, nr, nkr, M):
    from chimera_amd.device import DeviceArray, call
    s, In, e, b, Out, kx = case(nkx, nr, nkr, M)
    z = np.zeros((nkx, nkr, M), complex, order="F")
    eb = np.zeros((nkx, nr + 1, M, 6), complex, order="F")
    fwd = port.fb_scl_in(z.copy(order="F"), s, -3.7, kx, In)
    inv = port.fb_eb_out(eb.copy(order="F"), e, b, -3.7, kx, Out)
    assert rel_l2(gpu.fb_scl_in(z.copy(order="F"), s, -3.7, kx, In), fwd) < 1e-12
    assert rel_l2(gpu.fb_eb_out(eb.copy(order="F"), e, b, -3.7, kx, Out), inv) < 1e-12
    d = lambda a, t: DeviceArray.from_numpy(a, t)                                    # noqa: E731
    o, d_kx = DeviceArray((nkx, nkr, M), np.complex64), DeviceArray.from_numpy(kx)
    i, m = d(s, np.complex64), d(In, np.float32)
    call("chimera_fb_forward_c8", o.ptr, i.ptr, -3.7, d_kx.ptr, m.ptr, None, nkx, nr, M, nkr, 1, 0, None)
    assert rel_l2(o.numpy(), fwd) < 2e-6
    o, m = DeviceArray((nkx, nr + 1, M, 6), np.complex64), d(Out, np.float32)
    i, j = d(e, np.complex64), d(b, np.complex64)
    call("chimera_fb_inverse_c8", o.ptr, i.ptr, j.ptr, -3.7, d_kx.ptr, m.ptr, nkx, nr, M, nkr, 1, None)
    assert rel_l2(o.numpy(), inv) < 2e-6


@pytest.mark.parametrize("nkx", [4, 32, 64, 100, 256, 1024, 1025, 4096, 4095, 8192])
def test_filter(gpu, port, nkx):
    r = rng(4300 + nkx)
    print(f"case: fb_filtr nkx={nkx}", flush=True)
    v = C(r, nkx, 3, 1, 3)
    kx = 2 * np.pi * np.fft.fftfreq(nkx, 0.04)
    filt = np.linspace(0.0, 1.0, max(2, nkx // 3))
    assert rel_l2(gpu.fb_filtr(v.copy(order="F"), -3.7, kx, filt, 0),
                  port.fb_filtr(v.copy(order="F"), -3.7, kx, filt, 0)) < 1e-12
