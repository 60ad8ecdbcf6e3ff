"""The FP64 GEMM pipeline (tiles of 64 complex x) at the edges of its tiles,
against the FP64 oracle: matrices of fewer columns than a tile, column and x
remainders in 128-, 64- and 32-column tiles, K no multiple of the 16-deep stage,
and both kinds of segments with one and two accumulators.  The clamped loads of
such a tile stay inside the matrices, and none of what they read twice is stored.

Bar 1e-12 relative L2, that of the other tile tests in FP64: sums of at most
2 x 544 products, 1e-16 sqrt(1088) = 4e-15 with both orders.
"""
import numpy as np
import pytest

from tests._cases import C, F, rel_l2, rng
from tests.test_gemm_tiles_gpu import TOL64, say

pytestmark = pytest.mark.gpu


# 8192 x 40: 40 of 128 columns, K remainder 8; 2048 x 100: 64-column tiles, 36
# of the second one's; 1024 x 70: 32-column tiles, K remainder 6; 8192 x 1: one
# column, one row
@pytest.mark.timeout(900)
@pytest.mark.parametrize("nkx,nkr,M", [(8192, 40, 4), (2048, 100, 4), (1024, 70, 4), (8192, 1, 2)])
def test_transform_edges(gpu, port, nkx, nkr, M):
    say(f"case: fb_vec_in nkx={nkx} nkr={nkr} M={M}")
    r = rng(9100 + nkx + nkr)
    kx = 2 * np.pi * np.fft.fftfreq(nkx, 0.04)
    v, In = C(r, nkx, nkr + 1, M, 3), F(r, nkr, nkr, M)
    z = np.zeros((nkx, nkr, M, 3), complex, order="F")
    e = rel_l2(gpu.fb_vec_in(z.copy(order="F"), v, -3.7, kx, In), port.fb_vec_in(z.copy(order="F"), v, -3.7, kx, In))
    say(f"  {e:.2e}")
    assert e < TOL64


# 8190 x 160: 128-column tiles with 32 columns left, two x of the last tile
# missing; 4100 x 300: K remainder 12; 1030 x 544: 64-column tiles; 520 x 520:
# 32-column tiles, K remainder 8; 8192 x 33: one column past 32; 190 x 1024: three x
# tiles, fewer than XCDs; 830 x 544: 13, five more than XCDs
@pytest.mark.timeout(900)
@pytest.mark.parametrize("nkx,nkr,nko,name", [(8190, 160, 1, "div"), (8190, 160, 1, "rot"), (4100, 300, 1, "grad"),
                                              (4100, 300, 1, "graddiv"), (1030, 544, 1, "div"),
                                              (1030, 544, 1, "grad"), (520, 520, 2, "graddiv"),
                                              (520, 520, 2, "rot"), (8192, 33, 3, "graddiv"), (8192, 33, 3, "rot"),
                                              (190, 1024, 2, "rot"), (190, 1024, 2, "div"),
                                              (830, 544, 1, "rot"), (830, 544, 1, "graddiv")])
def test_operator_edges(gpu, port, nkx, nkr, nko, name):
    say(f"case: fb_{name} nkx={nkx} nkr={nkr} nko={nko}")
    r = rng(9200 + nkx + nkr)
    kx = 2 * np.pi * np.fft.fftfreq(nkx, 1.0)
    Dp, Dm = F(r, nkr, nkr, nko + 2), F(r, nkr, nkr, nko + 2)
    v, s = C(r, nkx, nkr, nko + 1, 3), C(r, nkx, nkr, nko + 1)
    if name == "graddiv":
        got, ref = (m.fb_graddiv(v.copy(order="F"), Dp, Dm, kx) for m in (gpu, port))
    else:
        out = np.zeros((nkx, nkr, nko + 1) + (() if name == "div" else (3,)), complex, order="F")
        got, ref = (getattr(m, "fb_" + name)(out.copy(order="F"), s if name == "grad" else v, Dp, Dm, kx)
                    for m in (gpu, port))
    e = rel_l2(got, ref)
    say(f"  {e:.2e}")
    assert e < TOL64
