"""The resident push + deposit (chimera_soa_push_deposit, _mixed) against the
oracle's dep_curr / dep_dens, at the sizes where its paths change: group and
wave remainders, unaligned arrays, every way a group's tile leaves the block
(all components at once, J then rho, one component at a time, past the slot,
no tile at all), both group sizes, and combines with and without row masks.

Bars.  FP64: 1e-12 of the largest value; the inputs are identical and the
geometry expressions the same, so what differs is the order of the sums and
the last bits of 1/gamma and 1/r (1e-15 per contribution), and of the pushed
positions: 1e-16 * u dt / gamma in units of dx = 0.1 is 1e-15 of a weight.
Mixed: the float32 inputs are the reference's too; every value is summed in
FP64 per group, rounded to float32 once and summed over the groups of a node
in float32 (at most a few dozen here): 2e-6 in relative L2.
"""
import sys

import numpy as np
import pytest

from tests._cases import Grid, particles, rel_l2, rel_max

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def cell_sorted(coord, mom, w, g):
    rp = np.sqrt(coord[1] ** 2 + coord[2] ** 2)
    key = np.floor((rp - g.Rgrid[0]) / g.dr) * g.nx + np.floor((coord[0] - g.leftX) / g.dx)
    o = np.argsort(key, kind="stable")
    return coord[:, o], mom[:, o], w[o]


def deposit(coord, half, mom, w, g, precision="fp64", dt=0.0, ld=None, curr=True, dens=True, shift=0.0):
    """(x, x_half, J, rho) of one call on grids that hold 1 + 2i beforehand."""
    from chimera_amd.device import DeviceArray, call
    n = w.size
    ld = n if ld is None else ld
    mixed = precision == "mixed"
    rt, ct = (np.float32, np.complex64) if mixed else (np.float64, np.complex128)

    def soa(a, t):
        d = DeviceArray((ld, 3), t)
        for c in range(3):
            d.write(c * ld, a[c])
        return d

    x, xh, u = soa(coord, np.float64), soa(half, np.float64), soa(mom, rt)
    wd = DeviceArray((ld,), rt)
    wd.write(0, w)
    sh = (g.nx, g.nkr + 1, g.nmod)
    J = DeviceArray.from_numpy(np.full(sh + (3,), 1 + 2j, ct, order="F"))
    R = DeviceArray.from_numpy(np.full(sh, 1 + 2j, ct, order="F"))
    Rg = DeviceArray.from_numpy(g.Rgrid)
    call("chimera_soa_push_deposit" + ("_mixed" if mixed else ""), x.ptr, xh.ptr, u.ptr, wd.ptr, ld, n, dt, g.leftX,
         g.leftX + shift, Rg.ptr, 1 / g.dx, 1 / g.dr, float(g.Rgrid[0]), float(g.Rgrid[-1]), g.nx - 1, g.nkr, g.nko,
         J.ptr if curr else None, R.ptr if dens else None, None)
    return x.numpy()[:n].T, xh.numpy()[:n].T, J.numpy() - (1 + 2j), R.numpy() - (1 + 2j)


def unfold_compare(got, ref):
    """got is unfolded; ref carries the ghost fold (grid_deps.f90:80-85)."""
    got = got.astype(np.complex128)
    got[:, 1] -= got[:, 0]
    got[:, 0] = 0
    return got, ref


def check(port, coord, half, new, mom, w, g, out, precision, shift=0.0, curr=True, dens=True):
    f = lambda a: np.asfortranarray(a, dtype=np.float64)   # noqa: E731
    args = (g.Rgrid, 1 / g.dx, 1 / g.dr)
    sh = (g.nx, g.nkr + 1, g.nmod)
    refs = []
    J = np.zeros(sh + (3,), complex, order="F")
    R = np.zeros(sh, complex, order="F")
    if curr:
        J = port.dep_curr(f(half), f(mom), f(w), J, g.leftX, *args)
    if dens:
        R = port.dep_dens(f(new), f(w), R, g.leftX + shift, *args)
    refs = [unfold_compare(out[2], J), unfold_compare(out[3], R)]
    for name, (got, ref) in zip(("J", "rho"), refs):
        if not np.any(ref):
            assert not np.any(got), name
            continue
        if precision == "fp64":
            err, bar = rel_max(got, ref), 1e-12
        else:
            err, bar = rel_l2(got, ref), 2e-6
        say(f"  {name} {err:.2e}")
        assert err < bar, (name, err)


# (nx, nkr, nko, n, order, precision): which path the groups take
CASES = [
    (13, 6, 1, 1, "shuffled", "fp64"),          # one particle
    (13, 6, 1, 255, "shuffled", "fp64"),        # group remainders; all components in one tile
    (13, 6, 1, 257, "shuffled", "mixed"),
    (13, 6, 0, 1000, "shuffled", "fp64"),
    (13, 6, 3, 1025, "shuffled", "fp64"),       # J then rho
    (13, 6, 3, 1025, "shuffled", "mixed"),
    (13, 6, 7, 700, "shuffled", "fp64"),        # one component at a time, past the slot
    (65, 16, 0, 3000, "shuffled", "fp64"),      # the same by its box
    (65, 16, 2, 3000, "shuffled", "fp64"),      # no tile
    (65, 16, 2, 3000, "shuffled", "mixed"),
    (65, 16, 2, 40000, "sorted", "fp64"),
    (65, 16, 3, 300001, "sorted", "fp64"),      # 512-particle groups
    (65, 16, 2, 300001, "sorted", "mixed"),
    (1024, 128, 1, 300002, "sorted", "fp64"),   # 256-particle groups, row masks
    (1024, 128, 1, 560000, "twice", "mixed"),   # two ordered sets, masks of two words
]


@pytest.mark.parametrize("nx,nkr,nko,n,order,precision", CASES)
def test_deposit_paths(port, nx, nkr, nko, n, order, precision):
    say(f"case: deposit nx={nx} nkr={nkr} nko={nko} n={n} {order} {precision}")
    g = Grid(nx=nx, nkr=nkr, nko=nko, leftX=-0.05 * nx)
    coord, mom, w = particles(g, n, seed=n)
    if order == "sorted":
        coord, mom, w = cell_sorted(coord, mom, w, g)
    elif order == "twice":
        h = n // 2
        parts = [cell_sorted(coord[:, s], mom[:, s], w[s], g) for s in (slice(0, h), slice(h, n))]
        coord, mom, w = np.hstack([p[0] for p in parts]), np.hstack([p[1] for p in parts]), np.hstack([p[2] for p in parts])
    if precision == "mixed":
        mom, w = mom.astype(np.float32), w.astype(np.float32)
    half = coord + 0.01
    # no push: J at the half-step positions as given, rho at the positions
    out = deposit(coord, half, mom, w, g, precision, shift=0.03)
    check(port, coord, half, coord, mom, w, g, out, precision, shift=0.03)


# Tiles of two or three node columns and hundreds of node rows, most of them more
# than a group has threads, with row masks (more than 1024 groups of 256
# particles) and without: no row of such a tile may be lost, whichever way it goes
# to the grid (all components at once, J then rho, one at a time).  "randcell": the order of Species.gen_randcell with
# one particle a cell (column by column, the radius fastest); "sheet": one column
# of cells, its particles in random order.
@pytest.mark.parametrize("nx,nkr,nko,n,order,curr", [(1025, 299, 0, 1024 * 299, "randcell", True),
                                                     (1025, 250, 0, 1024 * 250, "randcell", True),
                                                     (201, 500, 0, 600000, "sheet", True),
                                                     (201, 390, 1, 600000, "sheet", False)])
def test_deposit_tall_tiles(port, nx, nkr, nko, n, order, curr):
    say(f"case: deposit nx={nx} nkr={nkr} nko={nko} n={n} {order} curr={curr}")
    g = Grid(nx=nx, nkr=nkr, nko=nko, leftX=-0.05 * nx)
    r = np.random.default_rng(nkr)
    if order == "randcell":
        x = (g.leftX + g.dx * (np.arange(nx - 1)[:, None] + 0.5 * r.uniform(0, 1, (nx - 1, nkr)))).ravel()
        rr = (g.Rgrid[:-1] + g.dr * 0.5 * (1 + r.uniform(0.02, 1, (nx - 1, nkr)))).ravel()
    else:
        x = g.leftX + g.dx * (nx // 2 + r.uniform(0.02, 0.98, n))
        rr = r.uniform(0.02, g.Rgrid[-1] - 0.02, n)
    th = r.uniform(0, 2 * np.pi, n)
    coord = np.vstack([x, rr * np.sin(th), rr * np.cos(th)])
    mom, w = r.standard_normal((3, n)), r.uniform(0.1, 1.0, n)
    out = deposit(coord, coord, mom, w, g, curr=curr)
    check(port, coord, coord, coord, mom, w, g, out, "fp64", curr=curr)


@pytest.mark.parametrize("curr,dens", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("ld_extra", [0, 1, 37])
def test_deposit_push_and_parts(port, curr, dens, ld_extra):
    """With a push, J or rho alone, and arrays no vector load may take."""
    n = 1283
    say(f"case: push, curr={curr} dens={dens} ld={n + ld_extra}")
    g = Grid(nx=33, nkr=9, nko=2, leftX=-1.65)
    coord, mom, w = particles(g, n, seed=3, margin=0.2)
    dt = 0.05
    gam = np.sqrt(1 + (mom ** 2).sum(0))
    new = coord + mom * (dt / gam)
    half = 0.5 * (coord + new)
    out = deposit(coord, np.zeros_like(coord), mom, w, g, dt=dt, ld=n + ld_extra, curr=curr, dens=dens)
    assert rel_max(out[0], new) < 1e-15 and rel_max(out[1], half) < 1e-15
    check(port, half, half, new, mom, w, g, out, "fp64", curr=curr, dens=dens)


def test_deposit_skips_and_lost_particles(port):
    """Particles outside the grid (the reference would write outside its
    arrays) or not a number deposit nothing; nothing else changes.  (At rest and
    without weight: test_deposit_paths, whose particles have both.)"""
    say("case: skipped particles")
    g = Grid(nx=33, nkr=9, nko=2, leftX=-1.65)
    coord, mom, w = particles(g, 900, seed=8)
    ref = deposit(coord, coord, mom, w, g)
    bad = np.array([[g.leftX - 5, 0, 0], [g.leftX + 100, 0.1, 0], [0, 50.0, 0], [np.nan, 0.1, 0.1],
                    [0, np.nan, 0], [np.inf, 0, 0], [0, np.inf, 0]]).T
    c2 = np.hstack([bad, coord])
    m2 = np.hstack([np.ones((3, 7)), mom])
    w2 = np.hstack([np.ones(7), w])
    out = deposit(c2, c2, m2, w2, g)
    assert rel_max(out[2], ref[2]) < 1e-13 and rel_max(out[3], ref[3]) < 1e-13
    none = deposit(bad, bad, np.ones((3, 7)), np.ones(7), g)
    assert not np.any(none[2]) and not np.any(none[3])


# groups that all hand their tile on in a slot: every way the components share
# the LDS, both group sizes, one and several rounds of segments a wave
@pytest.mark.parametrize("nx,nkr,nko,n,order,precision", [
    (13, 6, 1, 20001, "shuffled", "fp64"), (13, 6, 3, 20001, "shuffled", "fp64"), (65, 16, 2, 300001, "sorted", "fp64"),
    (65, 16, 2, 300001, "sorted", "mixed"), (33, 16, 1, 40000, "sorted", "fp64"), (13, 6, 4, 300000, "sorted", "fp64")])
def test_deposit_same_bits(nx, nkr, nko, n, order, precision):
    """The sums of slotted tiles have one order: the same bits from call to call."""
    say(f"case: deposit bits nx={nx} nkr={nkr} nko={nko} n={n} {order} {precision}")
    g = Grid(nx=nx, nkr=nkr, nko=nko, leftX=-0.05 * nx)
    coord, mom, w = particles(g, n, seed=n)
    if order == "sorted":
        coord, mom, w = cell_sorted(coord, mom, w, g)
    first = deposit(coord, coord, mom, w, g, precision)
    for _ in range(5):
        again = deposit(coord, coord, mom, w, g, precision)
        assert all(np.array_equal(a, b) for a, b in zip(first, again))
