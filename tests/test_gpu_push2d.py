"""The 2D push in cell order against the FP64 oracle where it can go wrong:
every tile that has an instantiation, one cell to many passes' particles in a
tile, cells with more particles than one work item, ragged grids, offsets on
the node lines and half-cell lines, weights and ids, both gather ranges of
order 2, and the Courant number beyond which order 2 leaves its window."""
import numpy as np
import pytest

import orc
from gpu_util import make_context, norm64, random_state, rel, sorted_by_id

pytestmark = pytest.mark.gpu
# FP32 arithmetic and one FP32 sum per cell and pass against FP64: the bars
# that the other push tests hold against the same oracle
TOL_J, TOL_U, TOL_X = 2e-6, 1e-6, 8e-6


def _check(order, shape, npart, tile=(0, 0, 0), compat=orc.COMPAT_ALL, c=0.45, place=None, weights=False, seed=0):
    import tmpg
    nx, ny = shape
    p = dict(c=c, corr=1.025, c_omp=4.0, gamma0=0.5, ppc0=4.0, me=1.0, mi=16.0)
    f, pi, pe = random_state(2, order, nx, ny, 1, npart, seed=100 + 10 * order + seed)
    cfg = orc.make_cfg(2, order, nx, ny, 1, compat=compat, c=c)
    h = orc.extent(cfg)[3] // 2
    rng = np.random.default_rng(seed + 5)
    for prt in (pi, pe):
        if place is not None:
            place(prt, h + 1, rng)
        if weights:
            prt[6] = rng.choice(np.array([0.25, 1.0, 2.5], np.float32), prt.shape[1])
    nm = norm64(p)
    ctx = make_context(tmpg, 2, order, nx, ny, 1, p, compat=compat, tile=tile)
    ctx.set_fields(orc.fill_from_interior(cfg, f, np.float32)[:6])
    ctx.set_particles(0, pi)
    ctx.set_particles(1, pe)
    ctx.reset_currents()
    ctx.push_deposit()
    f6 = orc.fill_from_interior(cfg, f.astype(np.float64), np.float64)
    j3 = orc.zeros_grid(cfg, 3, np.float64)
    for s, (prt, qm, q) in enumerate(((pi, "qmi", "qi"), (pe, "qme", "qe"))):
        r = prt.astype(np.float64)
        orc.mover(cfg, f6, r, nm[qm])
        orc.deposit(cfg, j3, r, nm[q])
        got, ids = ctx.get_particles(s, with_ids=True)
        got = sorted_by_id(got, ids)
        assert rel(got[3:6], r[3:6]) < TOL_U
        np.testing.assert_array_equal(got[6], prt[6])
        for a, n in ((0, nx), (1, ny)):
            d = (got[a].astype(np.float64) - r[a] + 0.5 * n) % n - 0.5 * n
            assert np.abs(d).max() < TOL_X
    orc.fold(cfg, j3)
    sl = (slice(None),) + orc.interior_slices(cfg)
    assert rel(ctx.get_currents()[sl], j3[sl]) < TOL_J
    ctx.close()


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("tile", [(8, 8, 1), (16, 8, 1), (16, 16, 1)])
@pytest.mark.parametrize("shape,npart", [((33, 19), 40), ((16, 16), 9000), ((50, 40), 9001)])
def test_tiles_and_passes(order, tile, shape, npart):
    _check(order, shape, npart, tile)


@pytest.mark.parametrize("order", [1, 2, 3])
def test_weights(order):
    _check(order, (40, 24), 5000, weights=True)


def test_second_order_gather_without_the_quirk():
    _check(2, (40, 24), 5000, compat=0)


@pytest.mark.parametrize("order", [1, 2, 3])
def test_crowded_cells(order):
    """all particles in three cells: many work items for each"""
    def place(prt, base, rng):
        k = rng.integers(0, 3, prt.shape[1])
        prt[0] = base + np.array([2, 7, 8])[k] + prt[0] % 1
        prt[1] = base + np.array([3, 3, 15])[k] + prt[1] % 1
    _check(order, (24, 16), 3000, place=place)


@pytest.mark.parametrize("order", [1, 2, 3])
def test_offsets_on_nodes_and_half_cells(order):
    """offsets of exactly 0 and 1/2, where weights change their pieces"""
    def place(prt, base, rng):
        n = prt.shape[1]
        for a in (0, 1):
            prt[a] = np.floor(prt[a]) + rng.choice(np.array([0.0, 0.5, 0.25]), n)
    _check(order, (24, 18), 2000, place=place)


@pytest.mark.parametrize("order", [1, 2, 3])
def test_large_courant_number(order):
    """moves of up to 0.9 cells"""
    _check(order, (24, 18), 2000, c=0.9)


@pytest.mark.parametrize("tile", [(8, 8, 1), (16, 8, 1), (16, 16, 1)])
def test_every_move_leaves_the_window(tile):
    """order 3, nearly every particle crosses a cell boundary in y, in several
    passes: more moves than the list of a pass has room for (a quarter of its
    particles), so rows are added both from the list and at once"""
    def place(prt, base, rng):
        up = rng.random(prt.shape[1]) < 0.5
        prt[1] = np.floor(prt[1]) + np.where(up, 0.95, 0.05)
        prt[4] = np.where(up, 1.5, -1.5)
    _check(3, (24, 16), 6000, tile, place=place)


@pytest.mark.parametrize("order", [1, 2, 3])
def test_a_particle_that_is_not_a_number_stays_one(order):
    """a NaN momentum gives NaN positions, not a number inside the grid, on
    this push and the next, and leaves the other particles alone"""
    import tmpg
    nx, ny, n = 24, 18, 1500
    p = dict(c=0.45, corr=1.025, c_omp=4.0, gamma0=0.5, ppc0=4.0, me=1.0, mi=16.0)
    f, pi, pe = random_state(2, order, nx, ny, 1, n, seed=7)
    cfg = orc.make_cfg(2, order, nx, ny, 1)
    fields = orc.fill_from_interior(cfg, f, np.float32)[:6]
    bad = (3, 777, n - 1)
    out = []
    for nan in (False, True):
        if nan:
            for q, s in zip(bad, (1.0, -1.0, 1.0)):
                pi[3 + q % 3, q] = np.copysign(np.float32(np.nan), np.float32(s))
        ctx = make_context(tmpg, 2, order, nx, ny, 1, p)
        ctx.set_fields(fields)
        ctx.set_particles(0, pi)
        ctx.set_particles(1, pe)
        ctx.push_deposit()
        ctx.push_deposit()
        out.append([sorted_by_id(*ctx.get_particles(s, with_ids=True)) for s in (0, 1)])
        ctx.close()
    (a0, a1), (b0, b1) = out
    good = np.ones(n, bool)
    good[list(bad)] = False
    np.testing.assert_array_equal(a1, b1)
    np.testing.assert_array_equal(a0[:, good], b0[:, good])
    assert np.isnan(b0[:2, ~good]).all() and np.isnan(b0[3:6, ~good]).all()
