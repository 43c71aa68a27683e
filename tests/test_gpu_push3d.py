"""The 3D cell-sum push against the FP64 oracle where its windows and passes can
go wrong: tiles with more particles than records at every order, moves that
cross y, z or both, the Courant number beyond which order 2 leaves its narrow
window, offsets on the node and half-cell lines, weights, ragged tiles."""
import numpy as np
import pytest

import orc
from gpu_util import make_context, norm64, random_state, rel, sorted_by_id

pytestmark = pytest.mark.gpu
# the bars that the other push tests hold against the same oracle
TOL_J, TOL_U, TOL_X = 2e-6, 1e-6, 8e-6


def _check(order, shape, npart, compat=orc.COMPAT_ALL, c=0.45, place=None, weights=False, seed=0):
    import tmpg
    nx, ny, nz = shape
    p = dict(c=c, corr=1.025, c_omp=4.0, gamma0=0.5, ppc0=4.0, me=1.0, mi=16.0)
    f, pi, pe = random_state(3, order, nx, ny, nz, npart, seed=100 + 10 * order + seed)
    cfg = orc.make_cfg(3, order, nx, ny, nz, compat=compat, c=c)
    h = orc.extent(cfg)[3] // 2
    rng = np.random.default_rng(seed + 5)
    for prt in (pi, pe):
        if place is not None:
            place(prt, h + 1, rng)
        if weights:
            prt[6] = rng.choice(np.array([0.25, 1.0, 2.5], np.float32), prt.shape[1])
    nm = norm64(p)
    ctx = make_context(tmpg, 3, order, nx, ny, nz, p, compat=compat)
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
        for a, n in ((0, nx), (1, ny), (2, nz)):
            d = (got[a].astype(np.float64) - r[a] + 0.5 * n) % n - 0.5 * n
            assert np.abs(d).max() < TOL_X
    orc.fold(cfg, j3)
    sl = (slice(None),) + orc.interior_slices(cfg)
    assert rel(ctx.get_currents()[sl], j3[sl]) < TOL_J
    ctx.close()


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("shape,npart", [((8, 8, 4), 30), ((11, 9, 6), 3000), ((16, 8, 4), 9000)])
def test_tiles_and_passes(order, shape, npart):
    """(16, 8, 4): two tiles of 9000 particles, four passes of records each"""
    _check(order, shape, npart)


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("c", [0.1, 0.55])
def test_courant_numbers(order, c):
    """hardly any crossings, and moves of more than half a cell"""
    _check(order, (16, 12, 10), 5000, c=c)


@pytest.mark.parametrize("order", [2, 3])
def test_every_particle_crosses_y_and_z(order):
    def place(prt, base, rng):
        n = prt.shape[1]
        s = rng.choice([-1.0, 1.0], (2, n))
        for a in (0, 1):
            prt[1 + a] = np.floor(prt[1 + a]) + np.where(s[a] > 0, 0.95, 0.05)
            prt[4 + a] = s[a] * 1.5
    _check(order, (16, 16, 8), 2500, place=place)


@pytest.mark.parametrize("order", [1, 2, 3])
def test_weights(order):
    _check(order, (16, 8, 8), 3000, weights=True)


def test_second_order_gather_without_the_quirk():
    _check(2, (16, 8, 8), 3000, compat=0)


@pytest.mark.parametrize("order", [1, 2, 3])
def test_offsets_on_nodes_and_half_cells(order):
    def place(prt, base, rng):
        n = prt.shape[1]
        for a in (0, 1, 2):
            prt[a] = np.floor(prt[a]) + rng.choice(np.array([0.0, 0.5, 0.25]), n)
    _check(order, (16, 8, 8), 2000, place=place)


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("npart", [1023, 1400, 1405, 2302, 2304, 2809, 2816, 5632])
def test_record_space_edges(order, npart):
    """one tile whose particles just fit the records, or do not, also where
    the last round before a drain takes less than a whole one"""
    _check(order, (8, 8, 4), npart)


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("npart", [1200, 6000])
def test_crowded_cell(order, npart):
    """a beam whose particles all sit in one cell: their sum in one FP32 chain
    would lose about 2e-5 of J; in chains of at most 32, 2^-24 for each of the
    32 additions and of some ten roundings of a particle's own stay below 2.6e-6
    if none cancels, and the bar"""
    def place(prt, base, rng):
        for a in (0, 1, 2):
            prt[a] = base + 3 + prt[a] % 1
        prt[3:6] = 0.05 * rng.standard_normal((3, prt.shape[1]))
        prt[3] += 1.0
    _check(order, (16, 8, 8), npart, place=place)


def test_one_dense_tile_among_sparse_ones():
    """order 3 with a mean below the records of a pass, so the single-pass
    kernel runs, and one tile of 4200 particles: its waves beyond the record
    space give their slots back and deposit at once, crossers among them"""
    def place(prt, base, rng):
        first = rng.random(prt.shape[1]) < 0.47
        prt[0] = base + np.where(first, (prt[0] - base) % 8, prt[0] - base)
        m = rng.random(prt.shape[1]) < 0.5
        prt[1] = np.where(m, np.floor(prt[1]) + 0.95, prt[1])
        prt[4] = np.where(m, 1.5, prt[4])
    _check(3, (32, 8, 4), 3500, place=place)
