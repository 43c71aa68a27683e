"""The cell tiles of a context: what an explicit tile leaves open, and which
tiles fit a CU's LDS."""
import numpy as np
import pytest

from gpu_util import make_context, periodic_diff, random_state, rel, sorted_by_id

pytestmark = pytest.mark.gpu
P = dict(c=0.45, corr=1.025, c_omp=4.0, gamma0=0.5, ppc0=4.0, me=1.0, mi=16.0)


@pytest.mark.parametrize("dim,shape,tile,scheme,fits", [
    (2, (200, 100, 1), (200, 0, 0), 0, True),      # 8 rows on a small grid
    (2, (200, 100, 1), (200, 16, 0), 0, False),
    (2, (1600, 1600, 1), (200, 0, 0), 0, False),   # 16 rows on a large one
    (3, (32, 32, 32), (16, 16, 0), 1, False),      # 4 planes
    (3, (32, 32, 32), (16, 16, 2), 1, True),
    (3, (32, 32, 32), (16, 16, 0), 0, False),
    (3, (32, 32, 32), (0, 0, 8), 1, True),         # 8x8
])
def test_partly_explicit_tiles(dim, shape, tile, scheme, fits):
    import tmpg
    if not fits:
        with pytest.raises(Exception, match="LDS"):
            make_context(tmpg, dim, 1, *shape, P, tile=tile, scheme=scheme)
        return
    ctx = make_context(tmpg, dim, 1, *shape, P, tile=tile, scheme=scheme)
    assert np.isfinite(ctx.get_fields()).all()
    ctx.close()


def _cells(ctx, dim, shape, species=0):
    """cell coordinates of a species' particles in the library's order"""
    h, hz = ctx.ng // 2, ctx.ngz // 2
    p = ctx.get_particles(species)
    lo = (h + 1, h + 1, hz + 1)
    return [np.floor(p[a]).astype(np.int64) - lo[a] if a < dim else np.zeros(p.shape[1], np.int64) for a in range(3)]


def _tile_ids(c, shape, tile):
    nt = [-(-shape[a] // tile[a]) for a in range(3)]
    t = [c[a] // tile[a] for a in range(3)]
    return t[0] + nt[0] * (t[1] + nt[1] * t[2])


def _load(ctx, dim, shape, n, seed, species=(0, 1)):
    """n particles per species at rest, away from the cells' faces"""
    h, hz = ctx.ng // 2, ctx.ngz // 2
    for s in species:
        rng = np.random.default_rng(seed + s)
        p = np.zeros((7, n), np.float32)
        for a, lo in enumerate((h + 1, h + 1, hz + 1)):
            p[a] = lo + rng.integers(0, shape[a] if a < dim else 1, n) + 0.25 + 0.5 * rng.random(n)
        p[6] = 1.0
        ctx.set_particles(s, p)


@pytest.mark.parametrize("dim,order,compat,tile,sorts", [
    (3, 3, 7, (0, 0, 0), True), (3, 2, 0, (0, 0, 0), True), (3, 2, 7, (0, 0, 0), False), (3, 1, 7, (0, 0, 0), False),
    (3, 3, 7, (8, 8, 8), False), (3, 2, 7, (8, 8, 2), True), (3, 2, 0, (8, 8, 2), True), (3, 1, 7, (8, 8, 2), False),
    (2, 3, 7, (32, 8, 0), False), (2, 2, 7, (12, 12, 0), False),
])
def test_default_sort_goes_with_the_kernel(dim, order, compat, tile, sorts):
    """the default sorts (before the fourth step) only where the push that
    runs gains from it: the order within the tiles tells"""
    import tmpg
    shape = (16, 16, 8) if dim == 3 else (48, 24, 1)
    ctx = make_context(tmpg, dim, order, *shape, P, compat=compat, tile=tile, track_ids=False)
    _load(ctx, dim, shape, 12000, 11)
    ctx.step(4)
    c = _cells(ctx, dim, shape)
    ctx.close()
    size = [t or d for t, d in zip(tile, (8, 8, 4))] if dim == 3 else [tile[0], tile[1], 1]
    t = _tile_ids(c, shape, size)
    local = sum((c[a] % size[a]) * m for a, m in zip(range(3), (1, size[0], size[0] * size[1])))
    same = t[1:] == t[:-1]
    rising = np.mean(np.diff(local)[same] >= 0)
    assert (rising > 0.9) == sorts and (rising < 0.6) != sorts


@pytest.mark.parametrize("order,tile,ppc", [(1, (12, 12, 1), 6), (2, (32, 8, 1), 14), (3, (12, 12, 1), 3)])
def test_sorted_run_matches_unsorted_2d(order, tile, ppc):
    """tiles whose push reads the particles in stored order: sorted before every
    step and never, they hold the same particles and fields up to the order of
    the currents' additions (the bars of the sort's other tests)"""
    import orc
    import tmpg
    nx, ny = 48, 32
    f, pi, pe = random_state(2, order, nx, ny, 1, ppc * nx * ny, seed=60 + order, emax=0.02, bmax=0.05, umax=0.8)
    full = orc.fill_from_interior(orc.make_cfg(2, order, nx, ny, 1), f, np.float32)[:6]
    out = []
    for sort_every in (1, -1):
        ctx = make_context(tmpg, 2, order, nx, ny, 1, P, sort_every=sort_every, tile=tile)
        ctx.set_fields(full)
        ctx.set_particles(0, pi)
        ctx.set_particles(1, pe)
        ctx.step(6)
        out.append(([sorted_by_id(*ctx.get_particles(s, with_ids=True)) for s in (0, 1)], ctx.get_fields()))
        ctx.close()
    (ps, fs), (pu, fu) = out
    for s in (0, 1):
        for r, n in ((0, nx), (1, ny)):
            assert np.abs(periodic_diff(ps[s][r], pu[s][r], 0, n)).max() < 1e-4
        assert rel(ps[s][3:6], pu[s][3:6]) < 1e-6
    for q in range(6):
        assert rel(fs[q], fu[q]) < 1e-5


def _tile(ctx, shape):
    """the finest of the 2D default tiles that the particles run by (but for
    single ones whose rounded position lies across a face)"""
    c = _cells(ctx, 2, shape)
    for tile in ((8, 8, 1), (16, 8, 1), (16, 16, 1)):
        if np.mean(np.diff(_tile_ids(c, shape, tile)) < 0) < 1e-3:
            return tile
    return None


@pytest.mark.parametrize("n,order,ppc,c,tile", [
    (384, 2, 8, 0.6, (16, 16, 1)), (384, 2, 8, 0.45, (8, 8, 1)),           # a push without register sums
    (128, 2, 8, 0.6, (8, 8, 1)),
    (736, 1, 6, 0.45, (16, 16, 1)), (736, 1, 7, 0.45, (8, 8, 1)),          # eight tiles per CU
    (736, 2, 5, 0.45, (16, 16, 1)), (736, 2, 6, 0.45, (8, 8, 1)),
    (736, 3, 4, 0.45, (16, 8, 1)), (736, 3, 5, 0.45, (8, 8, 1)),
    (384, 1, 3, 0.45, (16, 16, 1)), (384, 1, 4, 0.45, (8, 8, 1)),          # two
    (384, 2, 2, 0.45, (16, 16, 1)), (384, 2, 3, 0.45, (8, 8, 1)),
])
def test_default_tiles_2d(n, order, ppc, c, tile):
    import tmpg
    ctx = make_context(tmpg, 2, order, n, n, 1, dict(P, c=c), track_ids=False)
    for s in (0, 1):
        ctx.load_uniform(s, ppc, 0.0, 0.01, 3 + s)
    assert _tile(ctx, (n, n, 1)) == tile
    ctx.close()


@pytest.mark.parametrize("loads,tile", [
    (((0, 2), (1, 14)), (8, 8, 1)), (((1, 14), (0, 2)), (8, 8, 1)),
    (((0, 4),), (16, 16, 1)), (((1, 6), (0, 0)), (16, 16, 1)), (((0, 1), (1, 1), (1, 8)), (8, 8, 1)),
])
@pytest.mark.parametrize("push", ["step", "push_deposit", "move"])
def test_tiles_go_with_all_particles(loads, tile, push):
    """the tiles of a run are those of its whole density, in whatever order and
    parts the species come"""
    import tmpg
    n = 384
    ctx = make_context(tmpg, 2, 1, n, n, 1, P, track_ids=False)
    for k, (s, ppc) in enumerate(loads):
        if ppc:
            ctx.load_uniform(s, ppc, 0.0, 0.01, 3 + k)
    before = [ctx.get_particles(s) for s in (0, 1)]
    if push == "step":
        ctx.step(1)
    else:
        getattr(ctx, push)()
    shape = (n, n, 1)
    for s in (0, 1):
        if before[s].shape[1]:
            c = _cells(ctx, 2, shape, s)
            assert np.mean(np.diff(_tile_ids(c, shape, tile)) < 0) < 1e-3
            finer = (8, 8, 1) if tile[0] == 16 else (8, 4, 1)
            assert np.mean(np.diff(_tile_ids(c, shape, finer)) < 0) > 0.01
        after = ctx.get_particles(s)
        assert after.shape == before[s].shape
        if push != "step":
            u0, u1 = (np.sort(x[3]) for x in (before[s], after))
            assert rel(u1, u0) < 1e-5 or u0.size == 0
    ctx.close()
