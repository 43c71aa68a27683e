"""The cell tiles of a context: what an explicit tile leaves open, and which
tiles fit a CU's LDS."""
import numpy as np
import pytest

from gpu_util import make_context

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
