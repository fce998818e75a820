"""Brute-force distance fields over grids with one or two short axes, at the
edges of each shape of a lane's block, bit for bit against the oracle."""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(31, 1, 1), (8193, 1, 1), (20000, 1, 1), (1, 32, 1), (1, 16389, 1), (2, 16415, 1),
                                  (1, 1, 32), (1, 1, 16385), (1, 3, 16383), (3, 2, 64), (129, 1, 257), (181, 97, 1),
                                  (1, 257, 129), (8191, 2, 1), (131, 257, 2)])
def test_short_axes(ctx, dims):
    rng = np.random.default_rng(sum(dims))
    for n in (1, 65, 515):
        pts = (rng.random((n, 3)) * np.array(dims)).astype(np.float32)
        d = ctx.to_device(pts)
        got = ctx.df_points(d, n, dims, 1, isoamd.DF_BRUTE).numpy()
        want = oracle.df_brute(oracle.normalize(pts, dims), dims, 1)
        assert np.array_equal(got.ravel(), want.ravel()), n
        d.free()
