"""Brute-force distance fields at the edges of a lane's block of samples, of a
workgroup's and of a wave's points, bit for bit against the oracle."""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 4, 4), (3, 5, 7), (8, 4, 1), (17, 9, 1), (1, 1, 130),
                                  (33, 2, 66), (130, 1, 3)])
def test_brute_block_edges(ctx, dims):
    rng = np.random.default_rng(sum(dims))
    for n in (1, 2, 63, 65, 511, 513, 4097):
        pts = (rng.random((n, 3)) * np.array(dims)).astype(np.float32)
        got = ctx.df_points(ctx.to_device(pts), n, dims, 1, isoamd.DF_BRUTE).numpy()
        want = oracle.df_brute(oracle.normalize(pts, dims), dims, 1)
        assert np.array_equal(got.ravel(), want.ravel()), (dims, n)
