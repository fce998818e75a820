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


@pytest.mark.parametrize("dims", [(5, 3, 2), (9, 9, 9), (70, 66, 71), (130, 70, 129)])
def test_tree_walk_over_few_bricks_equals_brute(ctx, dims):
    # one, two and four layers of samples to a wave (at most 4,096 and 16,384
    # bricks of 4 x 4 x 4, and more), ragged at the grid's ends
    rng = np.random.default_rng(sum(dims))
    n = 3000
    pts = (rng.random((n, 3)) * np.array(dims)).astype(np.float32)
    d = ctx.to_device(pts)
    brute = ctx.df_points(d, n, dims, 1, isoamd.DF_BRUTE).numpy()
    for _ in range(2):  # the variants' first call, then the kept one
        tree = ctx.df_points(d, n, dims, 1, isoamd.DF_LBVH).numpy()
        assert np.array_equal(tree, brute)
    d.free()


@pytest.mark.parametrize("dims", [(161, 160, 157), (162, 161, 165), (255, 258, 130)])
def test_tree_walk_between_bricks_and_columns_equals_brute(ctx, dims):
    # from 4 to 32 bricks per wave the tuner also times a wave per brick, with two
    # and with four samples per lane; every variant runs in the first call
    rng = np.random.default_rng(sum(dims))
    n = 2000
    pts = (rng.random((n, 3)) * np.array(dims)).astype(np.float32)
    d = ctx.to_device(pts)
    brute = ctx.df_points(d, n, dims, 1, isoamd.DF_BRUTE).numpy()
    for _ in range(2):
        assert np.array_equal(ctx.df_points(d, n, dims, 1, isoamd.DF_LBVH).numpy(), brute)
    d.free()
