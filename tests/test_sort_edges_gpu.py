"""The radix sort and the scans at the edges of their tiles, through the
sorted marching-cubes vertices: every tile size, the last bit of a key, and
vertices that no 64-bit key holds."""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("items", [None, "4", "8"])
@pytest.mark.parametrize("dims", [(2, 2, 2), (3, 63, 64), (64, 127, 31), (128, 64, 65), (257, 3, 129)])
def test_sorted_vertices(ctx, monkeypatch, dims, items):
    if items:
        monkeypatch.setenv("ISO_SORT_ITEMS", items)
    v = np.random.default_rng(dims[1]).random(dims).astype(np.float32)
    v[v > 0.98] = 0.5  # some vertices on grid points
    d = ctx.to_device(v)
    out, n, _ = ctx.mc_extract(d, dims, 0.5, isoamd.COMPAT_MC | isoamd.MC_SORTED)
    want, _ = oracle.mc(v.ravel(), dims, np.float32(0.5), ncls=oracle.mc_ncls_compat(*dims))
    assert n == want.shape[0] and (n == 0 or np.array_equal(out.numpy()[:n], want))


def test_vertices_without_a_key(ctx):
    # infinite samples of both signs side by side: t = inf / inf
    dims = (12, 11, 10)
    v = np.random.default_rng(5).random(dims).astype(np.float32)
    v[3, 4, 5], v[3, 4, 6], v[7, 7, 7] = np.inf, -np.inf, np.inf
    d = ctx.to_device(v)
    out, n, _ = ctx.mc_extract(d, dims, 0.5, isoamd.MC_SORTED)
    got = out.numpy()[:n]
    plain, m, _ = ctx.mc_extract(d, dims, 0.5, 0)
    raw = plain.numpy()[:m]
    assert n == m
    bits = raw.view(np.uint32)
    order = np.lexsort((bits[:, 2], bits[:, 1], bits[:, 0]))
    assert np.isnan(raw).any()
    assert np.array_equal(got.view(np.uint32), bits[order])


def test_large_tiles_and_scans(ctx):
    # 2.2M vertices: 16 keys per lane; blocks past the one-launch scan
    dims = (300, 128, 128)
    v = isoamd.gen_blobs(*dims, nblobs=8, noise=0.6, seed=9)
    iso = np.float32(np.median(v))
    d = ctx.to_device(v)
    out, n, _ = ctx.mc_extract(d, dims, float(iso), isoamd.COMPAT_MC | isoamd.MC_SORTED)
    want, _ = oracle.mc(v.ravel(), dims, iso, ncls=oracle.mc_ncls_compat(*dims))
    assert n == want.shape[0] and n > 2_200_000
    assert np.array_equal(out.numpy()[:n], want)
