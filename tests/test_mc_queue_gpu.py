"""Marching cubes where a wave's queue of crossings fills and wraps, a block's
isovalues take several rounds of 32, vertices fall on grid points, or the
brick is cut off by the grid: bit for bit against the oracle."""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


def _volume(kind, dims):
    rng = np.random.default_rng(dims[0])
    if kind == "noise":  # every edge crosses about a third of the isovalues
        return rng.random(dims).astype(np.float32)
    if kind == "levels":  # samples that equal isovalues: vertices on grid points
        return (rng.integers(0, 5, dims) / np.float32(4)).astype(np.float32)
    x, y, z = np.meshgrid(*[np.arange(n, dtype=np.float32) for n in dims], indexing="ij")
    return ((x + 2 * y + 3 * z) / np.float32(64)).astype(np.float32)


DIMS = [(2, 2, 2), (17, 5, 33), (16, 4, 16), (5, 18, 3), (33, 9, 6)]


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("kind", ["noise", "levels", "ramp"])
@pytest.mark.parametrize("compat", [True, False])
def test_one_isovalue(ctx, dims, kind, compat):
    v = _volume(kind, dims)
    d = ctx.to_device(v)
    flags = isoamd.MC_SORTED | (isoamd.COMPAT_MC if compat else 0)
    for iso in (0.25, 0.5, 0.73):
        out, n, st = ctx.mc_extract(d, dims, iso, flags)
        if compat:
            want, (active, total) = oracle.mc(v.ravel(), dims, np.float32(iso),
                                              ncls=oracle.mc_ncls_compat(*dims))
        else:
            xf = np.ascontiguousarray(v.transpose(2, 1, 0))
            want, (active, total) = oracle.mc(xf.ravel(), dims, np.float32(iso), interior=True)
        assert n == want.shape[0] and (st.active_cells, st.total_verts) == (active, total)
        assert n == 0 or np.array_equal(out.numpy()[:n], want)


@pytest.mark.parametrize("dims", [(17, 5, 33), (9, 18, 6)])
@pytest.mark.parametrize("kind", ["noise", "levels"])
@pytest.mark.parametrize("k", [33, 70])
def test_many_isovalues(ctx, dims, kind, k):
    # the distance fields of every isovalue's vertices: a vertex lost, doubled
    # into another isovalue or misplaced moves one of them
    v = _volume(kind, dims)
    isos = np.linspace(0.02, 0.98, k).astype(np.float32)
    if kind == "levels":
        isos[k // 2] = 0.5
    _, ids, st, fields = ctx.ism_volume(ctx.to_device(v), dims, isos, isoamd.EXTRACT_MC, 1, 32,
                                        isoamd.DF_LBVH, want_fields=True)
    got = fields.numpy()
    total = 0
    for i, iso in enumerate(isos):
        pts, _ = oracle.mc(v.ravel(), dims, iso, ncls=oracle.mc_ncls_compat(*dims))
        total += pts.shape[0]
        want = oracle.df_brute(oracle.normalize(pts, dims), dims, 1)
        assert np.array_equal(got[list(ids).index(i)].ravel(), want.ravel()), i
    assert st.total_points == total


@pytest.mark.parametrize("dims", [(2, 2, 2), (17, 5, 33), (9, 18, 6)])
@pytest.mark.parametrize("kind", ["noise", "levels"])
@pytest.mark.parametrize("k", [3, 33, 70])
def test_many_isovalues_of_the_approximation(ctx, dims, kind, k):
    v = _volume(kind, dims)
    isos = np.linspace(0.02, 0.98, k).astype(np.float32)
    isos[k // 2] = 0.5
    _, ids, st, fields = ctx.ism_volume(ctx.to_device(v), dims, isos, isoamd.EXTRACT_APPROX, 1, 32,
                                        isoamd.DF_LBVH, want_fields=True)
    got, total = fields.numpy(), 0
    for i, iso in enumerate(isos):
        cells = oracle.approx(v, iso)
        total += cells.shape[0]
        assert (i in list(ids)) == (cells.shape[0] > 0)
        if cells.shape[0]:
            want = oracle.df_brute(oracle.normalize(cells, dims), dims, 1)
            assert np.array_equal(got[list(ids).index(i)].ravel(), want.ravel()), i
    assert st.total_points == total
