"""Marching cubes of volumes with NaN samples: the entry points with and
without cell statistics take the same edges, those of a replay on the CPU.

The rule: a wave's 16 x 4 grid points (16 along the memory-fast axis) look at an
isovalue if one of their cells has a corner below it and one at or above it, NaN
corners aside; they then take every edge of theirs whose ends compare
differently with it, an edge from a sample below the isovalue to a NaN among
them.
"""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu
F = np.float32


def _volume(kind, dims):
    rng = np.random.default_rng(dims[0] + dims[2])
    v = rng.random(dims).astype(F)
    if kind != "noise":
        x, y, z = np.meshgrid(*[np.linspace(0, 1, n) for n in dims], indexing="ij")
        v = (np.abs(np.sin(5 * x + 3 * y) * np.cos(4 * z)) + 0.01 * v).astype(F)
    if kind == "half":
        v[dims[0] // 2:] = np.nan
    else:
        v[rng.random(dims) < 0.1] = np.nan
    return v


def _count(s, ncls, nc, iso, zfast):
    """Vertices and active cells of the sample array s[x, y, z] with nc cells per axis."""
    n = [c + 1 for c in nc]  # grid points
    at = [np.minimum(np.arange(q + 1), g - 1) for q, g in zip(n, s.shape)]
    p = s[np.ix_(*at)]
    gx, gy = s.shape[:2]
    cell = np.zeros([q + 1 for q in n], bool)  # cell[x + 1, y + 1, z + 1]
    x, y, z = np.meshgrid(*[np.arange(c) for c in nc], indexing="ij")
    cell[1:nc[0] + 1, 1:nc[1] + 1, 1:nc[2] + 1] = x + gx * (y + gy * z) < ncls

    def c(dx, dy, dz):
        return cell[1 - dx:n[0] + 1 - dx, 1 - dy:n[1] + 1 - dy, 1 - dz:n[2] + 1 - dz]

    xp, xm = c(0, 0, 0) | c(0, 0, 1), c(0, 1, 0) | c(0, 1, 1)
    yp, ym = c(1, 0, 0) | c(1, 0, 1), c(0, 0, 0) | c(0, 0, 1)
    zp = c(0, 0, 0) | c(1, 0, 0) | c(0, 1, 0) | c(1, 1, 0)

    def corner(i, j, k):
        return p[i:n[0] + i, j:n[1] + j, k:n[2] + k]

    corners = np.stack([corner(i, j, k) for i in (0, 1) for j in (0, 1) for k in (0, 1)])
    below = (corners < iso).any(0)
    above = (corners >= iso).any(0)
    hit = below & above & (xp | xm | yp | ym | zp)
    wave = (1, 4, 16) if zfast else (16, 4, 1)
    seen = np.zeros_like(hit)
    for i in range(0, n[0], wave[0]):
        for j in range(0, n[1], wave[1]):
            for k in range(0, n[2], wave[2]):
                b = np.s_[i:i + wave[0], j:j + wave[1], k:k + wave[2]]
                seen[b] = hit[b].any()
    total = 0
    f0 = corner(0, 0, 0)
    for axis, plus, minus in ((0, xp, xm), (1, yp, ym), (2, zp, np.zeros_like(zp))):
        f1 = corner(*(int(a == axis) for a in range(3)))
        cross = seen & ((f0 < iso) != (f1 < iso)) & (plus | minus)
        base = np.arange(n[axis], dtype=F).reshape([-1 if a == axis else 1 for a in range(3)])
        with np.errstate(all="ignore"):
            vp = base + (iso - f0) / (f1 - f0)
            vm = (base + F(1)) - (iso - f1) / (f0 - f1)
        at_grid = ((vp == base) | (vp == base + 1) | (vm == base) | (vm == base + 1)) & cross
        assert not at_grid.any()  # none to be counted once for several edges
        total += int((cross & plus).sum()) + int((cross & minus & ~(plus & (vp == vm))).sum())
    inside = (corners < iso).sum(0)
    return total, int((seen & c(0, 0, 0) & (inside > 0) & (inside < 8)).sum())


@pytest.mark.parametrize("compat", [True, False])
@pytest.mark.parametrize("kind", ["noise", "smooth", "half"])
@pytest.mark.parametrize("dims", [(20, 20, 20), (33, 9, 40), (5, 18, 17)])
def test_nan_samples_same_edges_in_every_form(ctx, dims, kind, compat):
    v = _volume(kind, dims)
    isos = np.array([0.113, 0.317, 0.529, 0.871], F)
    flags = isoamd.COMPAT_MC if compat else 0
    s = v.ravel().reshape(dims[::-1]).transpose(2, 1, 0) if compat else v
    nc = dims if compat else tuple(n - 1 for n in dims)
    ncls = oracle.mc_ncls_compat(*dims) if compat else 1 << 60
    d = ctx.to_device(v)
    _, ids, st, fields = ctx.ism_volume(d, dims, isos, isoamd.EXTRACT_MC, 1, 32, isoamd.DF_BRUTE,
                                        flags=flags | isoamd.COMPAT_NMI32, want_fields=True)
    got, total, row = fields.numpy(), 0, 0
    for i, iso in enumerate(isos):
        out, n, cells = ctx.mc_extract(d, dims, float(iso), flags)
        assert (n, cells.active_cells) == _count(s, ncls, nc, iso, not compat), iso
        total += n
        if n:
            want = ctx.df_points(out, n, dims, 1, isoamd.DF_BRUTE).numpy()
            assert list(ids)[row] == i and np.array_equal(got[row].ravel(), want.ravel())
            row += 1
    assert st.total_points == total and row == st.n_nonempty
    d.free()
