"""The NMI in double gives the same bits in every run and from both entry
points: pairs of exactly independent fields, whose NMI is the sums' rounding
alone, so that any other order of a sum shows.  Few bins (summed without a
list), listed ones, and more than a list holds; counts in LDS and past 16 bits."""
import numpy as np
import pytest

import isoamd

pytestmark = pytest.mark.gpu


def _fields(levels, scale, seed):
    """Six fields of levels values each, the even ones independent of the odd."""
    rng = np.random.default_rng(seed)
    r, c = (rng.integers(1, 9, levels) for _ in range(2))
    i = np.repeat(np.arange(levels), r)
    j = np.repeat(np.arange(levels), c)
    i, j = (a.ravel() for a in np.meshgrid(i, j, indexing="ij"))
    i, j = np.tile(i, scale), np.tile(j, scale)
    value = np.linspace(0, 1, levels).astype(np.float32)
    return np.stack([value[rng.permutation(levels)[i if q % 2 == 0 else j]] for q in range(6)])


@pytest.mark.parametrize("levels,H,scale", [(24, 48, 1), (40, 100, 1), (40, 256, 1), (52, 200, 1),
                                            (90, 128, 1), (110, 256, 1), (6, 256, 3000)])
def test_the_same_bits_every_time(ctx, levels, H, scale):
    f = _fields(levels, scale, levels + H)
    n, F = f.shape
    d = ctx.to_device(f)
    mins, maxs = ctx.field_interval(d, n, F)
    kw = dict(flags=isoamd.COMPAT_HIST_CHUNKS, mins=mins, maxs=maxs)
    first = ctx.hist_nmi(d, n, F, H, **kw)[0].numpy()
    odd = np.add.outer(np.arange(n), np.arange(n)) % 2 == 1
    assert np.all(np.abs(first[odd]) < 1e-12) and np.allclose(first[~odd], 1.0)
    for run in range(30):
        again = ctx.hist_nmi(d, n, F, H, no_alloc=run % 3 == 2, **kw)[0]
        assert np.array_equal(again.numpy().view(np.uint32), first.view(np.uint32)), run
        again.free()
    d.free()
