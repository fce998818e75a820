"""Values past the interval that a caller gives: their pair's map entry is
unspecified, but the counts of the bins before the interval's last are right, and
what the context keeps is untouched, so the next call's results are right.  The
second field alone exceeds the interval, by fewer bins than a row of the counts
has room for."""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


def _normal(ctx, H, flags, no_alloc):
    rng = np.random.default_rng(H)
    n, F = 3, 50001
    f = rng.random((n, F)).astype(np.float32)
    d = ctx.to_device(f)
    mins, maxs = ctx.field_interval(d, n, F)
    smap, joint, _, _ = ctx.hist_nmi(d, n, F, H, flags=flags, mins=mins, maxs=maxs, want_joint=True,
                                     no_alloc=no_alloc)
    iv = [oracle.interval(x) for x in f]
    for a in range(n):
        for b in range(n):
            h = oracle.hist_pair(f[a], f[b], H, *iv[a], *iv[b])
            assert np.array_equal(joint.numpy()[a, b], h)
            if flags & isoamd.COMPAT_NMI32:
                assert smap.numpy()[a, b] == np.float32(oracle.nmi_ref32(h, F))
    d.free()


@pytest.mark.parametrize("no_alloc", [False, True])
@pytest.mark.parametrize("flags", [isoamd.COMPAT_ALL, isoamd.COMPAT_HIST_CHUNKS])
@pytest.mark.parametrize("kind,H,top", [("flat", 200, 1.0525), ("noise", 130, 1.9), ("noise", 40, 3.0)])
def test_values_past_the_interval_leave_the_rest_alone(ctx, kind, H, top, flags, no_alloc):
    F = 400003
    rng = np.random.default_rng(H)
    if kind == "flat":  # one bin of the last row, past 32,768 counts
        x = np.full(F, 0.999, np.float32)
        y = np.full(F, top, np.float32)
        x[:3] = 0.0, 0.5, 0.25
        y[:3] = 0.0, 0.5, 0.25
    else:
        x = rng.random(F).astype(np.float32)
        y = (rng.random(F) * top).astype(np.float32)
    assert y.max() * H < (256 if H > 128 else 128)
    d = ctx.to_device(np.stack([x, y]))
    mins, maxs = ctx.to_device(np.zeros(2, np.float32)), ctx.to_device(np.ones(2, np.float32))
    _, joint, _, _ = ctx.hist_nmi(d, 1, F, H, multi=True, flags=flags, mins=mins, maxs=maxs,
                                  want_joint=True, no_alloc=no_alloc)
    h = oracle.hist_pair(x[y < 1], y[y < 1], H, 0.0, 1.0, 0.0, 1.0)
    assert np.array_equal(joint.numpy()[0, 0][:, :H - 1], h[:, :H - 1])
    d.free()
    _normal(ctx, H, flags, no_alloc)
