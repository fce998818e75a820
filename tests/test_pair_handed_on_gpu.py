"""More pairs than workgroups at a time, none cut up, whose 16-bit counters hand
on to 32-bit histograms that share cache lines with their neighbours' (an odd
number of bins): every pair's counts against the oracle."""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [131, 129])
def test_counts_handed_on_in_many_pairs(ctx, H):
    n, F = 26, 90001
    rng = np.random.default_rng(H)
    f = rng.random((n, F)).astype(np.float32)
    f[:, np.arange(F) % 5 != 0] = 0.0  # past 65,536 in the first bin
    f[::2, np.arange(F) % 10 == 5] = 1.0
    d = ctx.to_device(f)
    smap, joint, _, _ = ctx.hist_nmi(d, n, F, H, want_joint=True)
    got, j = smap.numpy(), joint.numpy()
    iv = [oracle.interval(x) for x in f]
    for a in range(n):
        for b in range(a, n):
            h = oracle.hist_pair(f[a], f[b], H, *iv[a], *iv[b])
            assert np.array_equal(j[a, b], h) and np.array_equal(j[b, a], h.T), (a, b)
            assert got[a, b] == np.float32(oracle.nmi_ref32(h, F)), (a, b)
    d.free()
