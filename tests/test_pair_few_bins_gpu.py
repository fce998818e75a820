"""Joint counts and NMI with few bins per axis and at the widths of a row of the
LDS histogram, in LDS and merged from slices, against the oracle."""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [1, 2, 3, 8, 16, 33, 64, 126, 128, 130])
@pytest.mark.parametrize("n,F", [(3, 9001), (2, 150001)])
def test_few_bins_match_the_oracle(ctx, n, F, H):
    rng = np.random.default_rng(H + F)
    f = rng.random((n, F)).astype(np.float32)
    f[1] = 0.3 * f[0] + 0.7 * f[1]
    d = ctx.to_device(f)
    iv = [oracle.interval(x) for x in f]
    for flags in (isoamd.COMPAT_ALL, isoamd.COMPAT_HIST_CHUNKS):
        smap, joint, rows, cols = ctx.hist_nmi(d, n, F, H, flags=flags, want_joint=True)
        got, j, r, c = (x.numpy() for x in (smap, joint, rows, cols))
        for a in range(n):
            for b in range(n):
                h = oracle.hist_pair(f[a], f[b], H, *iv[a], *iv[b])
                assert np.array_equal(j[a, b], h), (a, b)
                assert np.array_equal(r[a, b], h.sum(1)) and np.array_equal(c[a, b], h.sum(0))
                if flags & isoamd.COMPAT_NMI32:
                    assert got[a, b] == np.float32(oracle.nmi_ref32(h, F)), (a, b)
                elif H > 1:
                    want = oracle.nmi_f64(h, F)
                    assert abs(float(got[a, b]) - want) <= 2.0 ** -23 * abs(want) + 1e-9
    d.free()
