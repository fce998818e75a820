"""Few pairs, cut into slices: with room for the slices' histograms and without
(the scratch of the entry point that allocates nothing), counts that fit 16 bits
in a slice but not in the sum, and counts that 16-bit counters hand on."""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [63, 128, 200, 256])
@pytest.mark.parametrize("n,F,kind", [(2, 200001, "noise"), (2, 500003, "flat"), (2, 70001, "flat"),
                                      (12, 50001, "noise"), (12, 131071, "flat"), (1, 98304, "flat")])
def test_slices_match_the_oracle(ctx, n, F, kind, H):
    rng = np.random.default_rng(F + H)
    f = rng.random((n, F)).astype(np.float32)
    if kind == "flat":  # nine of ten voxels in the first bin
        f[:, np.arange(F) % 10 != 0] = 0.0
    d = ctx.to_device(f)
    iv = [oracle.interval(x) for x in f]
    mins = ctx.to_device(np.array([v[0] for v in iv], np.float32))
    maxs = ctx.to_device(np.array([v[1] for v in iv], np.float32))
    for kw in ({}, {"mins": mins, "maxs": maxs, "no_alloc": True}):
        smap, joint, _, _ = ctx.hist_nmi(d, n, F, H, want_joint=True, **kw)
        got, j = smap.numpy(), joint.numpy()
        for a, b in {(0, 0), (0, n - 1), (n - 1, 0), (n // 2, n - 1)}:
            h = oracle.hist_pair(f[a], f[b], H, *iv[a], *iv[b])
            assert np.array_equal(j[a, b], h), (a, b, bool(kw))
            assert got[a, b] == np.float32(oracle.nmi_ref32(h, F)), (a, b, bool(kw))
    d.free()
