"""The pair kernels' branches against the oracle, bit for bit: few and many
nonzero bins (listed or not), counts past 16 bits and past the 16-bit counters'
32,768, fields far from 0 (the subtracting form), odd bin counts, sizes around
a round of 8,192 voxels and around whole loads of 4, in both NMI modes."""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


def _fields(kind, F, seed):
    rng = np.random.default_rng(seed)
    if kind == "noise":  # nearly every bin takes part
        return rng.random((3, F)).astype(np.float32)
    if kind == "smooth":
        t = np.arange(F) / max(F, 2)
        return np.stack([np.abs(np.sin(9 * t) - 0.1 * k) for k in range(3)]).astype(np.float32)
    if kind == "far":  # |min| / range far above 1/16
        return (100.0 + rng.random((3, F))).astype(np.float32)
    f = np.zeros((3, F), np.float32)  # "flat": almost every voxel in one bin
    f[:, :: 97] = rng.random((3, len(range(0, F, 97)))).astype(np.float32)
    f[0, 0] = f[1, 0] = f[2, 0] = 1.0
    return f


@pytest.mark.parametrize("H", [17, 127, 128, 129, 255, 256])
@pytest.mark.parametrize("kind,F", [("noise", 40001), ("smooth", 8191), ("smooth", 8193),
                                    ("smooth", 5), ("far", 20003), ("flat", 300007),
                                    ("noise", 70000)])
def test_pair_counts_and_nmi_match_the_oracle(ctx, kind, F, H):
    f = _fields(kind, F, 7 * H + F)
    n = f.shape[0]
    d = ctx.to_device(f)
    smap, joint, rows, cols = ctx.hist_nmi(d, n, F, H, want_joint=True)
    got, j = smap.numpy(), joint.numpy()
    m64, _, _, _ = ctx.hist_nmi(d, n, F, H, flags=isoamd.COMPAT_HIST_CHUNKS)
    iv = [oracle.interval(x) for x in f]
    for a in range(n):
        for b in range(n):
            h = oracle.hist_pair(f[a], f[b], H, *iv[a], *iv[b])
            assert np.array_equal(j[a, b], h), (a, b)
            assert np.array_equal(rows.numpy()[a, b], h.sum(1)) and np.array_equal(
                cols.numpy()[a, b], h.sum(0))
            assert got[a, b] == np.float32(oracle.nmi_ref32(h, F)), (a, b)
            # the double form is rounded once to float; its sums are exact to 1e-12
            want = oracle.nmi_f64(h, F)
            assert abs(float(m64.numpy()[a, b]) - want) <= 2.0 ** -23 * abs(want) + 1e-9
    d.free()


def test_many_pairs_of_one_launch_match_single_pairs(ctx):
    # more pairs than workgroups at once, tiles with ragged edges, against the
    # same pairs alone
    rng = np.random.default_rng(3)
    n, F, H = 37, 9000, 200
    base = rng.random(F)
    f = np.stack([np.abs(base - 0.03 * k) for k in range(n)]).astype(np.float32)
    d = ctx.to_device(f)
    whole = ctx.hist_nmi(d, n, F, H)[0].numpy()
    for a, b in [(0, 36), (5, 8), (36, 36), (17, 18), (31, 32)]:
        pair = ctx.to_device(np.stack([f[a], f[b]]))
        one = ctx.hist_nmi(pair, 2, F, H)[0].numpy()
        assert whole[a, b] == one[0, 1] and whole[b, a] == one[1, 0] and whole[a, a] == one[0, 0]
        pair.free()
    d.free()
