"""The float-order NMI when its chains' inputs do not fit one launch, with many
counts past 16 bits, and over captured batches that share the context's room for
them: the oracle's values and the uncaptured batch's, bit for bit."""
import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mib", ["1", "8", None])
@pytest.mark.parametrize("H", [100, 128, 131, 256])
def test_many_large_counts(ctx, monkeypatch, H, mib):
    # six plateaus of about 80,000 voxels each, a few voxels between them
    if mib:
        monkeypatch.setenv("ISO_NMI_CHAIN_MIB", mib)
    rng = np.random.default_rng(H)
    n, F = 5, 500009
    f = rng.integers(0, 6, (n, F)).astype(np.float32) / 5
    f[1] = f[0]
    f[3] = 1 - f[0]
    f[:, ::1001] = rng.random((n, len(range(0, F, 1001))), dtype=np.float32)
    d = ctx.to_device(f)
    iv = [oracle.interval(x) for x in f]
    got = ctx.hist_nmi(d, n, F, H)[0].numpy()
    for a in range(n):
        for b in range(n):
            h = oracle.hist_pair(f[a], f[b], H, *iv[a], *iv[b])
            assert (h > 65535).sum() == (6 if a == b or {a, b} <= {0, 1, 3} else 0), (a, b)
            assert got[a, b] == np.float32(oracle.nmi_ref32(h, F)), (a, b)
    d.free()


@pytest.mark.parametrize("H", [64, 200])
def test_captured_batches_share_the_room(monkeypatch, H):
    def isos(v, k):
        return np.linspace(v.min(), v.max(), k + 2)[1:-1].astype(np.float32)

    with isoamd.Context(0) as c:
        layouts = []
        for i, (dims, k) in enumerate((((24, 20, 16), 5), ((40, 32, 28), 24), ((20, 20, 36), 9))):
            img = isoamd.gen_blobs(*dims, seed=i + 1)
            layouts.append((c.to_device(img), dims, isos(img, k)))

        def run(i, flags):
            v, dims, s = layouts[i]
            (got,), st = c.ism_batch([v], [dims], [s], ds=2, H=H, flags=isoamd.COMPAT_ALL | flags)
            return got, st.graph_replays

        # 0's graph, then a layout for which the room grows, then 0 again; the
        # launches of several rounds of pairs as well
        for mib in (None, "4"):
            if mib:
                monkeypatch.setenv("ISO_NMI_CHAIN_MIB", mib)
            for i in (0, 0, 1, 0, 2, 1, 0, 2, 2):
                got, replays = run(i, isoamd.BATCH_GRAPH)
                want, _ = run(i, 0)
                assert np.array_equal(got[0], want[0]) and list(got[1]) == list(want[1]), (i, mib)
            assert replays > 0
