"""The tree walk's forms one by one against brute force: waves that stay and a
wave per brick between 4 and 32 bricks for each that fits the chip, with two and
four samples per lane, and over few bricks one, two and four layers of samples to
a wave.  The autotuner's first call shows one form's fields only, the one that ran
last, so each is forced here."""
import numpy as np
import pytest

import isoamd

pytestmark = pytest.mark.gpu

WAVES = 8192  # on 256 CUs


def _bricks(dims, sets, layers):
    x, y, z = dims
    return -(-x // 4) * -(-y // 4) * -(-z // layers) * sets


def _points(dims, n):
    rng = np.random.default_rng(sum(dims) + n)
    p = rng.random((n, 3)) * np.array(dims)
    p[: n // 4] = p[: n // 4] * 0.05 + 0.3 * np.array(dims)  # a cluster
    return p.astype(np.float32)


@pytest.mark.parametrize("stay", ["4", "32"])
@pytest.mark.parametrize("dims,spl", [((161, 160, 157), "2"), ((162, 161, 165), "2"),
                                      ((255, 258, 130), "2"), ((255, 258, 130), "4"),
                                      ((301, 270, 205), "4")])
def test_waves_per_brick_and_waves_that_stay(ctx, monkeypatch, dims, spl, stay):
    layers = 4 * int(spl)
    assert 4 * WAVES <= _bricks(dims, 1, layers) < 32 * WAVES
    n = 3000
    pts = _points(dims, n)
    d = ctx.to_device(pts)
    want = ctx.df_points(d, n, dims, 1, isoamd.DF_BRUTE).numpy()
    monkeypatch.setenv("ISO_DF_LEAF", "64")
    monkeypatch.setenv("ISO_DF_SPL", spl)
    monkeypatch.setenv("ISO_DF_STAY", stay)
    assert np.array_equal(ctx.df_points(d, n, dims, 1, isoamd.DF_LBVH).numpy(), want)
    d.free()


# at most 4,096, at most 16,384 and more bricks of 4 x 4 x 4, sizes at both lines
@pytest.mark.parametrize("dims", [(5, 3, 2), (64, 64, 64), (65, 64, 64), (70, 66, 71), (103, 102, 101),
                                  (128, 64, 128), (128, 128, 64), (129, 64, 128), (130, 70, 129)])
@pytest.mark.parametrize("leaf", ["64", "24"])
def test_layers_of_samples_over_few_bricks(ctx, monkeypatch, dims, leaf):
    n = 3000
    pts = _points(dims, n)
    d = ctx.to_device(pts)
    want = ctx.df_points(d, n, dims, 1, isoamd.DF_BRUTE).numpy()
    monkeypatch.setenv("ISO_DF_LEAF", leaf)
    monkeypatch.setenv("ISO_DF_SPL", "1")
    assert np.array_equal(ctx.df_points(d, n, dims, 1, isoamd.DF_LBVH).numpy(), want)
    d.free()


@pytest.mark.parametrize("stay,spl", [("4", "2"), ("32", "2"), ("32", "4"), ("4", "1")])
@pytest.mark.parametrize("pool", ["0", "1"])
def test_forms_over_several_sets(ctx, monkeypatch, stay, spl, pool):
    dims, ds = (100, 92, 84), 1
    img = isoamd.gen_blobs(*dims, seed=8)
    isos = np.linspace(img.min(), img.max(), 22)[1:-1].astype(np.float32)
    d = ctx.to_device(img)
    _, _, st, want = ctx.ism_volume(d, dims, isos, isoamd.EXTRACT_MC, ds, 32, isoamd.DF_BRUTE,
                                    want_fields=True)
    for k, v in (("LEAF", "64"), ("SPL", spl), ("STAY", stay), ("POOL_LEAVES", pool)):
        monkeypatch.setenv("ISO_DF_" + k, v)
    _, _, _, got = ctx.ism_volume(d, dims, isos, isoamd.EXTRACT_MC, ds, 32, isoamd.DF_LBVH,
                                  want_fields=True)
    m = st.n_nonempty
    assert m >= 15 and np.array_equal(got.numpy()[:m], want.numpy()[:m])
