"""Ingest and equalised isovalues at the edges of their tiles, rounds and
counters, against the oracle bit for bit."""
import ctypes as C

import numpy as np
import pytest

import isoamd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (63, 2, 65), (64, 3, 64), (65, 1, 63), (128, 40, 129),
                                  (3, 5000, 2), (200, 1, 1), (1, 1, 300)])
def test_ingest_tile_edges(ctx, dims):
    X, Y, Z = dims
    file = np.random.default_rng(X + Z).standard_normal(X * Y * Z).astype(np.float32)
    img, lo, hi = ctx.volume_ingest(ctx.to_device(file), dims, -1.0, 1.0)
    want, wlo, whi = oracle.ingest(file, dims, -1.0, 1.0)
    assert np.array_equal(img.numpy(), want) and (lo, hi) == (wlo, whi)


def _values(kind, n):
    rng = np.random.default_rng(n)
    v = rng.random(n).astype(np.float32)
    if kind == "constant":
        v[:] = 0.25
    elif kind == "two":  # plateaus with a few values between
        v = np.where(v < 0.6, np.float32(0), np.where(v < 0.99, np.float32(1), v))
    elif kind == "few":  # whole numbers
        v = np.floor(v * 11).astype(np.float32)
    elif kind == "last":  # everything in the last bin but one value
        v[:] = 1.0
        v[0] = 0.0
    elif kind == "beyond":  # values outside the range given, and not finite
        v = v * 3 - 1
        v[:: 97] = np.inf
        v[1:: 97] = -np.inf
    return v


@pytest.mark.parametrize("k", [1, 7, 256, 70000])
@pytest.mark.parametrize("kind", ["spread", "constant", "two", "few", "last", "beyond"])
def test_equalised_values(ctx, kind, k):
    # a round is 4,096 voxels, an epoch 32,768; 9,000,001 gives each of 256
    # workgroups more than one epoch (counters hand on their half)
    for n in (1, 3, 4095, 4097, 32769, 262147, 9000001):
        v = _values(kind, n)
        lo, hi = (0.0, 1.0) if kind == "beyond" else (float(v.min()), float(v.max()))
        got = ctx.equalized_isovalues(ctx.to_device(v), lo, hi, k)
        # int(inf) is undefined in the oracle's C++ (x86: INT_MIN); the device's
        # saturates, as any value far outside the range does
        want = oracle.equalized_isovalues(np.clip(v, -1000, 1000), lo, hi, k)
        assert np.array_equal(got, want, equal_nan=True), (n, kind, k)


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_equalised_unaligned_image(ctx, shift):
    v = _values("spread", 50003)
    d = ctx.to_device(v)
    n, k = v.size - shift, 16
    out = np.empty(k, np.float32)
    st = isoamd.lib().iso_equalized_isovalues(ctx.h, C.c_void_p(d.ptr + 4 * shift), n, 0.0, 1.0, k,
                                              out.ctypes.data_as(C.c_void_p))
    assert st == 0
    assert np.array_equal(out, oracle.equalized_isovalues(v[shift:], 0.0, 1.0, k))
