"""The histogram kernels' fixed-point binning rule, replayed in IEEE float32 on
the CPU: u = floor(RN(v R + RN(-mn R - M))) (or RN(RN(v - mn) R - M) for fields
far from 0), R = 2^16 RN(1 / step), step = RN((mx - mn) / H).  Wherever u's low
half is at most 65535 - 2 M, its high half must be the reference's bin
min(trunc(RN((v - mn) / step)), H - 1) (JointHistogram.cu:63-75, :127-129).
Values at and beside the bin edges, at mn and mx, and random values, for every
bin count's margin.  The fused multiply-add is one rounding of the float64
value: v R - c needs at most 48 + 24 bits, so it is taken exactly in integers.
"""
from fractions import Fraction

import numpy as np
import pytest

F = np.float32


def _round32(x: Fraction) -> np.float32:
    """A rational rounded once to float32 (nearest even)."""
    f = F(float(x))  # at most one ulp off: pick the nearest neighbour exactly
    best = None
    for c in (np.nextafter(f, F(-np.inf)), f, np.nextafter(f, F(np.inf))):
        d = abs(Fraction(float(c)) - x)
        even = (int(np.array(c).view(np.int32)) & 1) == 0
        if best is None or d < best[0] or (d == best[0] and even):
            best = (d, c)
    return best[1]


def _fma(a, b, c):
    return _round32(Fraction(float(a)) * Fraction(float(b)) + Fraction(float(c)))


def _reference_bin(v, mn, step, H):
    a = F(v - mn)
    return min(int(F(a / step)), H - 1)


def _rule(mn, mx, H):
    step = F(F(mx - mn) / F(H))
    q = F(F(1.0) / step)
    m = 33 * H // 2048 + 1
    r = F(q * F(65536))
    subtract = not (F(abs(mn) * q) <= F(H * 0.0625))
    nm = F(-m) if subtract else _fma(-mn, r, F(-m))
    return step, r, nm, 65535 - 2 * m, subtract


def _fixed(v, mn, r, nm, subtract):
    z = float(_fma(F(v - mn) if subtract else v, r, nm))
    return int(z) if z > 0 else 0


@pytest.mark.parametrize("offset", [0.0, 1e-3, 0.05, 40.0, -3.0])
@pytest.mark.parametrize("H", [1, 2, 17, 31, 62, 63, 64, 124, 125, 128, 200, 248, 249, 255, 256])
def test_fixed_point_bins_are_the_reference_bins(H, offset):
    rng = np.random.default_rng(1000 * H + int(abs(offset) * 100))
    fast = total = 0
    for _ in range(4):
        width = F(abs(rng.normal()) * 10.0 ** rng.integers(-3, 2) + 1e-4)
        mn = F(offset * (1 + rng.random()) * (float(width) if abs(offset) < 1 else 1.0))
        mx = F(mn + width)
        if not mx > mn:
            continue
        step, r, nm, top, subtract = _rule(mn, mx, H)
        edges = (float(mn) + rng.integers(0, H + 1, 40) * float(step)).astype(F)
        v = np.concatenate([edges, np.nextafter(edges, F(np.inf)), np.nextafter(edges, F(-np.inf)),
                            rng.uniform(mn, mx, 100).astype(F), [mn, mx]])
        for x in v[(v >= mn) & (v <= mx)]:
            u = _fixed(x, mn, r, nm, subtract)
            total += 1
            if (u & 0xffff) <= top:
                fast += 1
                assert u >> 16 == _reference_bin(x, mn, step, H), (x, mn, mx, H)
    assert 0 < fast <= total


def test_margin_exceeds_the_error_bound():
    # E = (4 + 1/16) H 2^-8 (1 + 2^-20) units of 2^-16 < M for every bin count
    for H in range(1, 257):
        E = Fraction(65, 16) * Fraction(H, 256) * (1 + Fraction(1, 2 ** 20))
        assert 33 * H // 2048 + 1 > E
