"""The fixed-point binning rule (replayed in test_fixed_point_bins.py) over wide
ranges: fields from 1e-4 to some thousands wide that start up to 5e4 from 0, at
every bin's edge and beside it, at both ends and at random values.  Where the rule
takes its fast path the bin is the reference's, and random values seldom leave it."""
import numpy as np
import pytest

from test_fixed_point_bins import F, _fixed, _reference_bin, _rule


@pytest.mark.parametrize("H", [1, 7, 64, 100, 128, 255, 256])
def test_wide_ranges(H):
    rng = np.random.default_rng(H)
    slow = total = cases = 0
    for _ in range(24):
        mn = F(rng.uniform(-50, 50) * 10.0 ** rng.integers(-3, 4))
        mx = F(mn + abs(rng.normal()) * 10.0 ** rng.integers(-4, 4))
        if not mx > mn:
            continue
        cases += 1
        step, r, nm, top, subtract = _rule(mn, mx, H)
        edges = (float(mn) + rng.integers(0, H + 1, 12) * np.float64(step)).astype(F)
        edges = np.concatenate([edges, np.nextafter(edges, F(np.inf)), np.nextafter(edges, F(-np.inf)),
                                [mn, mx]])
        # as many values as the range tells apart: a narrow range far from 0 has few
        values = rng.uniform(mn, mx, 40).astype(F)
        for v, random in ((edges, False), (values, True)):
            for x in v[(v >= mn) & (v <= mx)]:
                u = _fixed(x, mn, r, nm, subtract)
                fast = (u & 0xffff) <= top
                if fast:
                    assert u >> 16 == _reference_bin(x, mn, step, H), (x, mn, mx, H)
                if random and (float(mx) - float(mn)) > 2.0 ** 12 * H * np.spacing(max(abs(mn), abs(mx))):
                    total += 1
                    slow += not fast
    assert cases > 10 and total > 100 and slow < 0.01 * total + 3
