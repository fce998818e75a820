"""A number that the autotuner keeps for the tree walk means one form, whatever
the sizes that it was measured with: a frozen tuner takes it for other sizes."""
import re

import numpy as np
import pytest

import isoamd

pytestmark = pytest.mark.gpu


def test_a_variants_number_means_one_form():
    # sizes with a wave per brick among the candidates and without
    with isoamd.Context(0) as c:
        for dims in ((40, 40, 40), (162, 161, 165), (255, 258, 130)):
            rng = np.random.default_rng(sum(dims))
            pts = (rng.random((2000, 3)) * np.array(dims)).astype(np.float32)
            d = c.to_device(pts)
            c.df_points(d, 2000, dims, 1, isoamd.DF_LBVH)
            d.free()
        lines = [s for s in c.tuning() if s.startswith("lbvh")]
    assert len(lines) == 3
    forms, timed = set(), []
    for s in lines:
        names, times = re.fullmatch(r"lbvh [^{]*\{(.*)\} \[key \w+\]:(.*) \| again .*", s).groups()
        forms.add(names)
        timed.append({int(v) for v in re.findall(r"(\d+): \d", times)})
    assert len(forms) == 1 and "or" not in forms.pop().split(" ")
    assert timed[0] == {8, 9, 10, 11}  # sorted points; 9: leaves of 48 points
    assert timed[1] == timed[2] == {8, 10, 11, 12}  # 12: by brick in its place
