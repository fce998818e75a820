"""A NaN among the isovalues has an empty surface and leaves the others as they
are, wherever it stands and in every entry point that takes a list."""
import numpy as np
import pytest

import isoamd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extractor", [isoamd.EXTRACT_MC, isoamd.EXTRACT_APPROX])
@pytest.mark.parametrize("at", [(3,), (0,), (1,), (0, 2, 5)])
def test_nan_isovalue_is_an_empty_surface(ctx, extractor, at):
    dims = (40, 36, 28)
    img = isoamd.gen_blobs(*dims, seed=3)
    plain = np.array([0.1, 0.3, 0.6], np.float32)
    isos, keep = list(plain), []
    for i in at:
        isos.insert(i, np.nan)
    isos = np.array(isos, np.float32)
    keep = np.flatnonzero(~np.isnan(isos))
    d = ctx.to_device(img)
    want_map, want_ids, want, want_f = ctx.ism_volume(d, dims, plain, extractor, 2, 64,
                                                      want_fields=True)
    smap, ids, st, f = ctx.ism_volume(d, dims, isos, extractor, 2, 64, want_fields=True)
    m = want.n_nonempty
    assert m == 3 and st.n_nonempty == m and st.total_points == want.total_points
    assert list(ids) == list(keep[want_ids])
    assert np.array_equal(f.numpy()[:m], want_f.numpy()[:m])
    want_map = want_map.numpy()[:m * m].reshape(m, m)
    assert np.array_equal(smap.numpy()[:m * m].reshape(m, m), want_map)
    (got,), _ = ctx.ism_batch([d], [dims], [isos], extractor, 2, 64)
    assert list(got[1]) == list(ids) and np.array_equal(got[0], want_map)
