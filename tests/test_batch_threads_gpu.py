"""Batches of different bin counts (and so of different LDS sizes) from several
threads at a time, each with a context of its own: every map equals the one
computed alone."""
import threading

import numpy as np
import pytest

import isoamd

pytestmark = pytest.mark.gpu


def test_batches_of_several_threads():
    dims = (20, 18, 16)
    img = isoamd.gen_blobs(*dims, seed=4)
    isos = np.linspace(img.min(), img.max(), 8)[1:-1].astype(np.float32)
    bins = (256, 129, 64, 128)
    errors = []

    def work(H):
        try:
            with isoamd.Context(0) as c:
                d = c.to_device(img)
                alone, ids, _, _ = c.ism_volume(d, dims, isos, ds=2, H=H)
                m = ids.size
                want = alone.numpy()[:m * m].reshape(m, m)
                gate.wait()
                for flags in (isoamd.COMPAT_ALL, isoamd.COMPAT_ALL | isoamd.BATCH_GRAPH) * 40:
                    (got,), _ = c.ism_batch([d], [dims], [isos], ds=2, H=H, flags=flags)
                    assert np.array_equal(got[0], want), H
        except Exception as e:  # the test's own assertion runs in the main thread
            errors.append((H, repr(e)))
            gate.abort()

    gate = threading.Barrier(len(bins), timeout=60)
    threads = [threading.Thread(target=work, args=(H,)) for H in bins]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
