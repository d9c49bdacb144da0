"""A context holds a bounded number of captured graphs.  A batch of one geometry runs its items, each with
weights of its own and so with graphs of its own, on one context: with more graphs than are held, items
(repeated ones too, whose graphs have been dropped) still equal their single solves bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_many_weights_on_one_context(pkg, scenes, gpu_available):
    c = dict(width=32, height=32, num_planes=3, start_plane=1000.0, plane_stepsize=50.0, wavelength=0.633,
             resolution=2.0, num_inverse_iterations=40, regularization_TV_param=0.01, num_tv_iterations=3, mode=7)
    holo, _ = scenes.disks_scene(scenes.optics_of(dict(c, regularization_param=0.01)), 3, 2.0, 4.0, 8, 0.01)
    weights = [0.002 + 0.0004 * k for k in range(100)]
    order = weights + weights[:5]
    items = [dict(params=pkg.make_params(**dict(c, regularization_param=w)), holo=holo,
                  volume=np.empty((3, 32, 32), np.complex64)) for w in order]
    pkg.reconstruct_multi(items)
    graphs = 0
    for k, w in enumerate(weights):
        if 5 <= k < 97 and k % 10:
            continue
        with pkg.SparseCompressiveHolo(pkg.make_params(**dict(c, regularization_param=w))) as rec:
            rec.inverseReconstruct(holo)
            want = rec.getVolume()
            graphs = max(graphs, rec.counters()["graphs"])
        for j in range(len(order)):
            if order[j] == w:
                assert np.array_equal(items[j]["volume"].view(np.uint32), want.view(np.uint32)), (k, j)
    # (at most 12 of a context's graphs do not depend on the weights)
    assert 12 < graphs <= 512 and len(weights) * (graphs - 12) > 256
