"""The mode-7 prox's scan for zero rows, which a solve takes once its iterates are nearly all zero
and a wave has at least 64 rows: the same volume, bit for bit, as the form without it.  Waves of 63
rows take no scan; the rows per wave only regroup the sums that the solve's decisions read, and a
voxel's value depends on no sum.  Sizes put strips of 64 - 2 n_tv columns, the wrap of a frame
narrower than a wave, groups of 4 and 64 scanned rows and the rows' wrap at their edges, and map lines
of 16, 32 and 64 voxels.  The context's counters say that the scan ran, and that it skipped rows where
the weights leave any quiet.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntv", [0, 1, 2, 5, 6, 8, 10])
@pytest.mark.parametrize("W,H,rows,tv", [(32, 128, 128, 0.01), (128, 96, 67, 0.01), (272, 208, 208, 0.002),
                                         (336, 400, 101, 0.05), (1280, 192, 64, 0.02), (2064, 128, 128, 0.02)])
def test_scan_keeps_the_volume(pkg, scenes, gpu_available, ntv, W, H, rows, tv):
    c = dict(width=W, height=H, num_planes=4, start_plane=1000.0, plane_stepsize=50.0, wavelength=0.633,
             resolution=2.0, num_inverse_iterations=40, regularization_param=0.1, regularization_TV_param=tv,
             num_tv_iterations=ntv, mode=7)
    holo, _ = scenes.disks_scene(scenes.optics_of(c), 1, 2.0, 3.0, 900 + W + ntv, 0.002)
    vols, stats, counts = [], [], []
    for r in (63, rows):
        with pkg.SparseCompressiveHolo(pkg.make_params(**c), pkg.Schedule.make(prox_rows=r)) as rec:
            stats.append(rec.inverseReconstruct(holo))
            vols.append(rec.getVolume())
            counts.append(rec.counters())
    assert counts[0]["prox_scan"] == 0
    if W > 32:
        assert counts[1]["prox_scan"] > 0
    if tv >= 0.02:
        assert counts[1]["scan_skipped"] > 1000
    assert list(stats[0]["restarts"]) == list(stats[1]["restarts"])
    sp = np.array(stats[1]["sparsity_it"][:-1])
    assert W == 32 or ((sp > 0) & (sp < 2e-3)).any(), sp  # the line below which y is scanned
    assert np.array_equal(vols[0].view(np.uint64), vols[1].view(np.uint64))
    np.testing.assert_allclose(stats[1]["f"], stats[0]["f"], rtol=1e-5)
