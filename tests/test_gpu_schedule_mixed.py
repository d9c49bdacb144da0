"""Schedules where one axis has a fixed-length FFT plan and the other a run-time plan: a context made
from the schedule that a context reports solves to the same bits, and the autotuner measures that
mix (what a context without a schedule runs) beside run-time plans along both axes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(pkg, scenes, W, H, Nz, seed, its=6):
    c = dict(width=W, height=H, num_planes=Nz, start_plane=1000.0, plane_stepsize=50.0, wavelength=0.633,
             resolution=2.0, num_inverse_iterations=its, regularization_param=0.01, regularization_TV_param=0.01,
             num_tv_iterations=5, mode=7)
    return pkg.make_params(**c), scenes.disks_scene(scenes.optics_of(c), 5, 2.0, 4.0, seed, 0.01)[0]


def _solve(pkg, p, holo, schedule=None):
    with pkg.SparseCompressiveHolo(p, schedule) as rec:
        rec.inverseReconstruct(holo)
        return rec.schedule(), rec.getVolume()


@pytest.mark.parametrize("W,H,mixed", [(272, 128, True), (128, 272, True), (208, 272, False), (128, 64, False)])
@pytest.mark.parametrize("path", [None, 0, 1])
def test_a_reported_schedule_gives_the_same_bits(pkg, scenes, gpu_available, W, H, mixed, path):
    p, holo = _case(pkg, scenes, W, H, 7, W + H)
    given = None if path is None else pkg.Schedule.make(fft_path=path, zchunk_fwd=3, zchunk_adj=2)
    got, vol = _solve(pkg, p, holo, given)
    if mixed:
        assert got["fft_path"] == (path or 0)
    again, vol2 = _solve(pkg, p, holo, pkg.Schedule.make(**{k: v for k, v in got.items() if k != "ms_per_iteration"}))
    assert again == got
    assert np.array_equal(vol.view(np.uint32), vol2.view(np.uint32))


def test_autotune_measures_the_mix(pkg, scenes, gpu_available):
    p, holo = _case(pkg, scenes, 272, 64, 4, 5)
    with pkg.SparseCompressiveHolo(p) as rec:
        default = rec.schedule()
    best, tried = pkg.autotune(p, holo, iterations=2)
    first = tried[0]
    assert all(first[k] == default[k] for k in ("fft_path", "max_radix", "zchunk_fwd", "zchunk_adj", "graphs"))
    assert {(t["fft_path"], t["max_radix"]) for t in tried} >= {(0, 16), (0, 8), (0, 4), (1, 16), (1, 8), (1, 4)}
    assert best.ms_per_iteration == min(t["ms_per_iteration"] for t in tried)
