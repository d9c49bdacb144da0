"""The scalars of an iteration reach the host with a number and a check word, and a block that is not the
iteration's, or not whole, is not used: with RIHVR_TEST_LATE_SCALARS the host finds the block published
before in the given iterations (of the first iteration too, where that is the solve before's or none; in
odd iterations only the first half of that block), and the solve must come out
the same bit for bit, volume, objectives and decisions, with every late block counted.  Without it
none is late.  With graphs and without, in the modes that hand scalars over, and with backtracks in
the same iterations."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solves(pkg, c, holos, graphs, late, backtracks=0):
    env = {"RIHVR_GRAPHS": str(int(graphs)), "RIHVR_TEST_LATE_SCALARS": str(late),
           "RIHVR_TEST_BACKTRACKS": str(backtracks)}
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        with pkg.SparseCompressiveHolo(pkg.make_params(**c)) as rec:
            out = [(rec.inverseReconstruct(h), rec.getVolume()) for h in holos]
            return out, rec.counters()
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("late,backtracks", [(0b1, 0), (0b110101, 0), (0b1100, 0b0100)])
@pytest.mark.parametrize("W,H,Nz,tv,mode", [(64, 64, 8, 0.01, 7), (272, 48, 3, 0.01, 7), (48, 64, 5, 0.0, 7),
                                            (64, 64, 6, 0.01, 6)])
def test_a_late_block_changes_nothing(pkg, scenes, gpu_available, W, H, Nz, tv, mode, late, backtracks, graphs):
    c = dict(width=W, height=H, num_planes=Nz, start_plane=1000.0, plane_stepsize=50.0, wavelength=0.633,
             resolution=2.0, num_inverse_iterations=8, regularization_param=0.01, regularization_TV_param=tv,
             num_tv_iterations=5, mode=mode)
    holos = [scenes.disks_scene(scenes.optics_of(c), 4, 2.0, 4.0, 60 + k, 0.01)[0] for k in range(2)]
    want, n0 = _solves(pkg, c, holos, graphs, 0, backtracks)
    got, n1 = _solves(pkg, c, holos, graphs, late, backtracks)
    assert n0["late_scalars"] == 0
    assert n1["late_scalars"] >= 2 * bin(late).count("1")
    for (sw, vw), (sg, vg) in zip(want, got):
        assert np.array_equal(vg.view(np.uint32), vw.view(np.uint32))
        for k in ("f", "ratio", "lim", "restart_sum"):
            np.testing.assert_array_equal(sg[k], sw[k])
        assert list(sg["backtracks"]) == list(sw["backtracks"])
        assert list(sg["restarts"]) == list(sw["restarts"])
