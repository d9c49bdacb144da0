"""The mode-7 prox's dense form, which a solve takes while its iterates are mostly non-zero:
against the FP32 oracle, at every number of TV iterations it is built for, strip and chunk edges
(a wave's strip is 64 - 2 n_tv columns, W from 16 up wraps inside one strip; chunks of 1, 7 and
all rows) and across the change between the two forms as a solve's iterates thin out.

Tolerances are those of the solver's other parity tests: 1e-4 relative L2 on a solve's volume,
1e-4 relative on its objectives (the reductions), equal decisions.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / max(np.linalg.norm(np.asarray(b)), 1e-30))


def cfg(W, H, Nz, its, reg, ntv):
    return dict(width=W, height=H, num_planes=Nz, start_plane=1000.0, plane_stepsize=50.0, wavelength=0.633,
                resolution=2.0, num_inverse_iterations=its, regularization_param=reg, regularization_TV_param=0.01,
                num_tv_iterations=ntv, mode=7)


def check(pkg, orc, scenes, c, rows, seed):
    holo, _ = scenes.disks_scene(scenes.optics_of(c), 4, 2.0, 4.0, seed, 0.01)
    sch = None if rows is None else pkg.Schedule.make(prox_rows=rows)
    with pkg.SparseCompressiveHolo(pkg.make_params(**c), sch) as rec:
        st = rec.inverseReconstruct(holo)
        vol = rec.getVolume()
    ref, _, _, rst = orc.solve(orc.make_params(**c), holo, None, "f32")
    assert rel(vol, ref) < 1e-4, rel(vol, ref)
    assert list(st["backtracks"]) == list(rst["backtracks"])
    assert list(st["restarts"]) == list(rst["restarts"])
    np.testing.assert_allclose(st["f"], rst["f"], rtol=1e-4)
    return st


@pytest.mark.parametrize("ntv", range(11))
@pytest.mark.parametrize("W,H,rows", [(16, 32, None), (64, 16, 1), (112, 48, 7), (272, 64, 64)])
def test_dense_prox_solves_to_the_oracle(pkg, orc, scenes, gpu_available, ntv, W, H, rows):
    # no L1 weight: all non-zero.  (Without a TV iteration either, one step would reach a zero
    # residual, A A^T being Nz I, and the next step's ratio test would divide rounding errors.)
    st = check(pkg, orc, scenes, cfg(W, H, 3, 5, 0.0 if ntv else 0.002, ntv), rows, 300 + W + ntv)
    assert st["sparsity"] > 0.05


def test_solve_that_thins_out(pkg, orc, scenes, gpu_available):
    st = check(pkg, orc, scenes, cfg(128, 96, 6, 40, 0.05, 5), None, 17)
    sp = st["sparsity_it"]
    assert sp[0] > 0.05 > sp[-1], sp  # the iterates cross the line between the two forms
