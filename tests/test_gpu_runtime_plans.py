"""The transforms of run-time length against the FP32 oracle: every radix of the plans and primes
above them, alone and repeated, along x and y; the narrow column strips of long columns; the
fewest passes; and solves wider than 1,024 columns, whose occupancy lines hold 32 or 64 voxels.

Tolerances are those of the operators' and solves' other parity tests (2e-5 and 1e-4 relative L2).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / max(np.linalg.norm(np.asarray(b)), 1e-30))


def cfg(W, H, Nz, its=5, reg=0.01):
    return dict(width=W, height=H, num_planes=Nz, start_plane=2500.0, plane_stepsize=20.0, wavelength=0.632,
                resolution=1.1, num_inverse_iterations=its, regularization_param=reg, regularization_TV_param=0.01,
                num_tv_iterations=3, mode=7)


# 16 x: 1; 5 7; 9 11; 13 17; 3 9, 25; 19, 31; 121, 2 3; powers above 1,024; 251 and a 2-column strip;
# strips of 8 and 4 columns
SHAPES = [(16, 16), (80, 112), (144, 176), (208, 272), (432, 400), (304, 496), (1936, 96), (2048, 4096), (4016, 32),
          (16, 1216), (32, 2304)]


@pytest.mark.parametrize("radix", [16, 4])
@pytest.mark.parametrize("W,H", SHAPES)
def test_operators_match_the_oracle(pkg, orc, gpu_available, W, H, radix):
    Nz = 3 if W * H < 1 << 20 else 1
    c = cfg(W, H, Nz)
    rng = np.random.default_rng(W + 3 * H)
    x = (rng.standard_normal((Nz, H, W)) + 1j * rng.standard_normal((Nz, H, W))).astype(np.complex64)
    r = rng.standard_normal((H, W)).astype(np.complex64)
    with pkg.SparseCompressiveHolo(pkg.make_params(**c), pkg.Schedule.make(fft_path=1, max_radix=radix)) as rec:
        est, g = rec.forward(x), rec.adjoint(r)
    p = orc.make_params(**c)
    assert rel(est, orc.forward(p, x, "f32")) < 2e-5
    assert rel(g, orc.adjoint(p, r, "f32")) < 2e-5


@pytest.mark.parametrize("W,H", [(1088, 48), (2064, 32), (48, 1104)])
def test_sparse_solve_matches_the_oracle(pkg, orc, scenes, gpu_available, W, H):
    """Iterates mostly zero (a strong L1 weight), so the column pass reads by the occupancy lines."""
    c = cfg(W, H, 4, its=12, reg=0.15)
    holo, _ = scenes.tracers_rods_scene(scenes.optics_of(c), 12, 1, W + H, 0.02, rod_len=(8.0, 16.0))
    with pkg.SparseCompressiveHolo(pkg.make_params(**c)) as rec:
        st = rec.inverseReconstruct(holo)
        vol = rec.getVolume()
    ref, _, _, rst = orc.solve(orc.make_params(**c), holo, None, "f32")
    assert 0 < np.count_nonzero(ref) < 0.05 * ref.size
    assert rel(vol, ref) < 1e-4, rel(vol, ref)
    assert list(st["restarts"]) == list(rst["restarts"]) and list(st["backtracks"]) == list(rst["backtracks"])
    np.testing.assert_allclose(st["f"], rst["f"], rtol=1e-4)
