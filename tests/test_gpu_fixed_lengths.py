"""Every length with a compile-time FFT plan, along x and along y, beside a fixed and a run-time length:
A and A^T against the FP32 oracle at the tolerance of the operators' other tests (2e-5 relative L2).
A row workgroup's threads are not a multiple of 64 at some lengths, and at 896 its last wave has fewer
lanes (32) than a row has strips (56): solves there, with every strip present, and with strips only
where that wave has no lane of its own, at the solves' tolerance (1e-4, equal decisions)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [16, 32, 48, 64, 80, 96, 128, 192, 256, 320, 384, 448, 512, 576, 640, 768, 832, 896, 1024]


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / max(np.linalg.norm(np.asarray(b)), 1e-30))


def cfg(W, H, Nz, its=6, reg=0.01):
    return dict(width=W, height=H, num_planes=Nz, start_plane=2500.0, plane_stepsize=20.0, wavelength=0.632,
                resolution=1.1, num_inverse_iterations=its, regularization_param=reg, regularization_TV_param=0.01,
                num_tv_iterations=3, mode=7)


@pytest.mark.parametrize("L", LENGTHS)
@pytest.mark.parametrize("other", [64, 112])
def test_operators_at_every_fixed_length(pkg, orc, gpu_available, L, other):
    rng = np.random.default_rng(L + other)
    for W, H in ((L, other), (other, L)):
        c = cfg(W, H, 5)
        x = (rng.standard_normal((5, H, W)) + 1j * rng.standard_normal((5, H, W))).astype(np.complex64)
        r = rng.standard_normal((H, W)).astype(np.complex64)
        with pkg.SparseCompressiveHolo(pkg.make_params(**c)) as rec:
            est, g = rec.forward(x), rec.adjoint(r)
        p = orc.make_params(**c)
        assert rel(est, orc.forward(p, x, "f32")) < 2e-5, (W, H)
        assert rel(g, orc.adjoint(p, r, "f32")) < 2e-5, (W, H)


@pytest.mark.parametrize("H", [64, 112])
@pytest.mark.parametrize("x0,reg", [(0, 0.01), (560, 0.3)])
def test_solves_at_896(pkg, orc, gpu_available, H, x0, reg):
    W, Nz = 896, 6
    c = cfg(W, H, Nz, its=10, reg=reg)
    p = orc.make_params(**c)
    rng = np.random.default_rng(H + x0)
    x = np.zeros((Nz, H, W), np.complex64)
    for _ in range(6):
        z, y, col = rng.integers(0, Nz), rng.integers(4, H - 4), rng.integers(x0 + 20, W - 40)
        x[z, y:y + 2, col:col + 2] = 1.0
    holo = orc.forward(p, x, "f32").astype(np.complex64)
    with pkg.SparseCompressiveHolo(pkg.make_params(**c)) as rec:
        st = rec.inverseReconstruct(holo)
        vol = rec.getVolume()
    ref, _, _, rst = orc.solve(p, holo, None, "f32")
    assert rel(vol, ref) < 1e-4, rel(vol, ref)
    assert list(st["backtracks"]) == list(rst["backtracks"]) and list(st["restarts"]) == list(rst["restarts"])
    np.testing.assert_allclose(st["f"], rst["f"], rtol=1e-4)
    if x0:
        assert 0 < np.count_nonzero(ref) and not ref[:, :, :512].any()
