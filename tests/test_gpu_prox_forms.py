"""The fused mode-7 prox's three forms (rows with data skip work; the same after a scan for runs of zero
rows; dense) give the same volume bit for bit whatever the iterates hold, so that a solve may change
between them: each forced for whole solves (RIHVR_TEST_PROX_FORM), from the zero start (volumes with
maps), from a dense start (without), and from a start with a NaN, which makes every gradient non-finite
and every row one to form.  The forms order the sums differently, so objectives agree to rounding (1e-5,
the bound of the scan's test) and decisions are equal.  And the rule's own choices: a scan that skips too
little is given up."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def cfg(W, H, Nz, ntv, reg=0.1, tv=0.02, its=12):
    return dict(width=W, height=H, num_planes=Nz, start_plane=1000.0, plane_stepsize=50.0, wavelength=0.633,
                resolution=2.0, num_inverse_iterations=its, regularization_param=reg, regularization_TV_param=tv,
                num_tv_iterations=ntv, mode=7)


def _solve(pkg, monkeypatch, c, holo, form, rows, warm=None):
    if form is None:
        monkeypatch.delenv("RIHVR_TEST_PROX_FORM", raising=False)
    else:
        monkeypatch.setenv("RIHVR_TEST_PROX_FORM", form)
    with pkg.SparseCompressiveHolo(pkg.make_params(**c), pkg.Schedule.make(prox_rows=rows)) as rec:
        st = rec.inverseReconstruct(holo, warm_start=warm)
        return rec.getVolume(), st, rec.counters()


@pytest.mark.parametrize("ntv", [0, 1, 2, 5, 8, 10])
@pytest.mark.parametrize("W,H,rows", [(32, 80, 80), (112, 64, 17), (272, 96, 67), (1280, 64, 64), (2064, 80, 80)])
@pytest.mark.parametrize("start", ["zero", "dense", "nan"])
def test_forms_give_the_same_volume(pkg, scenes, gpu_available, monkeypatch, ntv, W, H, rows, start):
    c = cfg(W, H, 3, ntv)
    holo, _ = scenes.disks_scene(scenes.optics_of(c), 2, 2.0, 3.0, W + ntv, 0.002)
    warm = None
    if start != "zero":
        rng = np.random.default_rng(W + H + ntv)
        warm = (0.05 * (rng.standard_normal((3, H, W)) + 1j * rng.standard_normal((3, H, W)))).astype(np.complex64)
        if start == "nan":
            warm[1, H // 2, W - 1] = np.nan
    vols = {}
    for form in ("rows", "scan", "dense"):
        v, st, n = _solve(pkg, monkeypatch, c, holo, form, rows, warm)
        assert n["prox_" + form] == sum(n[k] for k in ("prox_rows", "prox_scan", "prox_dense"))
        if start == "nan":
            assert n["scan_skipped"] == 0
        vols[form] = (v, st)
    v0, s0 = vols["rows"]
    assert np.isnan(v0).any() == (start == "nan")
    for form in ("scan", "dense"):
        v, st = vols[form]
        if start == "nan":  # (a NaN's bits are not specified)
            np.testing.assert_array_equal(v, v0)
        else:
            assert np.array_equal(v.view(np.uint32), v0.view(np.uint32)), form
            np.testing.assert_allclose(st["f"], s0["f"], rtol=1e-5)
        assert list(st["restarts"]) == list(s0["restarts"]) and list(st["backtracks"]) == list(s0["backtracks"])


def test_a_scan_that_skips_too_little_is_given_up(pkg, scenes, gpu_available, monkeypatch):
    # with so small a TV weight the gradient's differences leave no row quiet
    c = cfg(336, 400, 4, 5, tv=1e-4, its=40)
    holo, _ = scenes.disks_scene(scenes.optics_of(c), 1, 2.0, 3.0, 1241, 0.002)
    v, st, n = _solve(pkg, monkeypatch, c, holo, None, 101)
    assert 0 < n["prox_scan"] <= 6  # again only where the non-zeros have halved
    assert n["scan_skipped"] == 0 and n["prox_scan"] + n["prox_rows"] == 40
    v0, _, n0 = _solve(pkg, monkeypatch, c, holo, "rows", 101)
    assert n0["prox_scan"] == 0
    assert np.array_equal(v.view(np.uint32), v0.view(np.uint32))


@pytest.mark.parametrize("H,rows", [(1024, 700), (1040, 0)])
def test_tall_dense_chunks_keep_the_decisions(pkg, orc, scenes, gpu_available, monkeypatch, H, rows):
    """A wave's sums over hundreds of rows: decisions and objectives against the FP32 oracle."""
    c = cfg(64, H, 3, 5, reg=0.0, tv=0.01, its=8)
    holo, _ = scenes.disks_scene(scenes.optics_of(c), 6, 2.0, 4.0, H, 0.01)
    v, st, _ = _solve(pkg, monkeypatch, c, holo, "dense", rows)
    ref, _, _, rst = orc.solve(orc.make_params(**c), holo, None, "f32")
    assert np.linalg.norm(v - ref) < 1e-4 * np.linalg.norm(ref)
    assert list(st["restarts"]) == list(rst["restarts"]) and list(st["backtracks"]) == list(rst["backtracks"])
    np.testing.assert_allclose(st["f"], rst["f"], rtol=1e-4)
