"""RIHVR_PIPE_PLANES acts also where the default plane chunks do not divide the group: the chunks go down
to a divisor, and the grouped solve equals the one-stream solve with those chunks bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,Nz,group", [(1024, 64, 48, 16), (1024, 64, 53, 16)])
def test_groups_with_chunks_that_do_not_divide_them(pkg, scenes, gpu_available, monkeypatch, W, H, Nz, group):
    c = dict(width=W, height=H, num_planes=Nz, start_plane=1000.0, plane_stepsize=25.0, wavelength=0.633,
             resolution=2.0, num_inverse_iterations=6, regularization_param=0.01, regularization_TV_param=0.01,
             num_tv_iterations=5, mode=7)
    holo, _ = scenes.disks_scene(scenes.optics_of(c), 6, 2.0, 4.0, Nz, 0.01)

    def solve():
        with pkg.SparseCompressiveHolo(pkg.make_params(**c)) as rec:
            st = rec.inverseReconstruct(holo)
            return rec.getVolume(), st, rec.schedule(), rec.counters()

    _, _, plain, n = solve()
    assert n["graphs"] > 0  # one group: its iterations run as graphs
    assert group % plain["zchunk_fwd"] or group % plain["zchunk_adj"]
    monkeypatch.setenv("RIHVR_PIPE_PLANES", str(group))
    a, sta, grouped, n = solve()
    assert n["graphs"] == 0  # groups run without graphs
    assert group % grouped["zchunk_fwd"] == 0 and group % grouped["zchunk_adj"] == 0
    monkeypatch.delenv("RIHVR_PIPE_PLANES")
    monkeypatch.setenv("RIHVR_ZCHUNK", str(grouped["zchunk_fwd"]))
    monkeypatch.setenv("RIHVR_ZCHUNK_ADJ", str(grouped["zchunk_adj"]))
    b, stb, _, _ = solve()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    np.testing.assert_array_equal(sta["f"], stb["f"])
