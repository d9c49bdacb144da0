"""The dense prox's rows per wave: the rule's number is bounded (a lane sums its column's terms in 32 bits
over them), a caller's number holds, and the number that a context reports stands for both forms' rules."""
import pytest

pytestmark = pytest.mark.gpu


def _rows(pkg, W, H, Nz, rows=0):
    p = pkg.make_params(width=W, height=H, num_planes=Nz, start_plane=1000.0, plane_stepsize=25.0, wavelength=0.633,
                        resolution=2.0, num_inverse_iterations=1, regularization_param=0.01,
                        regularization_TV_param=0.01, num_tv_iterations=5)
    with pkg.SparseCompressiveHolo(p, pkg.Schedule.make(prox_rows=rows)) as rec:
        return rec.schedule()["prox_rows"], rec.counters()["dense_rows"]


@pytest.mark.parametrize("W,H,Nz", [(64, 64, 8), (256, 256, 32), (512, 2048, 100), (1024, 4096, 32)])
def test_the_rule_is_bounded_and_stands_for_itself(pkg, gpu_available, W, H, Nz):
    sparse, dense = _rows(pkg, W, H, Nz)
    assert 0 < dense <= min(H, 256)
    assert _rows(pkg, W, H, Nz, sparse) == (sparse, dense)
    given = sparse - 1 if sparse > 1 else 2
    assert _rows(pkg, W, H, Nz, given) == (given, given)
    assert _rows(pkg, W, H, Nz, H)[1] in (H, dense)
