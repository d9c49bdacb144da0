"""A and A^T on device tensors, which they read and write in place: the same bits as through host arrays,
for volumes that start an allocation, inside one, and at addresses that 16 does not divide, with what lies
around an output untouched; at fixed, run-time and mixed lengths."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,Nz", [(64, 64, 8), (272, 208, 3), (128, 272, 4), (272, 64, 3), (2064, 32, 2)])
@pytest.mark.parametrize("first", [0, 1, 6])
def test_device_arrays_equal_host_arrays(pkg, gpu_available, W, H, Nz, first):
    import torch
    p = pkg.make_params(width=W, height=H, num_planes=Nz, start_plane=1000.0, plane_stepsize=25.0, wavelength=0.633,
                        resolution=2.0, num_inverse_iterations=1, regularization_param=0.01,
                        regularization_TV_param=0.01, num_tv_iterations=5)
    rng = np.random.default_rng(W + H)
    x = (rng.standard_normal((Nz, H, W)) + 1j * rng.standard_normal((Nz, H, W))).astype(np.complex64)
    r = rng.standard_normal((H, W)).astype(np.complex64)
    n = x.size

    def on_device(a, shape):  # values 1 + 1j around it
        buf = torch.full((first + int(np.prod(shape)) + 5,), 1 + 1j, dtype=torch.complex64, device="cuda")
        view = buf[first:first + int(np.prod(shape))].view(shape)
        if a is not None:
            view.copy_(torch.from_numpy(a))
        return buf, view

    with pkg.SparseCompressiveHolo(p) as rec:
        est, g = rec.forward(x), rec.adjoint(r)
        _, xd = on_device(x, x.shape)
        _, rd = on_device(r, r.shape)
        eb, ed = on_device(None, r.shape)
        gb, gd = on_device(None, x.shape)
        assert xd.data_ptr() % 16 == 8 * (first % 2)
        torch.cuda.synchronize()
        rec.forward(xd, out=ed)
        rec.adjoint(rd, out=gd)
        rec.adjoint(r, out=gd)  # (host in, device out)
        est2 = rec.forward(xd, out=np.empty_like(r))
    assert np.array_equal(ed.cpu().numpy().view(np.uint32), est.view(np.uint32))
    assert np.array_equal(gd.cpu().numpy().view(np.uint32), g.view(np.uint32))
    assert np.array_equal(est2.view(np.uint32), est.view(np.uint32))
    assert torch.equal(xd.cpu(), torch.from_numpy(x))  # the input is read only
    for buf, m in ((gb, n), (eb, r.size)):
        around = torch.cat([buf[:first], buf[first + m:]]).cpu()
        assert torch.equal(around, torch.full_like(around, 1 + 1j))
