"""The preprocessing's write pass at the widths where its forms meet: rows of up to 512 pixels (one pair a
thread), more (two pairs a thread, 512 pixels apart), the second pair partly and wholly inside the row,
odd rows (one pixel a thread), and an output at an address that 16 does not divide (the same): every frame
the host function's bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("remove_bg", [False, True])
@pytest.mark.parametrize("size,pad,offset", [(2, 0, 0), (510, 0, 0), (512, 0, 0), (448, 32, 0), (513, 0, 0), (514, 0, 0),
                                             (960, 33, 0), (1024, 0, 0), (1026, 0, 0), (512, 0, 1), (514, 0, 1)])
def test_widths_equal_host(pkg, gpu_available, size, pad, offset, remove_bg):
    import torch
    rng = np.random.default_rng(size + pad)
    frames = rng.integers(0, 256, (2, size, size)).astype(np.uint8)
    back = (rng.random((size, size)) * 200).astype(np.float32) if remove_bg else None
    fp = pkg.FileParams()
    fp.roi_size = -1
    fp.solver.zero_padding = pad
    fp.remove_background = int(remove_bg)
    side = size + 2 * pad
    buf = torch.full((offset + 2 * side * side + 1,), 3 + 4j, dtype=torch.complex64, device="cuda")
    out = buf[offset:offset + 2 * side * side].view(2, side, side)
    dev_frames = torch.from_numpy(frames).cuda()
    torch.cuda.synchronize()
    pkg.prepare_holograms(fp, dev_frames, background=None if back is None else torch.from_numpy(back).cuda(), out=out)
    got = out.cpu().numpy()
    for k in range(2):
        want = pkg.prepare_hologram(fp, frames[k].astype(np.float32), back)
        assert np.array_equal(got[k].view(np.uint32), want.view(np.uint32))
    assert all(complex(v) == 3 + 4j for v in (*buf[:offset].cpu(), buf[-1].cpu()))
