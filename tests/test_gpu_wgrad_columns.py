"""The weight gradient's walk down columns of 16-voxel segments against the CPU oracle: columns of
one and two rows, chunks that start and end inside a column and that cross columns and planes,
partial last segments, planes of one column.  Tolerance: that of the other weight-gradient tests
(FP32 sums of exact BF16 products, 1e-5 relative L2)."""
import numpy as np
import pytest

from oracle import unet3d as U

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.ravel(a) - np.ravel(b)) / np.linalg.norm(np.ravel(b)))


@pytest.mark.parametrize("D,H,W", [(1, 1, 1), (3, 1, 17), (2, 2, 48), (1, 5, 16), (5, 3, 33), (1, 4999, 15), (2, 37, 131)])
def test_wgrad_columns(pkg, gpu_available, D, H, W):
    import torch
    rng = np.random.default_rng(1000 * D + 10 * H + W)
    x = U.bf16(rng.normal(size=(D, H, W, 32)))
    g = U.bf16(rng.normal(size=(D, H, W, 16)))

    def bits(a):
        return torch.from_numpy(U.bf16_bits(a).view(np.int16)).cuda()

    dw, db = pkg.conv3d_bf16_wgrad(bits(x), bits(g), None)
    edw, edb = U.conv_wgrad(x, g)
    assert _rel(dw.cpu().numpy(), edw) <= 1e-5
    assert _rel(db.cpu().numpy(), edb) <= 1e-5
