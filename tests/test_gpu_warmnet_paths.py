"""Paths of the network's first and small layers: images read directly by layer
0 (16-byte aligned) or packed first (any other address), and the number of
output blocks per workgroup, which follows the launch size.  Each is the same
sum in the same order, so results must be equal bit for bit: aligned against
shifted images, and a batch against its images one by one (16 x 16: one position
at the coarsest level; 48 x 80: partial tiles; 256 x 256: enough workgroups for
the wide form).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 16, 16), (3, 48, 80), (2, 128, 64), (4, 256, 256)])
def test_image_alignment_and_batch_do_not_change_bits(shape):
    import isg
    import torch
    print("network paths", shape, flush=True)
    b, H, W = shape
    n = isg.WarmNet(max_batch=b, max_pixels=H * W, seed=5)
    x = torch.from_numpy(np.random.default_rng(3).standard_normal(shape + (8,)).astype(np.float32)).cuda()
    buf = torch.empty(x.numel() + 1, dtype=torch.float32, device="cuda")
    shifted = buf[1:].view(x.shape)
    shifted.copy_(x)
    assert x.data_ptr() % 16 == 0 and shifted.data_ptr() % 16 == 4
    outs = []
    for src in (x, shifted):
        y = torch.zeros(shape + (2,), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        n.forward_dev(src.data_ptr(), y.data_ptr(), b, H, W)
        torch.cuda.synchronize()
        outs.append(y.cpu().numpy())
    np.testing.assert_array_equal(outs[0], outs[1])
    assert np.isfinite(outs[0]).all() and np.abs(outs[0]).max() > 0
    for k in range(b):
        np.testing.assert_array_equal(n.forward(x[k:k + 1].cpu().numpy())[0], outs[0][k])
