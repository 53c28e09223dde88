"""FP32 products of vectors that are aligned to one complex element (8 bytes) only:
the split-FP16 P2M and near field load 16 bytes at a time.  The same values at a
16-byte-aligned and at an 8-byte-aligned address, input and output, must give the
same bits.  Batches of 1, 2 and 5, every near-field and P2M kernel a choice can
name, guard elements on both sides of the output unchanged.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,nrhs", [(4, 1), (5, 2), (6, 5)])
@pytest.mark.parametrize("width", [-1, 16, 64, 128])
def test_element_aligned_vectors(level, nrhs, width):
    import isg
    import torch
    print("level", level, "nrhs", nrhs, "near field and P2M", width, flush=True)
    s = isg.Solver(level=level, numrx=16, max_rhs=nrhs, precision=1)
    s.tuning_set(1, 0, "near", 0, width)
    s.tuning_set(1, 0, "p2m", 0, width)
    rng = np.random.default_rng(level)
    x = torch.from_numpy((rng.standard_normal(nrhs * s.N) + 1j * rng.standard_normal(nrhs * s.N)).astype(np.complex64)).cuda()
    out = []
    for shift in (0, 1):
        src = torch.zeros(x.numel() + 4, dtype=torch.complex64, device="cuda")
        dst = torch.full((x.numel() + 4,), 7.0, dtype=torch.complex64, device="cuda")
        a, r = src[2 + shift:2 + shift + x.numel()], dst[2 + shift:2 + shift + x.numel()]
        a.copy_(x)
        assert a.data_ptr() % 16 == 8 * shift and r.data_ptr() % 16 == 8 * shift
        torch.cuda.synchronize()
        s.mlfma_f32_dev(a.data_ptr(), r.data_ptr(), nrhs)
        s.synchronize()
        assert bool((dst[:2 + shift] == 7).all()) and bool((dst[2 + shift + x.numel():] == 7).all())
        out.append(r.cpu().numpy())
    assert np.abs(out[0]).min() > 0
    np.testing.assert_array_equal(out[0], out[1])
    s.close()
