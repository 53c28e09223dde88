"""Split-FP16 P2M of the FP32 operator with the leaf level's M2M in the same
kernel, against the oracle's product: leaf sample counts at and around the range
it serves (64 and 76: separate kernels; 68, 72: its smallest and largest
multiples of 4), the smallest tree with parents (level 3: the leaf is level 2,
nothing to do; 4: one workgroup of parents per 32 boxes), an odd last pair of
right-hand sides, right-hand sides 16 decades apart.
Bar: 1e-5 of each right-hand side's own norm, the FP32 operator's.
"""
import numpy as np
import pytest

from conftest import oracle_for, rand_c, relerr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def isg():
    import isg as m
    return m


@pytest.mark.parametrize("level,res,S,nrhs", [(3, 0.1, 68, 4), (4, 0.095, 64, 5), (4, 0.1, 68, 5), (4, 0.105, 68, 4), (4, 0.108, 72, 7),
                                                (4, 0.12, 76, 4), (5, 0.11, 72, 5), (6, 0.1, 68, 17)])
def test_p2m_with_leaf_m2m_matches_oracle(isg, level, res, S, nrhs):
    import torch
    print("level", level, "res", res, "nrhs", nrhs, flush=True)
    o = oracle_for(level, res=res)
    assert o.numsamp[-1] == S
    base = [rand_c(np.random.default_rng(60 + k), o.N).astype(np.complex64).astype(np.complex128) for k in range(3)]
    ref = [o.mlfma(b) for b in base]
    scale = [10.0 ** (4 * (k % 5) - 8) for k in range(nrhs)]
    s = isg.Solver(level=level, numrx=16, max_rhs=nrhs, res=res, precision=1)
    s.tuning_set(1, 1 if nrhs >= 16 else 0, "p2m", 0, 128)
    x = torch.from_numpy(np.stack([base[k % 3] * scale[k] for k in range(nrhs)]).astype(np.complex64)).cuda()
    r = torch.empty_like(x)
    torch.cuda.synchronize()
    s.mlfma_f32_dev(x.data_ptr(), r.data_ptr(), nrhs)
    s.synchronize()
    R = r.cpu().numpy()
    errs = [relerr(R[k], ref[k % 3] * scale[k]) for k in range(nrhs)]
    print("max relative difference %.2e" % max(errs), flush=True)
    assert max(errs) < 1e-5, errs
    s.close()
