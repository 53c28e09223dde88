"""P2M with the leaf level's M2M in the same kernel (split FP16 of the FP32
operator; mirror-symmetric in FP64), against the oracle's product.  FP32: leaf sample counts at and around the range
it serves (64 and 76: separate kernels; 68, 72: its smallest and largest
multiples of 4), the smallest tree with parents (level 3: the leaf is level 2,
nothing to do; 4: one workgroup of parents per 32 boxes), an odd last pair of
right-hand sides, right-hand sides 16 decades apart.
FP64: axes and orbits of few and many directions (S = 40; 124: the last count
of two column blocks; 128: the general kernel), both tile widths.
Bars, of each right-hand side's own norm: FP32 1e-5; FP64 max(1e-12,
2e-15 |Y_P(x)|), P = S / 4 the order of the leaf translations, x their argument.
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


@pytest.mark.parametrize("level,res,S", [(3, 0.1, 68), (4, 0.045, 40), (4, 0.1, 68), (4, 0.25, 124), (4, 0.26, 128),
                                         (5, 0.11, 72)])
def test_fp64_p2m_with_leaf_m2m_matches_oracle(isg, level, res, S):
    from scipy.special import yv
    print("FP64 level", level, "res", res, flush=True)
    o = oracle_for(level, res=res)
    assert o.numsamp[-1] == S
    X = np.stack([rand_c(np.random.default_rng(80 + k), o.N) for k in range(3)])
    ref = [o.mlfma(x) for x in X]
    s = isg.Solver(level=level, numrx=16, max_rhs=3, res=res)
    tol = max(1e-12, 2e-15 * abs(yv(S // 4, 2 * s.k0 * 8 * res)))
    for nb in (16, 32, -1):
        s.tuning_set(0, 0, "p2m", 0, nb)
        R = s.mlfma_many(X)
        errs = [relerr(R[k], ref[k]) for k in range(3)]
        print("P2M %d: max relative difference %.2e (bar %.1e)" % (nb, max(errs), tol), flush=True)
        assert max(errs) < tol, (nb, errs)
    # the receiver product climbs to the root through the same kernel
    ra, oa = s.aggregate(X[0]), o.aggregate(X[0])
    assert relerr(ra, oa) < tol
    s.close()
