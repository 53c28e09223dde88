"""Near field + L2P in the mirror-symmetric basis (k_near_mfma, k_near_h16)
against the oracle's product, at the shapes where the folding can go wrong:
one 16-box tile (level 3), tiles on every edge (levels 4, 5), few and many leaf
directions (S = 40: orbits not a multiple of a k-step; 68; 124 and 128: the
split kernel's last size and the first that leaves it), every tile width.

Bars: FP64 max(1e-12, 2e-15 |Y_P(x)|) (two FP64 evaluations agree to
eps |Y_P(x)|, P = S / 4 the order of the leaf translations, x their argument);
FP32 1e-5, the FP32 operator's own.  A wrong mirror image, sign or orbit moves
whole boxes.
"""
import numpy as np
import pytest

from conftest import oracle_for, rand_c, relerr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def isg():
    import isg as m
    return m


@pytest.mark.parametrize("level,res", [(3, 0.1), (4, 0.05), (4, 0.25), (4, 0.26), (5, 0.1)])
def test_near_tiles_match_oracle(isg, level, res):
    import torch
    from scipy.special import yv
    print("near tiles, level", level, "res", res, flush=True)
    o = oracle_for(level, res=res)
    nrhs = 3
    X = np.stack([rand_c(np.random.default_rng(900 + k), o.N) for k in range(nrhs)]).astype(np.complex64)
    ref = [o.mlfma(X[k].astype(np.complex128)) for k in range(nrhs)]

    def check(R, tol, what):
        errs = [relerr(R[k], ref[k]) for k in range(nrhs)]
        print("%s: max relative difference %.2e (bar %.1e)" % (what, max(errs), tol), flush=True)
        assert max(errs) < tol, (what, errs)

    s = isg.Solver(level=level, numrx=16, max_rhs=nrhs, res=res)
    tol = max(1e-12, 2e-15 * abs(yv(s.numsamp[-1] // 4, 2 * s.k0 * 8 * res)))
    for nb in (16, 32):
        s.tuning_set(0, 0, "near", 0, nb)
        check(s.mlfma_many(X), tol, "FP64 near %d" % nb)
    s.close()
    s = isg.Solver(level=level, numrx=16, max_rhs=nrhs, res=res, precision=1)
    x = torch.from_numpy(X).cuda()
    r = torch.empty_like(x)
    torch.cuda.synchronize()
    for nb in (16, 32, 64, 128, -1):
        s.tuning_set(1, 0, "near", 0, nb)
        s.mlfma_f32_dev(x.data_ptr(), r.data_ptr(), nrhs)
        s.synchronize()
        check(r.cpu().numpy(), 1e-5, "FP32 near %d" % nb)
        if nb < 128:
            check(s.mlfma_many(X), 1e-5, "FP32 near %d, FP64 vectors" % nb)
    s.close()
