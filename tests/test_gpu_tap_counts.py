"""Chunked M2M and L2L with tap counts other than the compiled-in 30 and 60:
against the FP64 oracle (the operator with those taps; FP64 1e-12, FP32 1e-5, the
bars of the other operator tests), every level above the leaf's parents forced to
the chunked kernels, and the M2M time of 28 taps against that of 30.  One weight
load per tap and child made the former 1.9 times the latter; with one per tap it is
1.05.  Bar: 1.4, half way in the logarithm.
"""
import numpy as np
import pytest

from conftest import oracle_for, rand_c, relerr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def isg():
    import isg as m
    return m


def force_chunked(s, precision, nrhs):
    for i in range(s.level - 1):
        for stage in ("m2m", "l2l"):
            s.tuning_set(precision, 1 if nrhs >= 16 else 0, stage, i, 1)


@pytest.mark.parametrize("ninter", [2, 6, 28, 30, 36])
@pytest.mark.parametrize("precision", [0, 1])
def test_chunked_interpolation_matches_oracle(isg, ninter, precision):
    import torch
    print("taps", ninter, "precision", precision, flush=True)
    o = oracle_for(5, ninter=ninter)
    X = np.stack([rand_c(np.random.default_rng(k), o.N) for k in range(3)])
    s = isg.Solver(level=5, numrx=16, max_rhs=3, precision=precision, ninter=ninter, tuning=False)
    s.tuning_set(precision, 0, "leaf", 0, 0)
    force_chunked(s, precision, 3)
    if precision:
        X = X.astype(np.complex64).astype(np.complex128)
        x = torch.from_numpy(X.astype(np.complex64)).cuda()
        r = torch.empty_like(x)
        torch.cuda.synchronize()
        s.mlfma_f32_dev(x.data_ptr(), r.data_ptr(), 3)
        s.synchronize()
        Y = r.cpu().numpy()
    else:
        Y = s.mlfma_many(X)
    for k in range(3):
        assert relerr(Y[k], o.mlfma(X[k])) < (1e-5 if precision else 1e-12)
    s.close()


def test_m2m_time_does_not_jump_off_thirty_taps(isg):
    import torch
    us = {}
    for ninter in (28, 30):
        s = isg.Solver(level=7, numrx=16, max_rhs=2, ninter=ninter)  # 8192 boxes: every L2L is fused
        for i in (2, 3, 4):
            s.tuning_set(0, 0, "m2m", i, 1)
        x = torch.randn(2, s.N, dtype=torch.complex128, device="cuda")
        r = torch.empty_like(x)
        torch.cuda.synchronize()
        t = []
        for _ in range(6):
            s.profile(True)
            for _ in range(10):
                s.mlfma_dev(x.data_ptr(), r.data_ptr(), 2)
            ms, n = s.profile_read("interp")
            s.profile(False)
            t.append(1e3 * ms / n)
        us[ninter] = min(t)
        print("%d taps: M2M of levels 4 .. 2 %.1f us" % (ninter, us[ninter]), flush=True)
        s.close()
    assert us[28] < 1.4 * us[30]
