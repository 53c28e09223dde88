"""Fused downward pass (k_down_h16, k_down64: M2L and L2L of a level in one
kernel) against the oracle's product where it can go wrong: one 8 x 8 tile
(level 3 inside a level-4 tree), every grid edge, the last sample chunk partly
filled, 1 to 8 right-hand sides per workgroup with a partly filled last group,
windows of fewer and more taps (48 taps; 80 taps, too long: the separate
kernels), right-hand sides 16 decades apart (scales are taken per parent).

Bars: FP64 1e-12, FP32 1e-5 of each right-hand side's own norm, those of the
operator.  A wrong tap, shift, offset or scale moves whole boxes.
"""
import numpy as np
import pytest

from conftest import oracle_for, rand_c, relerr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def isg():
    import isg as m
    return m


# those with nrhs > 10 have enough boxes x right-hand sides for the rule (-1) to fuse every level
@pytest.mark.parametrize("level,ninter,nrhs", [(4, 30, 1), (4, 24, 115), (5, 30, 5), (5, 24, 29), (5, 40, 29), (6, 30, 11)])
def test_fused_downward_pass_matches_oracle(isg, level, ninter, nrhs):
    import torch
    print("down level", level, "ninter", ninter, "nrhs", nrhs, flush=True)
    o = oracle_for(level, ninter=ninter)
    base = [rand_c(np.random.default_rng(40 + k), o.N).astype(np.complex64).astype(np.complex128) for k in range(3)]
    ref = [o.mlfma(b) for b in base]
    scale = [10.0 ** (4 * (k % 5) - 8) for k in range(nrhs)]
    X = np.stack([base[k % 3] * scale[k] for k in range(nrhs)])

    def check(R, tol, what):
        errs = [relerr(R[k], ref[k % 3] * scale[k]) for k in range(nrhs)]
        print("%s: max relative difference %.2e (bar %.1e)" % (what, max(errs), tol), flush=True)
        assert max(errs) < tol, (what, errs)

    cls = 1 if nrhs >= 16 else 0
    for prec in (0, 1):
        s = isg.Solver(level=level, numrx=16, max_rhs=nrhs, ninter=ninter, precision=prec)
        x = torch.from_numpy(X).to(torch.complex64 if prec else torch.complex128).cuda()
        r = torch.empty_like(x)
        torch.cuda.synchronize()
        for leaf in (-1, 1, 0):
            s.tuning_set(prec, cls, "leaf", 0, leaf)
            (s.mlfma_f32_dev if prec else s.mlfma_dev)(x.data_ptr(), r.data_ptr(), nrhs)
            s.synchronize()
            check(r.cpu().numpy(), 1e-5 if prec else 1e-12, "FP%d leaf %d" % (32 if prec else 64, leaf))
        s.close()


# receivers: 16, one more and one fewer than a workgroup's 64 outputs
@pytest.mark.parametrize("level,ninter,nrhs,numrx", [(3, 30, 2, 65), (4, 24, 115, 63), (5, 30, 5, 16), (5, 40, 29, 64),
                                                     (6, 30, 8, 65)])
def test_receiver_products_match_oracle(isg, level, ninter, nrhs, numrx):
    """aggregate and aggregateh (no translations on the way down) at the same sizes; bar 1e-12."""
    import torch
    print("receivers level", level, "ninter", ninter, "nrhs", nrhs, "numrx", numrx, flush=True)
    o = oracle_for(level, numrx=numrx, ninter=ninter)
    xs = [rand_c(np.random.default_rng(140 + k), o.N) for k in range(3)]
    rs = [rand_c(np.random.default_rng(150 + k), numrx) for k in range(3)]
    down, up = [o.aggregateh(v) for v in rs], [o.aggregate(v) for v in xs]
    s = isg.Solver(level=level, numrx=numrx, max_rhs=nrhs, ninter=ninter)
    x = torch.from_numpy(np.stack([xs[k % 3] for k in range(nrhs)])).cuda()
    r = torch.from_numpy(np.stack([rs[k % 3] for k in range(nrhs)])).cuda()
    xo, ro = torch.empty_like(x), torch.empty_like(r)
    torch.cuda.synchronize()
    for leaf in (-1, 1, 0):
        s.tuning_set(0, 1 if nrhs >= 16 else 0, "leaf", 0, leaf)
        s.aggregate_dev(x.data_ptr(), ro.data_ptr(), nrhs)
        s.aggregateh_dev(xo.data_ptr(), r.data_ptr(), nrhs)
        s.synchronize()
        X, R = xo.cpu().numpy(), ro.cpu().numpy()
        errs = [max(relerr(X[k], down[k % 3]), relerr(R[k], up[k % 3])) for k in range(nrhs)]
        print("leaf %d: max relative difference %.2e" % (leaf, max(errs)), flush=True)
        assert max(errs) < 1e-12, (leaf, errs)
    s.close()
