"""BiCGSTAB's vector steps inside P2M (p, s and the contrast products formed
while P2M loads its input): batches whose systems stop at different iterations,
so that workgroups shared by two systems see each of them switched off, odd
batches, shared and per-system contrasts, forward and adjoint, and every P2M
kernel a choice can name.  Each system's solution must solve its own equation:
|b - A x| <= toli |b| by the oracle's FP64 product, with a tenth allowed for the
FP64 product's own difference; a system with a zero right-hand side keeps x = 0.
"""
import numpy as np
import pytest

from conftest import oracle_for, rand_c

pytestmark = pytest.mark.gpu

TOL = 1e-6


@pytest.fixture(scope="module")
def isg():
    import isg as m
    return m


@pytest.mark.parametrize("precision,nrhs,tiles", [(0, 1, (16, 32)), (0, 3, (16, 32)), (1, 3, (16, 32, 64)),
                                                  (1, 5, (16, 64, 128)), (1, 16, (128,))])
def test_systems_stop_on_their_own(isg, precision, nrhs, tiles):
    import torch
    level = 5
    o = oracle_for(level)
    rng = np.random.default_rng(7)
    # contrasts of different strength: different iteration counts
    g = np.stack([(0.02 + 0.3 * k / nrhs) * (rng.random(o.N) + 0.05j) for k in range(nrhs)])
    b = np.stack([rand_c(np.random.default_rng(70 + k), o.N) for k in range(nrhs)])
    if nrhs > 1:
        b[1] = 0
    s = isg.Solver(level=level, numrx=16, max_rhs=nrhs, precision=precision, toli=TOL)
    for nb in tiles:
        s.tuning_set(precision, 1 if nrhs >= 16 else 0, "p2m", 0, nb)
        for herm in (False, True):
            for stride in (0, o.N):
                print("P2M", nb, "precision", precision, "nrhs", nrhs, "adjoint", herm, "stride", stride, flush=True)
                gd, bd = torch.from_numpy(g).cuda(), torch.from_numpy(b).cuda()
                x = torch.zeros_like(bd)
                torch.cuda.synchronize()
                rc, info = s.bicgs_dev(x.data_ptr(), gd.data_ptr(), bd.data_ptr(), nrhs, herm, stride, True)
                X = x.cpu().numpy()
                for k in range(nrhs):
                    gk = g[k if stride else 0]
                    if not b[k].any():
                        assert not X[k].any()
                        continue
                    ax = X[k] - (np.conj(gk * o.mlfma(np.conj(X[k]))) if herm else o.mlfma(gk * X[k]))
                    rel = np.linalg.norm(b[k] - ax) / np.linalg.norm(b[k])
                    assert info[k]["status"] == 0 and rel < 1.1 * TOL, (k, info[k], rel)
    s.close()
