"""Replayed BiCGSTAB iterations against eager ones, at sizes that do capture a
graph: at most 8192 elements, and solves of more than 8 iterations.  The kernels
and their order are the same, so results and iteration counts are equal to the
last bit; the replay count says that the graph ran (graph = 1) or did not (graph
= 0, larger solves, live kernel timing).  Between two solves the context runs
other work (a product, a solve with the other operator side).

64x64 pixels, one and two systems: FP64, and mixed precision (P2M with its vector
steps and M2M, the fused downward pass, the near field's post steps, the
residual's partials in the product's input) with the near field and P2M by rule
and on the split-FP16 kernels.
"""
import numpy as np
import pytest

from conftest import oracle_for, rand_c

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def isg():
    import isg as m
    return m


def solves(isg, graph, precision, nrhs, split, timing=False):
    """Forward, adjoint, forward again on one context: solutions, iteration counts, replays."""
    import torch
    o = oracle_for(4)
    g = 0.3 * rand_c(np.random.default_rng(1), o.N) * o.k0 ** 2
    b = np.stack([rand_c(np.random.default_rng(2 + k), o.N) for k in range(nrhs)])
    s = isg.Solver(level=4, max_rhs=nrhs, precision=precision, toli=1e-6 if precision else 1e-10, iti=300, graph=graph)
    if split:
        s.tuning_set(1, 0, "near", 0, 128)
        s.tuning_set(1, 0, "p2m", 0, 128)
    s.profile(timing)
    gd, bd = torch.from_numpy(g).cuda(), torch.from_numpy(b).cuda()
    xs, its = [], []
    for herm in (False, True, False):
        x, r = torch.zeros_like(bd), torch.empty_like(bd)
        torch.cuda.synchronize()
        _, info = s.bicgs_dev(x.data_ptr(), gd.data_ptr(), bd.data_ptr(), nrhs, herm, 0, True)
        s.mlfma_dev(x.data_ptr(), r.data_ptr(), nrhs)
        s.synchronize()
        xs += [x.cpu().numpy(), r.cpu().numpy()]
        its += [i["iters"] for i in info]
    if timing:
        assert s.profile_read("near_fp32" if precision else "near")[1] > 0
    n = s.graph_replays()
    s.close()
    return xs, its, n


@pytest.mark.parametrize("precision,nrhs,split", [(0, 1, False), (0, 2, False), (1, 1, False), (1, 2, False), (1, 1, True),
                                                  (1, 2, True)])
def test_replayed_iterations_equal_eager_ones(isg, precision, nrhs, split):
    print("graph replays: precision", precision, "nrhs", nrhs, "split", split, flush=True)
    eager, it0, n0 = solves(isg, 0, precision, nrhs, split)
    replayed, it1, n1 = solves(isg, 1, precision, nrhs, split)
    print("iterations", it1, "replayed", n1, flush=True)
    assert n0 == 0 and n1 >= 3  # each of the three solves replays at least one
    assert it0 == it1
    for a, b in zip(eager, replayed):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("precision", [0, 1])
def test_timing_and_larger_solves_run_eagerly(isg, precision):
    print("no replays: precision", precision, flush=True)
    assert solves(isg, 1, precision, 1, False, timing=True)[2] == 0
    assert solves(isg, 1, precision, 3, False)[2] == 0
