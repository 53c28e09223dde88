"""BiCGSTAB's alpha and omega where k_bi_reduce sums the near field's partials
first (from 2^24 partials read a launch up): FP64 1024^2 x 16 (both sums exactly
at and above that line), FP32 2048^2 x 8.  Each system must solve its own
equation, |b - A x| <= toli |b| by the FP64 product with a tenth allowed for the
product's own difference; a system with a zero right-hand side keeps x = 0.

And the sums' cost: with every P2M workgroup summing every partial, a launch at
8192^2 took 7.3 times one at 4096^2 (4 times the unknowns, 16 times the reads);
with them summed once it must stay below 5.5 times, half way in the logarithm
between linear and that.
"""
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-6


@pytest.fixture(scope="module")
def isg():
    import isg as m
    return m


def case(N, nrhs, k0):
    """Contrasts of different strength (different iteration counts), random right-hand sides, the second zero."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    w = torch.linspace(0.02, 0.2, nrhs, dtype=torch.float64, device="cuda")[:, None]
    g = w * torch.rand(nrhs, N, dtype=torch.float64, device="cuda", generator=gen) * torch.tensor(1 + 0.05j, device="cuda")
    b = torch.randn(nrhs, N, dtype=torch.complex128, device="cuda", generator=gen)
    b[1] = 0
    return g.to(torch.complex128), b


@pytest.mark.parametrize("level,nrhs,precision", [(8, 16, 0), (9, 8, 1)])
@pytest.mark.parametrize("herm", [False, True])
def test_reduced_sums_solve(isg, level, nrhs, precision, herm):
    import torch
    print("level", level, "nrhs", nrhs, "precision", precision, "adjoint", herm, flush=True)
    s = isg.Solver(level=level, numrx=16, max_rhs=nrhs, precision=precision, toli=TOL)
    g, b = case(s.N, nrhs, s.k0)
    x = torch.zeros_like(b)
    torch.cuda.synchronize()
    _, info = s.bicgs_dev(x.data_ptr(), g.data_ptr(), b.data_ptr(), nrhs, herm, s.N, True)
    y = (x.conj() if herm else g * x).resolve_conj().contiguous()
    gy = torch.empty_like(y)
    torch.cuda.synchronize()
    s.mlfma_dev(y.data_ptr(), gy.data_ptr(), nrhs)
    s.synchronize()
    ax = x - ((g * gy).conj() if herm else gy)
    for k in range(nrhs):
        if k == 1:
            assert not bool(x[k].abs().any())
            continue
        rel = float((b[k] - ax[k]).norm() / b[k].norm())
        assert info[k]["status"] == 0 and info[k]["iters"] > 0 and rel < 1.1 * TOL, (k, info[k], rel)
    s.close()


def test_p2m_step_cost_grows_with_the_unknowns(isg):
    import torch
    us = {}
    for level in (10, 11):
        s = isg.Solver(level=level, numrx=16, max_rhs=1, toli=1e-30, iti=3)
        gen = torch.Generator(device="cuda")
        gen.manual_seed(3)
        g = torch.rand(s.N, dtype=torch.float64, device="cuda", generator=gen).to(torch.complex128)
        b = torch.randn(s.N, dtype=torch.complex128, device="cuda", generator=gen)
        x = torch.zeros_like(b)
        torch.cuda.synchronize()
        t = []
        for _ in range(3):
            s.profile(True)
            s.bicgs_dev(x.data_ptr(), g.data_ptr(), b.data_ptr(), 1, False, 0, True)
            ms, n = s.profile_read("p2m")
            s.profile(False)
            t.append(ms / n)
        us[level] = 1e3 * min(t)
        print("level %d: P2M with its vector step %.1f us" % (level, us[level]), flush=True)
        s.close()
        del g, b, x
    assert us[11] < 5.5 * us[10]
