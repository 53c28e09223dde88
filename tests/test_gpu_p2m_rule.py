"""FP32 P2M by the built-in rule where it cannot take the leaf level's M2M along
(36 taps: a window too long; res 0.05 and 0.13: 44 and 80 leaf samples): the split
kernel from 256 workgroups of 32 boxes x 2 systems on, the dense one below.  The
rule must give the bits of the kernel it stands for, in products and in the solver
(P2M with its vector steps), and they must differ from the other kernel's.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{"ninter": 36}, {"res": 0.05}, {"res": 0.13}], ids=["36taps", "res0.05", "res0.13"])
@pytest.mark.parametrize("level,nrhs,kernel", [(7, 4, 128), (7, 5, 128), (6, 16, 128), (6, 14, 32), (5, 5, 16), (7, 3, 32)])
def test_rule_without_leaf_m2m(kw, level, nrhs, kernel):
    import isg
    import torch
    print(kw, "level", level, "nrhs", nrhs, "kernel", kernel, flush=True)
    other = 16 if kernel == 128 else 128
    s = isg.Solver(level=level, numrx=16, max_rhs=nrhs, precision=1, toli=1e-4, **kw)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(level)
    b = torch.randn(nrhs, s.N, dtype=torch.complex128, device="cuda", generator=gen)
    g = torch.full((s.N,), 0.3 + 0.01j, dtype=torch.complex128, device="cuda")
    x32 = b.to(torch.complex64)
    res = {}
    for value in (-1, kernel, other):
        s.tuning_set(1, 1 if nrhs >= 16 else 0, "p2m", 0, value)
        r, x = torch.empty_like(x32), torch.zeros_like(b)
        torch.cuda.synchronize()
        s.mlfma_f32_dev(x32.data_ptr(), r.data_ptr(), nrhs)
        s.synchronize()
        s.bicgs_dev(x.data_ptr(), g.data_ptr(), b.data_ptr(), nrhs, False, 0, True)
        res[value] = (r, x)
    for a, c in zip(res[-1], res[kernel]):
        assert bool((a == c).all())
    if nrhs >= 4:  # (below, the split kernel without M2M is not run at all)
        for a, c in zip(res[-1], res[other]):
            assert not bool((a == c).all())
    s.close()
