"""The fused launches switched on after Initialize: calls that need no factors, and
sweeps that the fused launches do not take, work on the factors as they stand;
the first sweep that they take factors once more.  Against the oracle (FP64
fronts, 1e-10 relative)."""
import numpy as np
import pytest

from conftest import rand_block
from test_gpu_parity import _oracle, _problem, _rel

pytestmark = pytest.mark.gpu


def test_switched_on_after_initialize(torch_cuda):
    import psp_amd
    torch = torch_cuda
    disc, vel = _problem(20, 18, 26)
    o = _oracle(disc, vel)
    l2n = o.local_to_natural()
    h = psp_amd.DistHelmholtz(disc)
    h.Initialize(vel)
    h.set_solve_tiling(fused=1)
    rng = np.random.default_rng(77)

    def check(call, k, want):
        X = rand_block(rng, o.N, k)
        x = torch.from_numpy(X).cuda()
        y = call(x)
        torch.cuda.synchronize()
        assert _rel(y.cpu().numpy()[l2n], want(X[l2n])) < 1e-10

    def inplace(f):
        return lambda x: (f(x), x)[1]

    def multiply(x):
        y = torch.empty_like(x)
        h.Multiply(x, y)
        return y

    check(inplace(h.PreconditionNoAlloc), 8, o.precondition)
    check(multiply, 8, o.multiply)
    check(inplace(h.Precondition), 3, o.precondition)
    check(inplace(h.Precondition), 8, o.precondition)
    check(inplace(h.PreconditionNoAlloc), 8, o.precondition)
    check(inplace(h.Precondition), 17, o.precondition)
    h.set_solve_tiling(fused=0)
    check(inplace(h.Precondition), 8, o.precondition)
