"""The Arnoldi step: cycles around the edges of a group of basis vectors (8), the
longest that two passes take (64) and one step more, odd numbers of right-hand
sides; iterations and solutions are the oracle's (modified Gram-Schmidt step by
step in FP64)."""
import numpy as np
import pytest

from conftest import rand_block
from test_gpu_parity import _helm, _oracle, _problem, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 5, 130])
@pytest.mark.parametrize("m", [1, 7, 8, 9, 17, 64, 65])
def test_cycles_match_oracle(torch_cuda, m, k):
    torch = torch_cuda
    disc, vel = _problem(12, 10, 24)
    o, h = _oracle(disc, vel), _helm(disc, vel)
    B = rand_block(np.random.default_rng(210 + m + k), o.N, k)
    tol = 1e-12 if m > 1 else 1e-3
    ref, st, rep = o.solve(B, m=m, rel_tol=tol, max_its=90)
    x = torch.from_numpy(B).cuda()
    r = h.Solve(x, m, tol, maxIts=90, raise_on_error=False)
    torch.cuda.synchronize()
    assert r.iterations == rep.iterations and r.restarts == rep.restarts
    # both reach tol; they differ by the operator's condition times the rounding
    assert _rel(x.cpu().numpy(), ref) < 1e-9
