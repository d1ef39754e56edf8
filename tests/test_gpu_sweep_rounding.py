"""Rounding of a sweep's vectors and sums.  A sweep is linear in its block, so
M(u + v) - M(u) - M(v) is what its own roundings leave, the factors' errors
aside; GMRES with FP32 fronts cannot get below a multiple of it.  Bound: twice
the spacing of the front precision at 1, relative to the result, one spacing and
a half being the most of a form that sums every 64 columns on their own."""
import numpy as np
import pytest

from conftest import rand_block
from test_gpu_parity import _problem

pytestmark = pytest.mark.gpu


# the right-hand sides of each kernel: up to 8, up to 16, passes of 32
@pytest.mark.parametrize("k", [1, 5, 8, 12, 16, 24, 40])
@pytest.mark.parametrize("precision,eps", [("fp32", 2.0 ** -23), ("fp64", 2.0 ** -52)])
def test_sums_round_little(torch_cuda, precision, eps, k):
    import psp_amd
    torch = torch_cuda
    left = []
    for seed, grid in enumerate([(24, 20, 26), (17, 23, 31), (40, 40, 24)]):
        disc, vel = _problem(*grid)
        h = psp_amd.DistHelmholtz(disc, precision=precision)
        h.Initialize(vel)
        rng = np.random.default_rng(900 + seed)
        u, v = (torch.from_numpy(rand_block(rng, disc.nx * disc.ny * disc.nz, k)).cuda()
                for _ in range(2))
        w = u + v
        for x in (u, v, w):
            h.Precondition(x)
        torch.cuda.synchronize()
        left.append(float(torch.linalg.norm(w - u - v) / torch.linalg.norm(w)) / eps)
    assert max(left) < 2, left
