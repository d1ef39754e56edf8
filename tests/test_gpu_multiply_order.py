"""The operator's work order (strips of y lines, parts of the order per XCD, one
or two right-hand sides per thread): blocks that need one and several strips, the
last one shorter, odd and even numbers of right-hand sides."""
import numpy as np
import pytest

from conftest import rand_block
from test_gpu_parity import _helm, _oracle, _problem, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(40, 27, 20), (7, 3, 23)])
@pytest.mark.parametrize("k", [1, 2, 33, 64])
def test_strips_match_oracle(torch_cuda, nx, ny, nz, k):
    torch = torch_cuda
    disc, vel = _problem(nx, ny, nz)
    o, h = _oracle(disc, vel), _helm(disc, vel)
    l2n = o.local_to_natural()
    X = rand_block(np.random.default_rng(190 + k), o.N, k)
    xd = torch.from_numpy(X).cuda()
    yd = torch.full_like(xd, float("nan"))
    h.Multiply(xd, yd)
    torch.cuda.synchronize()
    # 7 products a row: a few roundings of the largest
    assert _rel(yd.cpu().numpy()[l2n], o.multiply(X[l2n])) < 1e-14
