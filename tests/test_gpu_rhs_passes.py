"""Blocks of more than 16 right-hand sides: the front-solve launches take them
32 at a time, one workgroup per tile and pass.  Around the edges of a pass, with
and without inner slices, sums in the launch and in a launch of their own."""
import numpy as np
import pytest

from conftest import rand_block
from test_gpu_parity import _oracle, _problem, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiling", [dict(), dict(min_tiles=4096, max_split=16),
                                    dict(min_tiles=4096, max_split=16, xcd_reduce=0),
                                    dict(min_tiles=1, max_split=1)])
@pytest.mark.parametrize("k", [17, 31, 32, 33, 65, 256])
def test_passes_match_oracle(torch_cuda, k, tiling):
    import psp_amd
    torch = torch_cuda
    disc, vel = _problem(17, 14, 26)
    o = _oracle(disc, vel)
    l2n = o.local_to_natural()
    X = rand_block(np.random.default_rng(130 + k), o.N, k)
    ref = o.precondition(X[l2n])
    # FP64: the oracle's rounding; FP32: the sweep's 1e-4 of the other tests
    for precision, tol in (("fp64", 1e-10), ("fp32", 1e-4)):
        h = psp_amd.DistHelmholtz(disc, precision=precision)
        h.set_solve_tiling(**tiling)
        h.Initialize(vel)
        xd = torch.from_numpy(X).cuda()
        h.Precondition(xd)
        torch.cuda.synchronize()
        assert _rel(xd.cpu().numpy()[l2n], ref) < tol


@pytest.mark.parametrize("off", [(), (1,), (0, 1, 2)])
def test_merged_batch_of_sliced_passes(torch_cuda, off):
    # sliced tiles of one and several passes in merged launches, members `off`
    # with their sums in a reduce launch: each equals its own solve
    import psp_amd
    from test_gpu_batch_merged import _alone, _batch, _sources
    torch = torch_cuda
    helms, Bs = [], []
    for j, (nx, ny, nz, k) in enumerate([(15, 13, 24, 70), (16, 14, 22, 33), (12, 11, 26, 5)]):
        disc, vel = _problem(nx, ny, nz)
        h = psp_amd.DistHelmholtz(disc)
        h.set_solve_tiling(min_tiles=4096, max_split=16, xcd_reduce=0 if j in off else 1)
        h.Initialize(vel)
        helms.append(h)
        Bs.append(_sources(nx, ny, nz, k, 170 + j))
    ref = [_alone(torch, h, B, 1e-9) for h, B in zip(helms, Bs)]
    for (x, r), (xr, rr) in zip(zip(*_batch(torch, helms, Bs, 1e-9)), ref):
        assert r.iterations == rr.iterations and torch.equal(x, xr)
