"""GPU test: volumes of a ragged set that share a launch on the chip equal lone
solves through the per-iteration kernels bit for bit."""
import numpy as np
import pytest

from test_gpu_onchip import _fields, _solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes,iters,update,bound", [
    ([(9, 12, 15), (20, 7, 11), (1, 1, 50), (5, 33, 8)], 40, 7, 0.0),           # one work-group each
    ([(24, 30, 37), (33, 61, 67), (40, 3, 300), (2, 2, 1100)], 25, 5, 0.0),     # ragged bricks
    ([(64, 64, 64)] * 5 + [(17, 16, 15)] * 6, 12, 30, 0.0),                     # more than one launch
    ([(90, 91, 70), (95, 80, 96), (128, 128, 128), (140, 150, 151)], 12, 5, 0.0),  # some left alone
    ([(24, 30, 37), (30, 31, 29), (20, 20, 20)], 300, 10, 4e-3),                # stops apart
])
def test_volumes_side_by_side_equal_lone_solves(dev, shapes, iters, update, bound):
    from miccai2016_amd.processing.continuous_cut_anisotropic_gpu import CmfCutQAnisotropicGpu
    torch = dev.torch
    print(shapes, flush=True)
    f = [_fields(dev, s, "axial", seed) for seed, s in enumerate(shapes)]
    p = CmfCutQAnisotropicGpu.CutParameters()
    p.num_iter, p.update, p.error_bound, p.steps = iters, update, bound, 0.16
    cut = CmfCutQAnisotropicGpu(p, dev)
    pack = lambda k: torch.cat([x[k].reshape(-1) for x in f])
    sizes = [int(np.prod(s)) for s in shapes]
    offs = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    u = pack(0)
    cut.execute_ragged_device(u, pack(1), pack(2), pack(3), pack(4), shapes, offs, f[0][6] ** 2)
    for s, x, o, n, r in zip(shapes, f, offs, sizes, cut.last_result):
        want = _solve(dev, x, s, 1, iters, update, bound)
        assert torch.equal(u[o:o + n], want[0].reshape(-1)), s
        assert (r.iterations, r.stopped, r.ncrit) == want[1], s
        # sums of up to 2^21 float32 terms in two orders
        np.testing.assert_allclose(r.last_crit, want[2][-1], rtol=1e-5)
