"""GPU test: the first pair of a batch tunes the sweeps once per volume shape and
context, and only where they can run its solves."""
import numpy as np
import pytest

from test_gpu_chip_fallbacks import _counts
from test_gpu_onchip import ATV, _fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eigs,bound,first", [
    ((1, 0.3, 0.1), 0.0, 4),    # no sweep takes these
    ((1, ATV, ATV), 0.0, 2),
    ((1, ATV, ATV), 1e9, 2),    # stops at its first iteration: nothing to time
])
def test_batches_tune_once(dev, eigs, bound, first):
    from miccai2016_amd.device import DeviceContext
    from miccai2016_amd.processing.continuous_cut_anisotropic_gpu import CmfCutQAnisotropicGpu
    dev, shape = DeviceContext(0), (100, 101, 99)   # a context that has met no shape
    u0, q, _, cs, ct, _, _ = _fields(dev, shape, "axial")
    gms = 4 * dev.upload(np.random.default_rng(1).random(shape, dtype=np.float32))
    p = CmfCutQAnisotropicGpu.CutParameters()
    p.num_iter, p.update, p.error_bound, p.steps = 100, 30, bound, 0.16
    cut = CmfCutQAnisotropicGpu(p, dev)
    w, d = np.float32([0.02, 0.1, 0.4, 2]), np.float32([1, 30, 5, 9])
    outs = []
    for on_chip in (first, 4, 4):
        at = _counts(dev)
        u = u0.reshape(1, -1).repeat(4, 1)
        cut.execute_batched_device(u, 4, w, d, q, gms, cs, ct, shape, eigs)
        assert _counts(dev)[0] - at[0] == on_chip
        outs.append((u, [(r.iterations, r.stopped, r.ncrit) for r in cut.last_result]))
    for u, res in outs[1:]:
        assert dev.torch.equal(u, outs[0][0]) and res == outs[0][1]
