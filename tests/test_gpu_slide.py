"""GPU tests: passes over a window of planes that slides through the volume (the
automatic method of volumes beyond the chip's registers) equal the per-iteration
kernels bit for bit."""
import threading

import numpy as np
import pytest

from test_gpu_onchip import _fields, _solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,kind,iters,update,bound,scaling", [
    ((256, 256, 256), "axial", 33, 30, 0.0, (1, 1, 1)),     # full passes and a remainder
    ((101, 250, 250), "axial", 40, 20, 0.0, (2, 1, 1.5)),   # ragged tiles, an odd last plane
    ((100, 250, 250), "axial", 300, 10, 6e-3, (1, 1, 1)),   # stops at a criterion
    ((5, 600, 800), "seeded", 21, 20, 0.0, (1, 1, 1)),      # fewer planes than levels
    ((3, 1000, 900), "seeded", 7, 30, 0.0, (1, 1, 1)),      # one short pass
    ((30, 60, 2000), "seeded", 23, 7, 0.0, (1, 2, 1)),      # rows in two tiles
    ((700, 64, 65), "seeded", 31, 30, 0.0, (1, 1, 1)),      # eight runs of planes
])
def test_sliding_passes_equal_per_iteration_kernels(dev, shape, kind, iters, update, bound, scaling):
    f = _fields(dev, shape, kind)
    print(shape, kind, flush=True)
    got = _solve(dev, f, shape, 0, iters, update, bound, scaling)
    want = _solve(dev, f, shape, 1, iters, update, bound, scaling)
    assert dev.torch.equal(got[0], want[0])
    assert got[1] == want[1]
    # sums of up to 2^24 float32 terms in two orders
    np.testing.assert_allclose(got[2], want[2], rtol=1e-5)


def test_sliding_passes_of_two_threads_equal_lone_solves(dev):
    """Whichever does not get the device's compute units to itself solves
    another way, with the same result."""
    from miccai2016_amd.device import DeviceContext
    shape = (64, 200, 220)
    f = [_fields(dev, shape, "seeded", seed) for seed in (5, 6)]
    want = [_solve(dev, k, shape, 1, 60, 30)[0] for k in f]
    dev.torch.cuda.synchronize()
    got, errors = [[], []], []

    def work(k):
        try:
            ctx = DeviceContext(0)
            with dev.torch.cuda.stream(dev.torch.cuda.Stream()):
                for _ in range(4):
                    got[k].append(_solve(ctx, f[k], shape, 0, 60, 30)[0])
                ctx.synchronize()
        except Exception as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for k in range(2):
        assert len(got[k]) == 4 and all(dev.torch.equal(u, want[k]) for u in got[k])
