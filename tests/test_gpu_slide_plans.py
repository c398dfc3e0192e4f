"""GPU tests: sliding passes under each kind of plan equal the per-iteration
kernels bit for bit."""
import pytest

from test_gpu_chip_fallbacks import _counts
from test_gpu_onchip import _fields, _solve
from test_slide_plan import _plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,iters", [((40, 512, 512), 33), ((64, 400, 400), 33)])
def test_one_run_of_planes_per_tile(dev, shape, iters):
    """Planes of more than 128 tiles leave the window one run of 8 planes."""
    f = _fields(dev, shape, "seeded")
    print(shape, flush=True)
    got = _solve(dev, f, shape, 0, iters, 30)
    want = _solve(dev, f, shape, 1, iters, 30)
    assert dev.torch.equal(got[0], want[0])
    assert got[1] == want[1]


def test_long_windows(dev):
    """One tile and a rare criterion: hundreds of iterations a pass."""
    shape = (4000, 32, 32)
    f = _fields(dev, shape, "axial")
    print(shape, flush=True)
    got = _solve(dev, f, shape, 0, 1010, 1000)
    want = _solve(dev, f, shape, 1, 1010, 1000)
    assert dev.torch.equal(got[0], want[0])
    assert got[1] == want[1]


def test_no_criterion_after_the_first(dev):
    """The largest interval between criteria."""
    shape = (132, 160, 160)
    f = _fields(dev, shape, "seeded")
    print(shape, flush=True)
    got = _solve(dev, f, shape, 0, 20, 2 ** 31 - 1)
    want = _solve(dev, f, shape, 1, 20, 2 ** 31 - 1)
    assert dev.torch.equal(got[0], want[0])
    assert got[1] == want[1] and len(got[2]) == 1


@pytest.mark.parametrize("shape,kind,iters,update,levels,slots", [
    ((10, 500, 500), "seeded", 33, 30, 3, 1),      # one run of planes, two columns of tiles
    ((80, 500, 501), "seeded", 25, 30, 3, 1),      # columns one voxel short
    ((17, 300, 290), "seeded", 40, 30, 6, 2),
    ((33, 256, 256), "seeded", 40, 30, 15, 4),     # little more than one window
    ((33, 256, 256), "seeded", 7, 30, 15, 4),      # one short pass
    ((300, 33, 1025), "seeded", 40, 30, 15, 4),    # three columns of tiles
    ((130, 160, 160), "axial", 62, 30, 30, 8),     # eight runs of planes
    ((700, 64, 65), "seeded", 125, 60, 60, 16),
])
def test_plans_equal_per_iteration_kernels(dev, shape, kind, iters, update, levels, slots):
    cus = dev.torch.cuda.get_device_properties(dev.device).multi_processor_count
    plan = _plan(shape, update, kind == "seeded", cus)
    if cus == 256:
        assert (plan[0], plan[3]) == (levels, slots)
    f = _fields(dev, shape, kind)
    print(shape, kind, plan, flush=True)
    at = _counts(dev)
    got = _solve(dev, f, shape, 0, iters, update)
    solves, passes, refused, given_up = _counts(dev) - at
    # of three iterations or more each
    assert solves == refused == given_up == 0 and 1 <= passes <= iters // 3 and passes >= (iters - 2) // levels
    want = _solve(dev, f, shape, 1, iters, update)
    assert dev.torch.equal(got[0], want[0])
    assert got[1] == want[1]
