"""GPU tests: sliding passes under each kind of plan equal the per-iteration
kernels bit for bit."""
import pytest

from test_gpu_onchip import _fields, _solve

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
