"""GPU tests: solves that cannot have the device's compute units to themselves
take other methods, with the same results."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_onchip import ATV, _fields, _solve

pytestmark = pytest.mark.gpu


def _counts(dev):
    """Solves finished on the chip, sliding passes launched, launches refused."""
    c = (C.c_int64 * 3)()
    dev.check(dev.lib.mh_cmf_chip_counts(dev.handle, C.byref(c)))
    return np.array(c[:])


@pytest.fixture
def units(dev):
    """Sets the compute units that plans count on."""
    yield lambda n: dev.check(dev.lib.mh_cmf_set_chip_units(dev.handle, n))
    dev.check(dev.lib.mh_cmf_set_chip_units(dev.handle, 0))


@pytest.mark.parametrize("shape,kind", [
    ((150, 150, 150), "axial"), ((96, 128, 128), "pointwise"),   # beyond one device's registers
    ((256, 256, 256), "axial"), ((64, 200, 220), "seeded")])     # sliding passes
def test_launches_the_device_refuses(dev, units, shape, kind):
    """Plans for twice the device's compute units need more work-groups at once
    than it holds."""
    f = _fields(dev, shape, kind)
    print(shape, kind, flush=True)
    want = _solve(dev, f, shape, 1, 40, 30)
    units(512)
    at = _counts(dev)
    got = _solve(dev, f, shape, 0, 40, 30)
    solves, _, refused = _counts(dev) - at
    assert solves == 0 and refused >= 1
    assert dev.torch.equal(got[0], want[0])
    assert got[1] == want[1]


@pytest.mark.parametrize("shape,kind,passes", [
    ((128, 128, 128), "axial", 0), ((80, 96, 72), "pointwise", 0),
    ((256, 256, 256), "axial", 1), ((64, 200, 220), "seeded", 1)])
def test_methods_of_the_device_to_itself(dev, shape, kind, passes):
    f = _fields(dev, shape, kind)
    at = _counts(dev)
    _solve(dev, f, shape, 0, 40, 30)
    solves, slid, refused = _counts(dev) - at
    assert (solves == 0 and slid > 0 if passes else solves == 1 and slid == 0) and refused == 0


@pytest.mark.parametrize("n", [7, 32, 100])
def test_plans_for_a_part_of_the_device(dev, units, n):
    shape = (33, 61, 67)
    f = _fields(dev, shape, "axial")
    want = _solve(dev, f, shape, 1, 25, 5)
    units(n)
    got = _solve(dev, f, shape, 0, 25, 5)
    assert dev.torch.equal(got[0], want[0]) and got[1] == want[1]


def test_refused_sets_and_batches(dev, units):
    from miccai2016_amd.processing.continuous_cut_anisotropic_gpu import CmfCutQAnisotropicGpu
    torch = dev.torch
    p = CmfCutQAnisotropicGpu.CutParameters()
    p.num_iter, p.update, p.error_bound, p.steps = 40, 30, 0.0, 0.16
    cut = CmfCutQAnisotropicGpu(p, dev)
    shapes = [(96, 96, 96), (90, 95, 100), (99, 80, 90)]   # 12 work-groups of each 8 planes
    f = [_fields(dev, s, "axial", seed) for seed, s in enumerate(shapes)]
    want = [_solve(dev, k, s, 1, 40, 30)[0].reshape(-1) for k, s in zip(f, shapes)]
    pack = lambda k: torch.cat([x[k].reshape(-1) for x in f])
    offs = np.concatenate([[0], np.cumsum([w.numel() for w in want])[:-1]])
    u0, q, _, cs, ct, _, _ = f[0]
    gms, w, d = 4 * f[0][2] ** 2, np.float32([0.3, 0.6]), np.float32([2.0, 9.0])
    outs = []
    for n in (0, 1000):
        units(n)
        at = _counts(dev)
        u = pack(0)
        cut.execute_ragged_device(u, pack(1), pack(2), pack(3), pack(4), shapes, offs, (1, ATV, ATV))
        assert torch.equal(u, torch.cat(want)), n
        v = u0.reshape(1, -1).repeat(2, 1)
        cut.execute_batched_device(v, 2, w, d, q, gms, cs, ct, shapes[0], (1, ATV, ATV))
        outs.append(v)
        solves, _, refused = _counts(dev) - at
        assert (solves == 5 and refused == 0) if n == 0 else (solves < 5 and refused > 0)
    assert torch.equal(*outs)
