"""GPU tests: solves that cannot have the device's compute units to themselves
take other methods, with the same results."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_onchip import ATV, _fields, _solve

pytestmark = pytest.mark.gpu


def _counts(dev):
    """Solves finished on the chip, sliding passes launched, launches refused and
    given up."""
    c = (C.c_int64 * 4)()
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
    solves, _, refused, _ = _counts(dev) - at
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
    solves, slid, refused, given_up = _counts(dev) - at
    assert (solves == 0 and slid > 0 if passes else solves == 1 and slid == 0)
    assert refused == given_up == 0


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
        solves, _, refused, _ = _counts(dev) - at
        assert (solves == 5 and refused == 0) if n == 0 else (solves < 5 and refused > 0)
    assert torch.equal(*outs)


@pytest.fixture
def lost_group(dev):
    """Sets the solve or pass from which a work-group is missing."""
    yield lambda n: dev.check(dev.lib.mh_cmf_set_lost_group(dev.handle, n))
    dev.check(dev.lib.mh_cmf_set_lost_group(dev.handle, -1))


@pytest.mark.parametrize("shape,kind,iters,update,bound,lost", [
    ((96, 96, 96), "axial", 40, 7, 0.0, 0),
    ((60, 64, 70), "pointwise seeded", 25, 10, 0.0, 0),
    ((33, 61, 67), "general", 40, 1, 0.0, 0),
    ((24, 30, 37), "axial", 400, 1, 1e-4, 0),
    ((256, 256, 256), "axial", 70, 30, 0.0, 0),            # the first sliding pass
    ((256, 256, 256), "axial", 70, 30, 0.0, 3),            # a later one
    ((64, 200, 220), "seeded", 65, 30, 0.0, 1),
    ((80, 500, 501), "seeded", 35, 30, 0.0, 5),
    ((100, 250, 250), "axial", 300, 10, 6e-3, 0),          # stops at a criterion
])
def test_solves_given_up_are_done_again(dev, lost_group, shape, kind, iters, update, bound, lost):
    f = _fields(dev, shape, kind)
    print(shape, kind, lost, flush=True)
    want = _solve(dev, f, shape, 1, iters, update, bound)
    lost_group(lost)
    at = _counts(dev)
    got = _solve(dev, f, shape, 0, iters, update, bound)
    solves, passes, refused, given_up = _counts(dev) - at
    assert solves == refused == 0 and given_up >= 1 and passes >= lost
    assert dev.torch.equal(got[0], want[0])
    assert got[1] == want[1]
    # sums of up to 2^24 float32 terms in two orders
    np.testing.assert_allclose(got[2], want[2], rtol=1e-5)


def test_sets_and_batches_given_up_are_done_again(dev, lost_group):
    from miccai2016_amd.processing.continuous_cut_anisotropic_gpu import CmfCutQAnisotropicGpu
    torch = dev.torch
    p = CmfCutQAnisotropicGpu.CutParameters()
    p.num_iter, p.update, p.error_bound, p.steps = 40, 7, 2e-3, 0.16
    cut = CmfCutQAnisotropicGpu(p, dev)
    shapes = [(64, 64, 64), (33, 61, 67), (9, 12, 15), (70, 60, 50)]
    f = [_fields(dev, s, "axial", seed) for seed, s in enumerate(shapes)]
    want = [_solve(dev, k, s, 1, 40, 7, 2e-3)[0].reshape(-1) for k, s in zip(f, shapes)]
    pack = lambda k: torch.cat([x[k].reshape(-1) for x in f])
    offs = np.concatenate([[0], np.cumsum([w.numel() for w in want])[:-1]])
    shape, solves = (24, 30, 37), 90
    u0, q, _, cs, ct, _, _ = _fields(dev, shape, "axial")
    gms = 4 * dev.upload(np.random.default_rng(1).random(shape, dtype=np.float32))
    w = np.geomspace(0.02, 2, solves).astype(np.float32)
    d = np.geomspace(1, 30, solves).astype(np.float32)
    batches = []
    for n in (-1, 0):
        lost_group(n)
        at = _counts(dev)
        u = pack(0)
        cut.execute_ragged_device(u, pack(1), pack(2), pack(3), pack(4), shapes, offs, (1, ATV, ATV))
        assert torch.equal(u, torch.cat(want)), n
        v = u0.reshape(1, -1).repeat(solves, 1)
        cut.execute_batched_device(v, solves, w, d, q, gms, cs, ct, shape, (1, ATV, ATV))
        batches.append((v, [(r.iterations, r.stopped, r.ncrit) for r in cut.last_result]))
        done, _, refused, given_up = _counts(dev) - at
        assert refused == 0
        # the set's launch is undone as a whole; of the batch's solves, side by side, some
        # have all their work-groups
        assert (done == 4 + solves and given_up == 0) if n < 0 else 0 < done < solves and given_up == 2
    for v, res in batches[1:]:
        assert torch.equal(v, batches[0][0]) and res == batches[0][1]
