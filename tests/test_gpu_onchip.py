"""GPU tests: solves that stay on the chip (the automatic method of volumes
that fit) equal the per-iteration kernels bit for bit."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ATV = 10 ** -1.5


def _fields(dev, shape, kind, seed=3):
    """(u0, eigs, alpha, cs, ct, labels, const_sqevals) device tensors."""
    rng = np.random.default_rng(seed)
    up = lambda *s: dev.upload(rng.random(s, dtype=np.float32))
    u0, cs, ct, alpha = up(*shape), up(*shape), up(*shape), 0.5 * up(*shape)
    q = 6 * (up(*shape, 3) - 0.5)
    labels = None
    if "seeded" in kind:
        marks = rng.integers(0, 4, shape) * (rng.random(shape) < 0.1)
        labels = dev.upload(marks, dtype=np.uint8)
    if "pointwise" in kind:
        return u0, dev.torch.cat([(0.1 + 0.9 * up(*shape, 3)).sqrt(), q], -1).contiguous(), alpha, cs, \
            ct, labels, None
    eigs = (1, 0.3, 0.1) if "general" in kind else (1, ATV, ATV)
    return u0, q, alpha, cs, ct, labels, np.sqrt(eigs)


def _solve(dev, f, shape, mode, iters, update, bound=0.0, scaling=(1, 1, 1)):
    from miccai2016_amd.processing.continuous_cut_anisotropic_gpu import CmfCutQAnisotropicGpu
    p = CmfCutQAnisotropicGpu.CutParameters()
    p.num_iter, p.update, p.error_bound, p.steps = iters, update, bound, 0.16
    cut = CmfCutQAnisotropicGpu(p, dev)
    u = f[0].clone()
    try:
        dev.check(dev.lib.mh_cmf_set_sweep(dev.handle, mode, 0, 0))
        cut.execute_device(u, *f[1:5], labels=f[5], const_sqevals=f[6], shape=shape, scaling=scaling)
    finally:
        dev.check(dev.lib.mh_cmf_set_sweep(dev.handle, 0, 0, 0))
    r = cut.last_result
    return u, (r.iterations, r.stopped, r.ncrit), cut.last_criteria


@pytest.mark.parametrize("shape,kind,iters,update,bound,scaling", [
    ((8, 8, 8), "axial", 7, 3, 0.0, (1, 1, 1)),            # one work-group
    ((1, 1, 50), "axial", 9, 2, 0.0, (1, 1, 1)),           # axes of length one
    ((3, 700, 2), "axial", 30, 5, 0.0, (1, 1, 1)),         # split along axis 1 only
    ((2, 3, 900), "axial", 30, 5, 0.0, (1, 1, 1)),         # split along axis 2
    ((24, 30, 37), "axial", 400, 1, 1e-4, (1, 1, 1)),      # stops at a criterion
    ((33, 61, 67), "general", 40, 10, 0.0, (2, 1, 1)),
    ((80, 96, 72), "pointwise", 25, 10, 0.0, (2, 1, 1.5)),
    ((50, 40, 30), "pointwise seeded", 25, 10, 0.0, (1, 1, 1)),
    ((101, 117, 90), "seeded", 25, 30, 0.0, (1, 1, 1)),    # ragged bricks on every axis
    ((9, 300, 290), "axial", 25, 13, 0.0, (1, 1, 1)),
    ((128, 128, 128), "axial", 25, 30, 0.0, (1, 1, 1)),    # every compute unit full
    ((129, 128, 129), "axial", 12, 5, 0.0, (1, 1, 1)),     # beyond it
])
def test_onchip_solves_equal_per_iteration_kernels(dev, shape, kind, iters, update, bound, scaling):
    f = _fields(dev, shape, kind)
    print(shape, kind, flush=True)
    got = _solve(dev, f, shape, 0, iters, update, bound, scaling)
    want = _solve(dev, f, shape, 1, iters, update, bound, scaling)
    assert dev.torch.equal(got[0], want[0])
    assert got[1] == want[1]
    # sums of up to 2^21 float32 terms in two orders
    np.testing.assert_allclose(got[2], want[2], rtol=1e-5)


def test_onchip_nan_stops_and_spreads_as_in_the_kernels(dev):
    shape = (20, 33, 40)
    f = _fields(dev, shape, "axial")
    f[1][3, 32, 39, 1] = float("nan")
    got = _solve(dev, f, shape, 0, 50, 4)
    want = _solve(dev, f, shape, 1, 50, 4)
    assert got[1] == want[1] and got[1][1] == 1
    assert dev.torch.equal(got[0].isnan(), want[0].isnan())
    assert dev.torch.equal(got[0].nan_to_num(), want[0].nan_to_num())


@pytest.mark.parametrize("shape,solves", [((24, 30, 37), 37), ((64, 64, 64), 9), ((128, 128, 120), 2)])
def test_onchip_batches_equal_lone_solves(dev, shape, solves):
    """Solves side by side (several per launch) and one after another."""
    from miccai2016_amd.processing.continuous_cut_anisotropic_gpu import CmfCutQAnisotropicGpu
    u0, q, _, cs, ct, _, sq = _fields(dev, shape, "axial")
    gms = 4 * dev.upload(np.random.default_rng(1).random(shape, dtype=np.float32))
    w, d = np.geomspace(0.02, 2, solves).astype(np.float32), np.geomspace(1, 30, solves).astype(np.float32)
    p = CmfCutQAnisotropicGpu.CutParameters()
    p.num_iter, p.update, p.error_bound, p.steps = 40, 7, 2e-3, 0.16
    cut = CmfCutQAnisotropicGpu(p, dev)
    u = u0.reshape(1, -1).repeat(solves, 1)
    cut.execute_batched_device(u, solves, w, d, q, gms, cs, ct, shape, (1, ATV, ATV))
    res = [(r.iterations, r.stopped, r.ncrit) for r in cut.last_result]
    a = dev.empty(u0.numel())
    for s in range(solves):
        dev.check(dev.lib.mh_nonterminal_weight(dev.handle, dev.ptr(gms), u0.numel(), float(w[s]),
                                                float(d[s]), dev.ptr(a), dev.stream))
        want = _solve(dev, (u0, q, a, cs, ct, None, sq), shape, 1, 40, 7, 2e-3)
        assert dev.torch.equal(u[s], want[0].reshape(-1)), s
        assert res[s] == want[1], s


def test_onchip_solves_of_two_threads_equal_lone_solves(dev):
    """Two threads with their own contexts and streams: whichever does not get
    the device's compute units to itself solves another way, with the same
    result."""
    from miccai2016_amd.device import DeviceContext
    shape = (60, 64, 70)
    f = [_fields(dev, shape, "axial", seed) for seed in (5, 6)]
    want = [_solve(dev, k, shape, 1, 200, 10)[0] for k in f]
    dev.torch.cuda.synchronize()
    got, errors = [[], []], []

    def work(k):
        try:
            ctx = DeviceContext(0)
            with dev.torch.cuda.stream(dev.torch.cuda.Stream()):
                for _ in range(6):
                    got[k].append(_solve(ctx, f[k], shape, 0, 200, 10)[0])
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
        assert len(got[k]) == 6 and all(dev.torch.equal(u, want[k]) for u in got[k])
