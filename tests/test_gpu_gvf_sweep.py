"""GPU test: several GVF steps per launch equal one step per launch bit for bit
in every tile shape, at ragged tiles, chunks and short axes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,iters,update", [
    ((40, 30, 48), 13, 0), ((31, 25, 51), 14, 4), ((29, 21, 59), 13, 0), ((17, 13, 75), 15, 5),
    ((70, 96, 96), 13, 0), ((97, 95, 121), 15, 6), ((2, 3, 200), 11, 0), ((3, 200, 2), 9, 3),
    ((150, 2, 2), 10, 0), ((160, 161, 162), 7, 0)])
@pytest.mark.parametrize("mode", [0, 2])
def test_gvf_sweeps_equal_single_steps(dev, shape, iters, update, mode):
    from miccai2016_amd.processing.gradient_vector_flow import GvfGpu, GvfParameters
    rng = np.random.default_rng(4)
    v = rng.uniform(-0.5, 0.5, size=shape + (3,)).astype(np.float32)
    print(shape, mode, flush=True)
    outs, mags = [], []
    try:
        for m in (1, mode):
            dev.check(dev.lib.mh_gvf_set_sweep(dev.handle, m))
            seen = []
            p = GvfParameters()
            p.mu, p.tol, p.maxiter, p.update, p.normalize = 0.3, 0, iters, update, False
            p.callback = (lambda g, i, d: seen.append((i, d))) if update else None
            outs.append(GvfGpu(v, p, (2.0, 1.0, 1.5), cl_program_loader=dev).execute())
            mags.append(seen)
    finally:
        dev.check(dev.lib.mh_gvf_set_sweep(dev.handle, 0))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    assert [i for i, _ in mags[0]] == [i for i, _ in mags[1]]
    # sums of up to 2^23 positive float32 terms in two orders
    np.testing.assert_allclose([d for _, d in mags[0]], [d for _, d in mags[1]], rtol=1e-5)
