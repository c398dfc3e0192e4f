"""GPU test: each way to take several steps of the flow per launch equals one step
per launch bit for bit, with voxels of unequal sides, on volumes whose plan takes it."""
import numpy as np
import pytest

from test_gvf_plan import plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,levels,tile", [
    ((128, 128, 128), 2, (11, 64)), ((159, 130, 127), 2, (11, 64)),
    ((208, 116, 176), 2, (12, 60)), ((500, 100, 60), 2, (12, 60)),
    ((96, 96, 96), 3, (12, 50)), ((110, 110, 110), 3, (10, 58)), ((90, 95, 74), 3, (6, 74)),
    ((119, 145, 170), 3, (10, 58)), ((61, 170, 193), 3, (12, 50)),      # ragged tiles and chunks
    ((150, 128, 141), 4, (24, 24)), ((175, 183, 159), 4, (24, 24)), ((220, 215, 210), 4, (24, 24))])
def test_every_shape_equals_single_steps(dev, shape, levels, tile):
    from miccai2016_amd.processing.gradient_vector_flow import GvfGpu, GvfParameters
    cus = dev.torch.cuda.get_device_properties(dev.device).multi_processor_count
    if cus == 256:
        assert plan(shape)[:2] == (levels, tile)
    rng = np.random.default_rng(4)
    v = rng.uniform(-0.5, 0.5, size=shape + (3,)).astype(np.float32)
    print(shape, plan(shape, 200, cus), flush=True)
    outs, mags = [], []
    try:
        for mode in (1, 0):
            dev.check(dev.lib.mh_gvf_set_sweep(dev.handle, mode))
            seen = []
            p = GvfParameters()
            p.mu, p.tol, p.maxiter, p.update, p.normalize = 0.3, 0, 13, 9, False
            p.callback = lambda g, i, d: seen.append((i, d))
            outs.append(GvfGpu(v, p, (2.0, 1.0, 1.5), cl_program_loader=dev).execute())
            mags.append(seen)
    finally:
        dev.check(dev.lib.mh_gvf_set_sweep(dev.handle, 0))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    assert [i for i, _ in mags[0]] == [i for i, _ in mags[1]]
    # sums of up to 2^24 positive float32 terms in two orders
    np.testing.assert_allclose([d for _, d in mags[0]], [d for _, d in mags[1]], rtol=1e-5)
