"""GPU test: the eigensolver and the vesselness update read and write voxels in
pairs of floats where the arrays are aligned to them, one by one elsewhere, with
the same results."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 257, 70001])
@pytest.mark.parametrize("off_in,off_out", [(0, 0), (2, 0), (1, 0), (0, 1), (3, 5)])
def test_eigs_and_vesselness_at_any_alignment(dev, n, off_in, off_out):
    torch = dev.torch
    h = np.random.default_rng(n).normal(size=6 * n).astype(np.float32)
    out = []
    for a, b in ((0, 0), (off_in, off_out)):
        src, dst = dev.zeros(6 * n + 8), dev.zeros(6 * n + 8)
        src[a:a + 6 * n] = dev.upload(h)
        norm, val, quat = dev.zeros(1), dev.zeros(n), dev.zeros(3 * n)
        e = dst[b:b + 6 * n]
        dev.check(dev.lib.mh_eigs(dev.handle, dev.ptr(src[a:a + 6 * n]), dev.ptr(e), n, 20,
                                  dev.ptr(norm), dev.stream))
        dev.check(dev.lib.mh_update_vesselness(dev.handle, dev.ptr(val), dev.ptr(quat), dev.ptr(e), n,
                                               0.5, 0.5, -1.0, dev.ptr(norm), 1, dev.stream))
        out.append((e.clone(), norm, val, quat))
        assert not dst[:b].any() and not dst[b + 6 * n:].any()
    for x, y in zip(*out):
        assert torch.equal(x, y)
    lam = out[0][0].reshape(n, 6)[:, :3]
    assert torch.equal(out[0][1], (lam ** 2).sum(1).sqrt().max().reshape(1)) or \
        abs(float(out[0][1]) / float((lam.double() ** 2).sum(1).sqrt().max()) - 1) < 4e-7
