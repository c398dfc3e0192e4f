"""CPU tests: the steps per launch of the gradient vector flow."""
import ctypes as C
import math
import random

import pytest

from miccai2016_amd import _lib


def plan(shape, iters=200, cus=256):
    """(steps per launch, tile sides, planes per chunk, work-groups)"""
    out = (C.c_int * 4)()
    levels = _lib.lib().mh_gvf_plan(_lib.dims3(shape), iters, cus, out)
    return levels, tuple(out[:2]), out[2], out[3]


def test_plans_cover_the_volume():
    rng = random.Random(3)
    for _ in range(2000):
        m = math.exp(rng.uniform(math.log(4), math.log(300)))
        s = tuple(max(2, round(m * rng.uniform(0.3, 3))) for _ in range(3))
        iters, cus = rng.choice([1, 2, 3, 4, 200]), rng.choice([32, 256])
        levels, tile, chunk, groups = plan(s, iters, cus)
        assert 1 <= levels <= min(iters, 4)
        if levels > 1:
            want = math.ceil(s[1] / tile[0]) * math.ceil(s[2] / tile[1]) * math.ceil(s[0] / chunk)
            assert 1 <= chunk <= s[0] and groups == want
            # the partial sums of a launch go where one step's per work-group do
            assert groups <= math.ceil(s[0] * s[1] * s[2] / 256)


@pytest.mark.parametrize("shape,levels,tile", [
    ((80, 80, 80), 1, (0, 0)), ((128, 128, 128), 2, (11, 64)), ((208, 116, 176), 2, (12, 60)),
    ((96, 96, 96), 3, (12, 50)), ((110, 110, 110), 3, (10, 58)), ((90, 95, 74), 3, (6, 74)),
    ((150, 128, 141), 4, (24, 24)), ((220, 215, 210), 4, (24, 24))])
def test_every_shape_is_taken_somewhere(shape, levels, tile):
    assert plan(shape)[:2] == (levels, tile)


def test_two_and_three_steps():
    assert plan((150, 128, 141), 2)[0] == 2 and plan((150, 128, 141), 3)[0] == 3
    assert plan((150, 128, 141), 1)[0] == 1


def test_planes_beyond_a_buffer_resource():
    """2^29 voxels a plane and more: two steps per launch."""
    assert plan((3, 30000, 20000))[0] == 2 and plan((2, 20000, 50000))[0] == 2
