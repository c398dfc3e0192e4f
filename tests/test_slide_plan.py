"""CPU tests: the plans of the sliding passes keep within the device, and each
is one the kernel takes."""
import ctypes as C
import itertools
import os
import subprocess
import sys

import numpy as np
import pytest

from miccai2016_amd import _lib

LDS = 160 * 1024
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _plan(shape, update, seeded=0, cus=256, iters=500):
    """(levels, tile sides, tiles, runs of planes, LDS bytes)"""
    P = _lib.CmfParams()
    P.rcc, P.const_evals, P.num_iter, P.update = 5.0, 1, iters, update
    for k, e in enumerate((1.0, 10 ** -1.5, 10 ** -1.5)):
        P.rs[k], P.ss[k], P.sqev[k] = 1.0, 0.16, np.sqrt(e)
    out = (C.c_int * 6)()
    levels = _lib.lib().mh_cmf_slide_plan(_lib.dims3(shape), C.byref(P), seeded, cus, out)
    return levels, tuple(out[:2]), tuple(out[2:4]), out[4], out[5]


def test_long_windows_keep_within_the_lds():
    """One tile, a long axis 0 and a rare criterion: a window of as many runs of
    planes as the masks beside them leave room for."""
    for shape, update in itertools.product([(4000, 32, 32), (9000, 30, 29), (60000, 16, 16)],
                                           [31, 200, 840, 1000, 5000]):
        for seeded in (0, 1):
            levels, _, tiles, slots, lds = _plan(shape, update, seeded)
            if levels:
                assert lds <= LDS, (shape, update)
                assert tiles[0] * tiles[1] * slots <= 256
                assert levels <= 4 * slots - 1
    assert _plan((4000, 32, 32), 1000)[0] >= 3   # still taken


def _in_subprocess(code):
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT,
                       env=dict(os.environ, PYTHONPATH=os.pathsep.join([ROOT, os.path.dirname(__file__)])))
    return r.returncode, r.stdout.strip(), r.stderr[-500:]


@pytest.mark.parametrize("seeded", [0, 1])
def test_criteria_rarer_than_any_window(seeded):
    """Up to the largest interval, which some programs switch the criterion off
    with, the plan is that of the rarest criterion a window can reach."""
    intervals = [1024, 5000, 2 ** 29, 2 ** 31 - 5, 2 ** 31 - 2, 2 ** 31 - 1]
    shapes = [(132, 160, 160), (256, 256, 256), (64, 300, 300), (4000, 32, 32), (40, 512, 512)]
    rc, out, err = _in_subprocess(
        "from test_slide_plan import _plan\n"
        f"for s in {shapes}: print([_plan(s, k, {seeded}) for k in {intervals}])")
    assert rc == 0, err   # (an integer division by zero ends the process)
    taken = 0
    for line, shape in zip(out.splitlines(), shapes):
        plans = eval(line)
        assert all(p == plans[0] for p in plans), (shape, plans)
        taken += plans[0][0] > 0
    assert taken >= 2
