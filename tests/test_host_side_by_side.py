"""CPU test: a ragged set is left to the solvers that need no room of their own on
the device where the side-by-side launch finds none."""
import numpy as np
import pytest
import torch

from miccai2016_amd.processing.continuous_cut_anisotropic_gpu import CmfCutQAnisotropicGpu


class FullDevice:
    """A context whose device has no room; a call into the library fails the test."""
    torch, handle, stream = torch, None, None
    ptr = staticmethod(lambda t: None)

    def bytes(self, nbytes):
        raise torch.OutOfMemoryError("no room")

    @property
    def lib(self):
        pytest.fail("called without its workspace")


def test_no_room_for_the_launch():
    cut = CmfCutQAnisotropicGpu(CmfCutQAnisotropicGpu.CutParameters(), FullDevice())
    shapes, offsets = [(4, 5, 6), (3, 3, 3)], [0, 120]
    f = torch.zeros(147)
    got = cut._solve_side_by_side(f, f, f, f, f, shapes, offsets, np.ones(3), None)
    assert got == [None, None]
