"""The forward's walks by the detector's pitch: a wave's 64 rays staged whole, staged in
pieces (8-fold) or read straight from memory (4- and 2-fold), around the pitches and image
widths where the one goes over into the other (128 staged pixels of a row).  Every entry of
A comes from the same function on every walk, so the forward's are compared bit for bit
with the adjoint's, which never walks rows."""
import pytest

import test_gpu_orbit as orbit

pytestmark = pytest.mark.gpu

GEOMS = [
    (128, 101, 16, 16, 1.40, 1.0, 400.0), (129, 97, 16, 16, 1.95, 1.0, 420.0),
    (130, 92, 16, 16, 2.00, 1.0, 500.0), (131, 60, 16, 32, 3.0, 1.0, 0.0),
    (257, 185, 12, 12, 2.0, 1.0, 1000.0), (256, 270, 12, 24, 1.36, 1.0, 0.0),
    (384, 70, 8, 8, 8.0, 1.0, 1300.0), (385, 30, 8, 16, 20.0, 0.7, 0.0),
    (300, 150, 10, 20, 2.9, 1.0, 0.0), (301, 61, 7, 7, 7.0, 1.0, 800.0),
]


@pytest.mark.parametrize("flags", [1, 3, 7])
@pytest.mark.parametrize("geo", GEOMS)
def test_entries(geo, flags):
    orbit.test_entries_of_forward_and_adjoint_are_equal(geo, flags)


@pytest.mark.parametrize("flags", [1, 3, 7])
@pytest.mark.parametrize("geo", [(600, 110, 60, 60, 8.0, 1.0, 2000.0),
                                 (600, 300, 60, 120, 2.9, 1.0, 0.0)])
def test_stack_against_general_kernels(geo, flags):
    """Four views to a work-group: 2e-6 of the output's norm, the bar of the symmetric
    kernels elsewhere."""
    import torch
    from imgrecsrc_amd.projector import Projector
    P, G = Projector([geo] * 12), Projector([geo], symmetric=False)
    P.set_tune(flags=flags)
    x = torch.rand(geo[0] ** 2, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    r = G.forward(x).double()
    for s in P.unpack_sinos(P.forward(x.repeat(12))):
        assert float((s.reshape(-1).double() - r).norm() / r.norm()) < 2e-6
