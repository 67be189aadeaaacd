"""A small plan's own launch shapes.  A one-slice plan under 225 pixels wide gathers the
adjoint's bins from the sinogram and, with few forward items, walks with sixteen waves; in a
plan of many adjoint steps the same slice reads the orbit sinogram and takes up to its own
number of work-groups of eight waves.  Both add the same numbers in the same order, so every
slice has the bits it has alone; and one-slice plans agree with the general kernels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (200^2, 555 odd views: 188e3 adjoint steps on its own)
BIG = (200, 290, 555, 555, 1.0, 1.0, 700.0)
SLICES = [
    (64, 91, 72, 72, 1.0, 1.0, 250.0),      # D4 fan: one work-group an item
    (93, 135, 360, 360, 1.0, 1.0, 400.0),   # D4 fan, several
    (93, 136, 536, 1072, 1.0, 1.05, 0.0),   # D4 half turn, even detector, more than 256 items
    (128, 129, 150, 720, 0.8, 0.9, 0.0),    # D4 arc: views without rows
    (60, 90, 302, 604, 1.0, 1.0, 0.0),      # D4 half turn
    (100, 145, 181, 362, 1.0, 1.0, 0.0),    # V4 half turn
    (72, 75, 90, 90, 1.3, 1.0, 300.0),      # V4 fan, a detector that cuts the corners off
    (128, 185, 181, 181, 1.0, 1.0, 600.0),  # Z2 fan
    (5, 9, 7, 7, 1.0, 1.0, 0.0),            # Z2 parallel, the smallest image
    (224, 320, 300, 600, 1.0, 1.0, 0.0),    # the widest
]


def test_slices_keep_their_bits_in_a_batch():
    import torch
    from imgrecsrc_amd.projector import Projector
    geoms = SLICES + [BIG]
    B = Projector(geoms)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.rand(B.img_elems, device="cuda", generator=g)
    y = torch.randn(B.sino_elems, device="cuda", generator=g)
    s, b = B.unpack_sinos(B.forward(x)), B.unpack_images(B.adjoint(y))
    f = B.unpack_images(B.fbp(y))
    xs, ys = B.unpack_images(x), B.unpack_sinos(y)
    for i, geo in enumerate(geoms):
        P = Projector([geo])
        for _ in range(2):
            assert torch.equal(P.forward(xs[i].reshape(-1)), s[i].reshape(-1)), geo
            assert torch.equal(P.adjoint(ys[i].reshape(-1)), b[i].reshape(-1)), geo
            assert torch.equal(P.fbp(ys[i].reshape(-1)), f[i].reshape(-1)), geo


@pytest.mark.parametrize("geo", SLICES)
def test_against_general_kernels(geo):
    """Both paths hold FP32 weights and compensated sums: 2e-6 of the output's norm, the bar
    of the symmetric kernels elsewhere."""
    import torch
    from imgrecsrc_amd.projector import Projector
    P, G = Projector([geo]), Projector([geo], symmetric=False)
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.rand(P.img_elems, device="cuda", generator=g)
    y = torch.rand(P.sino_elems, device="cuda", generator=g)
    for a, r in ((P.forward(x), G.forward(x)), (P.adjoint(y), G.adjoint(y))):
        a, r = a.double(), r.double()
        assert float((a - r).norm() / r.norm()) < 2e-6
