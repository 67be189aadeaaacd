"""The ways the symmetric adjoint reads its bins.  A small plan's adjoint gathers them from
the sinogram, a larger one reads the orbit sinogram; a parallel slice whose tiles' bins fit one
staged piece (pitch above about 0.39) reads them without looking at the range, others check
it and stage what is left piece by piece, and fan slices always check.  All of them give a pixel
the same weights and values in the same order: adjoint and FBP are compared bit for bit, or
against the general kernels at the symmetric kernels' bar."""
import pytest

import test_gpu_orbit as orbit
from test_gpu_projector import WINDOW_CASES

pytestmark = pytest.mark.gpu

# enough adjoint steps on its own (188e3) for its plan to read orbit sinograms
COMPANION = (200, 290, 555, 555, 1.0, 1.0, 700.0)


@pytest.mark.parametrize("geo,flags", WINDOW_CASES)
def test_gathered_and_orbit_bins_are_equal(geo, flags):
    import torch
    from imgrecsrc_amd.phantom import gaussian
    from imgrecsrc_amd.projector import Projector
    one, two = Projector([geo]), Projector([geo, COMPANION])
    y = torch.from_numpy(gaussian((geo[2], geo[1]), 13)).cuda().reshape(-1)
    both = torch.cat([y, torch.zeros(COMPANION[1] * COMPANION[2], device="cuda")])
    for shape in (dict(), dict(adj_seg=4, adj_split=3), dict(adj_seg=1, adj_split=2)):
        for P in (one, two):
            P.set_tune(flags=flags, **shape)
        for a, b in ((one.adjoint(y), two.adjoint(both)), (one.fbp(y), two.fbp(both))):
            assert torch.equal(a, two.unpack_images(b)[0].reshape(-1)), shape
            assert not torch.any(two.unpack_images(b)[1])


EDGE = [(n, int(1.5 * n / p), P, 2 * P, p, rate, 0.0)
        for n, P in ((40, 12), (63, 15)) for p, rate in
        ((0.30, 1.0), (0.385, 1.0), (0.391, 1.0), (0.392, 1.0), (0.40, 1.0), (0.45, 4.0), (0.5, 3.0))]


@pytest.mark.parametrize("flags", [1, 3, 7])
@pytest.mark.parametrize("geo", EDGE)
def test_around_one_staged_piece(geo, flags):
    import torch
    from imgrecsrc_amd.projector import Projector
    orbit.test_entries_of_forward_and_adjoint_are_equal(geo, flags)
    P, G = Projector([geo]), Projector([geo], symmetric=False)
    P.set_tune(flags=flags)
    y = torch.rand(P.sino_elems, device="cuda", generator=torch.Generator("cuda").manual_seed(4))
    a, r = P.adjoint(y).double(), G.adjoint(y).double()
    assert float((a - r).norm() / r.norm()) < 2e-6
