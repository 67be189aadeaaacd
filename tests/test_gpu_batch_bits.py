"""A slice's sums are its own: whatever else a plan holds, and in either work order, a slice
has the bits of a one-slice plan.  What a launch chooses by its size (which waves and
work-groups add the same partial sums, in the same order) is met at each of its branches:
few and many items, four views to a work-group with one segment, one group, several groups
or all of a slice's rows each, partial sums in several pieces, and the beam-hardening store."""
import pytest

pytestmark = pytest.mark.gpu

MIXED = [
    (64, 91, 72, 72, 1.0, 1.0, 250.0), (93, 136, 268, 536, 1.0, 1.05, 0.0),
    (128, 129, 75, 360, 0.8, 0.9, 0.0), (100, 145, 91, 182, 1.0, 1.0, 0.0),
    (128, 185, 91, 91, 1.0, 1.0, 600.0), (224, 320, 150, 300, 1.0, 1.0, 0.0),
    (256, 367, 180, 360, 1.0, 1.0, 0.0), (300, 427, 149, 298, 1.0, 1.0, 0.0),
    (255, 363, 181, 181, 1.0, 1.0, 1000.0), (512, 729, 180, 180, 1.0, 1.0, 2000.0),
    (513, 729, 91, 91, 1.0, 1.0, 2000.0), (512, 729, 182, 364, 1.0, 1.0, 0.0),
    (640, 340, 50, 50, 2.9, 1.0, 2600.0), (641, 160, 25, 25, 6.0, 1.0, 2600.0),
    (700, 1000, 180, 180, 1.0, 1.0, 2800.0), (5, 9, 7, 7, 1.0, 1.0, 0.0),
    (40, 61, 36, 72, 1.0, 1.0, 0.0)]

# one slice, how many of it
STACKS = [
    ((64, 91, 72, 72, 1.0, 1.0, 250.0), 60),      # four views, a group each
    ((40, 61, 36, 36, 1.0, 1.0, 250.0), 50),      # two groups in one work-group
    ((128, 185, 90, 180, 1.0, 1.0, 0.0), 260),    # all groups in one work-group
    ((256, 367, 180, 360, 1.0, 1.0, 0.0), 64),    # two groups of eight each
    ((512, 729, 90, 180, 1.0, 1.0, 0.0), 3),      # one segment each
    ((512, 729, 360, 720, 1.0, 1.0, 0.0), 31),    # all groups, large slices
    ((700, 1000, 360, 360, 1.0, 1.0, 2800.0), 48),  # a group each, in two pieces
    ((64, 99, 536, 1072, 1.0, 1.0, 0.0), 970),    # all groups, in two pieces
    ((300, 427, 91, 182, 1.0, 1.0, 0.0), 20),     # 4-fold
    ((301, 427, 91, 91, 1.0, 1.0, 1300.0), 20),   # 2-fold
]


def _run(P, x, y):
    return P.forward(x), P.adjoint(y), P.fbp(y)


def _compare(geoms, which, orders):
    import torch
    from imgrecsrc_amd.projector import Projector
    B = Projector(geoms)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand(B.img_elems, device="cuda", generator=g)
    y = torch.randn(B.sino_elems, device="cuda", generator=g)
    xs, ys = B.unpack_images(x), B.unpack_sinos(y)
    alone = {i: _run(Projector([geoms[i]]), xs[i].reshape(-1), ys[i].reshape(-1)) for i in which}
    for flags in orders:
        B.set_tune(flags=flags)
        out = _run(B, x, y)
        batch = (B.unpack_sinos(out[0]), B.unpack_images(out[1]), B.unpack_images(out[2]))
        for i in which:
            for name, a, b in zip(("forward", "adjoint", "fbp"), alone[i], batch):
                assert torch.equal(a.reshape(-1), b[i].reshape(-1)), (name, geoms[i], flags)


def test_mixed_batch():
    _compare(MIXED, range(len(MIXED)), (1, 9))


@pytest.mark.parametrize("split", [1, 3])
def test_mixed_batch_of_one_shape(split):
    """The same under a shape that is set: four views to a work-group or one."""
    import torch
    from imgrecsrc_amd.projector import Projector
    shape = dict(fwd_seg=4, fwd_split=split, adj_seg=4, adj_split=split)
    B = Projector(MIXED)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand(B.img_elems, device="cuda", generator=g)
    y = torch.randn(B.sino_elems, device="cuda", generator=g)
    B.set_tune(**shape)
    out = _run(B, x, y)
    batch = (B.unpack_sinos(out[0]), B.unpack_images(out[1]), B.unpack_images(out[2]))
    for i, (xi, yi) in enumerate(zip(B.unpack_images(x), B.unpack_sinos(y))):
        P = Projector([MIXED[i]])
        P.set_tune(**shape)
        for a, b in zip(_run(P, xi.reshape(-1), yi.reshape(-1)), batch):
            assert torch.equal(a.reshape(-1), b[i].reshape(-1)), MIXED[i]


@pytest.mark.parametrize("geo,count", STACKS)
def test_stack(geo, count):
    _compare([geo] * count, (0, count // 2, count - 1), (1, 9))


@pytest.mark.parametrize("geo,count", [STACKS[2], STACKS[3], STACKS[6], STACKS[7], STACKS[9],
                                       (STACKS[4][0], 2)])
def test_gradient_of_a_stack(geo, count):
    """The ray weights stored by the forward, and so the gradient, do not depend on the
    batch either (the cost is one sum over all slices)."""
    import numpy as np
    import torch
    from imgrecsrc_amd import bhc
    from imgrecsrc_amd.projector import Projector
    B, P = Projector([geo] * count), Projector([geo])
    g = torch.Generator(device="cuda").manual_seed(2)
    alpha = torch.rand(B.img_elems, device="cuda", generator=g) * 0.02
    Imea = torch.rand(B.sino_elems, device="cuda", generator=g) * 0.9 + 0.05
    knots = np.logspace(-2, 2, 10)
    Ie = np.full(8, 0.1)
    _, grad = bhc.poissLAlpha(Imea, Ie, alpha, B, 0.5, knots)
    parts, images, sinos = (B.unpack_images(grad), B.unpack_images(alpha), B.unpack_sinos(Imea))
    assert bool(torch.isfinite(grad).all()) and bool(grad.abs().max() > 0)
    for i in (0, count - 1):
        _, one = bhc.poissLAlpha(sinos[i].reshape(-1), Ie, images[i].reshape(-1), P, 0.5, knots)
        assert torch.equal(one.reshape(-1), parts[i].reshape(-1))
