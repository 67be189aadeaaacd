"""The forward whose work-groups take four neighbouring canonical views, at the sizes where
it can go wrong: fewer than four views left at the end of a walk, both walks, rays that
cross more pixels than are staged (walked view by view), images narrower than the staged
columns, and row splits that leave empty shares.  A large empty slice of the same group in
the plan brings the launch to the size from which this kernel is used.

An image of one pixel gives single entries of A, which no order of summation changes: they
are compared bit for bit with the kernel that walks one view per work-group.  On a random
image both add at most 40 products of a block of rows in FP32 (2^-24 each) and the blocks
with compensation: 40 * 2^-24 = 2.4e-6 of the largest sum."""
import numpy as np
import pytest

from test_gpu_orbit import GEOMS
from test_sym_decomposition import choose_group

pytestmark = pytest.mark.gpu

BIG = {1: (1024, 1024, 136, 136, 1.0, 1.0, 4096.0), 2: (1024, 1024, 150, 150, 1.0, 1.0, 4096.0),
       3: (1023, 1024, 75, 75, 1.0, 1.0, 4096.0)}
MORE = [(64, 91, 72, 72, 1.0, 1.0, 250.0), (255, 367, 181, 181, 1.0, 1.0, 900.0),
        (200, 300, 30, 240, 1.0, 1.0, 0.0), (320, 280, 50, 50, 2.2, 1.0, 1300.0),
        (700, 340, 26, 26, 2.9, 1.0, 2100.0)]


@pytest.mark.parametrize("flags", [1, 3, 7])
@pytest.mark.parametrize("geo", GEOMS + MORE)
def test_equal_to_one_view_per_work_group(geo, flags):
    import torch
    from imgrecsrc_amd.projector import Projector
    n, W, npj = geo[:3]
    grp = choose_group(geo[3], npj, geo[6] > 0, flags, n=n)[0]
    if not grp:
        pytest.skip("no symmetry used")
    one, two = Projector([geo]), Projector([BIG[grp], geo])
    for P in (one, two):
        P.set_tune(flags=flags)
    assert one.modes() == [grp] and two.modes() == [grp, grp]
    one.set_tune(fwd_seg=2, fwd_split=1)
    lead = BIG[grp][0] ** 2
    rng = np.random.default_rng(11)
    lo = n // 2 - (n - 1) // 2
    px = [r * n + c for r, c in rng.integers(lo, n, (8, 2))] + [lo * n + lo, n * n - 1]
    images = [torch.rand(n * n, device="cuda", generator=torch.Generator("cuda").manual_seed(3))]
    for p in px:
        x = torch.zeros(n * n, device="cuda")
        x[p] = 1.0
        images.append(x)
    for split in (1, 3, 8):
        two.set_tune(fwd_seg=4, fwd_split=split)
        for i, x in enumerate(images):
            a = one.forward(x)
            b = two.forward(torch.cat([torch.zeros(lead, device="cuda"), x]))
            assert not torch.any(b[:-npj * W])
            b = b[-npj * W:]
            if i:
                assert torch.equal(a, b)
            else:
                err = ((a - b).abs().max() / a.abs().max().clamp_min(1e-30)).item()
                print(f"{geo} group {grp} split {split}: {err:.2e}")
                assert err <= 2.4e-6
