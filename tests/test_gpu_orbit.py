"""The symmetric kernels' staged reads at the sizes where they can go wrong: waves whose
rays cross more pixels than are staged at once (coarse detectors), pixels whose bins span
more than are staged at once (fine detectors), sources close to the image, images and
detectors narrower than one wave, and plans whose orbit workspaces take several chunks.

Forward and adjoint stage different things in different pieces but evaluate every entry of
A through the same function, so the entries that the two give are compared bit for bit."""
import numpy as np
import pytest

from test_gpu_projector import _proj
from test_sym_decomposition import choose_group

pytestmark = pytest.mark.gpu

GEOMS = [
    (150, 70, 40, 40, 5.0, 1.0, 400.0),     # coarse fan detector: rows in several pieces
    (151, 66, 40, 80, 6.0, 0.8, 0.0),       # coarse parallel, folded
    (400, 140, 22, 22, 3.1, 1.1, 1500.0),   # coarse, 4-fold
    (300, 131, 15, 15, 2.6, 1.0, 700.0),    # coarse, 2-fold, both walks
    (65, 700, 16, 16, 0.15, 1.0, 200.0),    # fine fan detector: bins in several pieces
    (64, 650, 20, 40, 0.14, 1.3, 0.0),      # fine parallel, folded
    (60, 500, 9, 9, 0.2, 0.9, 150.0),       # fine, 2-fold
    (60, 81, 24, 24, 1.0, 1.0, 45.0),       # the source just outside the image's disc
    (61, 64, 13, 13, 1.4, 1.0, 45.5),
    (5, 4, 8, 8, 1.0, 1.0, 9.0),            # smallest image and detector
    (6, 5, 6, 12, 1.0, 1.0, 0.0),
    (33, 65, 12, 12, 0.6, 1.0, 90.0),       # one pixel / one bin past a tile
    (130, 193, 10, 20, 1.0, 1.0, 0.0),
]


@pytest.mark.parametrize("flags", [1, 3, 7])
@pytest.mark.parametrize("geo", GEOMS)
def test_entries_of_forward_and_adjoint_are_equal(geo, flags):
    """Columns of A at 24 pixels and rows at up to three rays through each of them."""
    import torch
    n, W, npj = geo[:3]
    P = _proj(geo, flags)
    assert P.modes() == [choose_group(geo[3], geo[2], geo[6] > 0, flags, n=n)[0]] != [0]
    rng = np.random.default_rng(7)
    lo = n // 2 - (n - 1) // 2  # first row / column the projector reads
    px = [r * n + c for r, c in rng.integers(lo, n, (20, 2))]
    px += [lo * n + lo, lo * n + n - 1, (n - 1) * n + lo, n * n - 1]  # the corners
    for seg, split in ((8, 1), (2, 3)):
        P.set_tune(fwd_seg=seg, adj_seg=seg, fwd_split=split, adj_split=split)
        cols = []
        for p in px:
            x = torch.zeros(n * n, device="cuda")
            x[p] = 1.0
            cols.append(P.forward(x).cpu().numpy())
        cols = np.stack(cols)
        rays = set()
        for c in cols:
            hit = np.flatnonzero(c)
            rays.update(rng.choice(hit, min(3, hit.size), replace=False).tolist())
        assert len(rays) > 8
        for r in sorted(rays):
            y = torch.zeros(npj * W, device="cuda")
            y[r] = 1.0
            row = P.adjoint(y).cpu().numpy()
            assert np.array_equal(row[px], cols[:, r]), (geo, flags, seg, r)


def test_orbit_workspace_chunks_match_single_slices():
    """Two slices whose orbit images do not fit one chunk of workspace (2^30 floats) run in
    two chunks: the same bits as one-slice plans."""
    import torch
    from imgrecsrc_amd.projector import Projector
    geoms = [(11600, 9, 8, 8, 300.0, 1.0, 60000.0), (11600, 7, 4, 8, 500.0, 1.0, 0.0)]
    g = torch.Generator(device="cuda").manual_seed(5)
    B = Projector(geoms)
    x = torch.rand(B.img_elems, device="cuda", generator=g)
    y = torch.rand(B.sino_elems, device="cuda", generator=g)
    s, b = B.unpack_sinos(B.forward(x)), B.unpack_images(B.adjoint(y))
    xs, ys = B.unpack_images(x), B.unpack_sinos(y)
    for i, geo in enumerate(geoms):
        P = Projector([geo])
        assert torch.equal(P.forward(xs[i].reshape(-1)), s[i].reshape(-1))
        assert torch.equal(P.adjoint(ys[i].reshape(-1)), b[i].reshape(-1))
        assert bool(torch.isfinite(s[i]).all())
