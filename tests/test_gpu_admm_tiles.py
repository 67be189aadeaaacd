"""The two-tap ADMM's output launch on images of more tiles than it has work-groups (1024
tiles of 32^2): a work-group then synthesises several tiles through the same LDS.  With two
levels the next tile's coarse level is written right where waves may still be reading this
tile's approximations, so the barrier between the tiles is what this guards; one and three
levels go the other ways through the loop.

Two taps do not cross from one image of a stack into the next, so a stack is the same solve
as the tall image.  FP64 restatement, at the bar of the other ADMM cases (FP32 output, 1e-6
of the largest value)."""
import numpy as np
import pytest

from oracle import wavelet_oracle as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [1, 2, 3])
@pytest.mark.parametrize("rows,cols,batch", [(1056, 1088, 1), (512, 480, 9)])
def test_output_of_many_tiles(L, rows, cols, batch):
    import torch
    from imgrecsrc_amd.wavelet import Wavelet, daubcqf
    assert (rows // 32) * (cols // 32) * batch > 1024
    h = daubcqf(2)[0]
    a = np.random.default_rng(L).standard_normal((batch * rows, cols)).astype(np.float32)
    w = Wavelet(rows, cols, h, L, batch=batch)
    u, most = 0.3, 2
    ref, itr_ref = W.admm(a.astype(np.float64), u, h, L, 1e-12, most)
    x = torch.from_numpy(a.ravel()).cuda()
    for _ in range(3):
        out, itr = w.admm(x, u, relativeTol=1e-12, maxItr=most)
        assert itr == itr_ref
        err = np.abs(out.cpu().numpy().reshape(a.shape) - ref).max() / np.abs(ref).max()
        print(f"{batch}x{rows}x{cols} L={L}: {err:.2e}")
        assert err <= 1e-6
