"""The TV iteration's launch over several work-groups: a group's pixels at its edges (256,
one past, an image of 1024 groups and past it, where a group has two runs of pixels), a
stack, and iteration counts at the edges of the host's batches of eight, against the FP64
oracle at the bar of the other TV cases (images are FP32, 6e-8 of their largest value)."""
import numpy as np
import pytest

from oracle import tv_oracle as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tv", ["iso", "l1"])
@pytest.mark.parametrize("rows,cols,batch,iters", [
    (2, 2, 1, 9), (16, 16, 1, 7), (257, 3, 1, 8), (16, 17, 3, 16), (2, 300, 1, 17), (20, 20, 1, 0),
    (512, 512, 1, 3), (513, 512, 1, 9), (90, 97, 40, 8)])
def test_groups_and_batches_match_oracle(tv, rows, cols, batch, iters):
    import torch
    from imgrecsrc_amd.tv import TV
    rng = np.random.default_rng(rows * cols + iters)
    x = (rng.standard_normal((rows, cols)) + 0.5).astype(np.float32)
    w = TV(rows, cols, tv=tv, batch=batch)
    xt = torch.from_numpy(np.tile(x.ravel(), batch)).cuda()  # equal images stop together
    for _ in range(2):  # a second call meets the first one's fields
        out, itr = w.denoise(xt, 0.2, 1e-12, iters)
        got = out.cpu().numpy().reshape(batch, rows, cols)
        if iters == 0:
            assert itr == 0 and not got.any()
            continue
        ref, itr_ref = T.denoise(x.astype(np.float64), 0.2, tv, 1e-12, iters)
        err = np.abs(got - ref).max() / np.abs(ref).max()
        print(f"{tv} {batch}x{rows}x{cols}: {itr} iterations (oracle {itr_ref}), {err:.2e}")
        assert itr == itr_ref
        assert err <= 1e-6
