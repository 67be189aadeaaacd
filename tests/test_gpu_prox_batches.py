"""The prox loops' host side: solves that stop in the first, a middle and the last batch of
eight iterations while the next batch is already queued, one after the other on one
context, and a stream that is being captured (refused: the host reads the loop state).
FP64 oracle at the bar of the other prox cases (images are FP32, 6e-8 of their largest)."""
import numpy as np
import pytest

from oracle import tv_oracle as T
from oracle import wavelet_oracle as W

pytestmark = pytest.mark.gpu


def _image(seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((64, 64)) + 2.0).astype(np.float32)


def test_tv_stops_between_batches():
    import torch
    from imgrecsrc_amd.tv import TV
    w = TV(64, 64)
    batches = set()
    for k, (eps, most) in enumerate([(0.5, 40), (2e-2, 40), (2e-3, 40), (1e-12, 24), (0.5, 3),
                                     (4e-3, 1000), (0.5, 1000)]):
        x = _image(k)
        out, itr = w.denoise(torch.from_numpy(x).cuda(), 0.5, eps, most)
        got = out.cpu().numpy()
        ref, itr_ref = T.denoise(x.astype(np.float64), 0.5, "iso", eps, most)
        assert itr == itr_ref
        assert np.abs(got - ref).max() <= 1e-6 * np.abs(ref).max()
        batches.add((itr + 7) // 8)
    assert len(batches) >= 3


@pytest.mark.parametrize("taps", [2, 4])
def test_admm_stops_between_batches(taps):
    import torch
    from imgrecsrc_amd.wavelet import Wavelet, daubcqf
    h = daubcqf(taps)[0]
    w = Wavelet(64, 64, h, 3)
    batches = set()
    for k, (u, tol, most) in enumerate([(0.3, 1e-3, 100), (0.02, 1e-3, 100), (0.3, 1e-9, 1000),
                                        (0.3, 1e-12, 15), (5.0, 1e-5, 1000), (0.3, 1e-3, 0)]):
        a = _image(k)
        out, itr = w.admm(torch.from_numpy(a).cuda(), u, relativeTol=tol, maxItr=most)
        ref, itr_ref = W.admm(a.astype(np.float64), u, h, 3, tol, most)
        assert itr == itr_ref
        assert np.abs(out.cpu().numpy() - ref).max() <= 1e-6 * np.abs(ref).max()
        batches.add((itr + 7) // 8)
    assert len(batches) >= 3


def test_refused_under_capture():
    import torch
    from imgrecsrc_amd.tv import TV
    from imgrecsrc_amd.wavelet import Wavelet, daubcqf
    w, v = TV(64, 64), Wavelet(64, 64, daubcqf(2)[0], 3)
    x = torch.from_numpy(_image(0)).cuda()
    for call in (lambda: w.denoise(x, 0.5), lambda: v.admm(x, 0.3)):
        ref = call()[0]
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            y = x + 1.0
            with pytest.raises(RuntimeError):
                call()
        g.replay()
        assert torch.equal(y, x + 1.0) and torch.equal(call()[0], ref)
