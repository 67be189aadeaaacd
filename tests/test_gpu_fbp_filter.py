"""The ramp filter's tiles: 256 outputs, four views and 1024-tap chunks of a work-group,
each at its edges and one past them, parallel and fan, against the FP64 oracle.  On a 16^2
image the rounding of positions (1e-6 px) and of the filter's sums (a few 1e-7 of the
samples) stay an order below the 1e-5 bar of the golden FBP cases."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [1, 2, 63, 64, 255, 256, 257, 511, 1023, 1024, 1025, 1100, 2049])
@pytest.mark.parametrize("npj,full,d", [(12, 24, 0.0), (13, 13, 3000.0), (3, 40, 0.0)])
def test_filter_tiles_against_fp64(oracle_mod, W, npj, full, d):
    import torch
    from imgrecsrc_amd.phantom import gaussian
    from imgrecsrc_amd.projector import Projector
    from test_gpu_projector import ANGLE_MODE
    geo = (16, W, npj, full, 1.0, 1.0, d)
    other = (8, 5, 6, 12, 1.0, 1.0, 0.0)  # a narrower slice in the same launch
    P = Projector([geo, other])
    cf = oracle_mod.conf(*geo, angle_mode=ANGLE_MODE[P.modes()[0]])
    y = gaussian((npj, W), 41)
    flat = np.concatenate([y.ravel(), gaussian((6, 5), 42).ravel()])
    b = P.unpack_images(P.fbp(torch.from_numpy(flat).cuda()))[0].cpu().numpy()
    b64 = oracle_mod.fbp(cf, y)
    err = np.linalg.norm(b - b64) / max(np.linalg.norm(b64), 1e-30)
    print(f"W={W} np={npj} d={d}: {err:.2e}")
    assert err <= 1e-5
