"""L1 + D-SSIM in bands of few and of many rows (the band height follows from
the image's size): edge rows and columns of bands, strips and images against
the oracle, at the tolerances of the loss op's other sizes (f32 blurs of 121
taps, sums in double)."""

import numpy as np
import pytest

import oracle
from conftest import announce

pytestmark = pytest.mark.gpu


# One pixel; bands of four rows with one, two and three rows left over; a
# strip's 74 columns and one more; many bands of one strip; enough pixels that
# the bands are long and four workgroups share a CU.
@pytest.mark.parametrize("W,H", [(1, 1), (3, 5), (74, 4), (75, 6), (20, 7), (33, 700), (1999, 301)])
def test_bands_match_fp64_oracle(gpu, W, H):
    import splattar_amd as sa
    rng = np.random.default_rng(W * H)
    x = rng.random((H, W, 3)).astype(np.float32)
    y = np.clip(x + rng.normal(0, 0.15, x.shape), 0, 1).astype(np.float32)
    img = gpu.alloc(np.float32, (H, W, 4))
    dl = gpu.alloc(np.float32, (H, W, 4))
    img.write(np.concatenate([x, np.ones((H, W, 1), np.float32)], axis=2))
    loss = sa.SsimLoss(gpu, W, H, 0.2, img, dl, dssim_scale=0.5)
    loss.target.write(np.concatenate([y, np.ones((H, W, 1), np.float32)], axis=2))
    announce(f"l1_ssim bands {W}x{H}")
    loss.encode()
    l1, dssim = loss.read_losses()
    got = dl.read()
    _, ref_dl, ref_l1, ref_ss = oracle.l1_ssim(x.astype(np.float64), y.astype(np.float64), 0.2, 0.5)
    assert abs(l1 - ref_l1) <= 1e-6 * ref_l1
    assert abs(dssim - 0.5 * (1 - ref_ss)) <= 1e-5 * abs(0.5 * (1 - ref_ss))
    assert np.linalg.norm(got[..., :3] - ref_dl) / np.linalg.norm(ref_dl) < 1e-4
    assert np.all(got[..., 3] == 0.0)
    loss.close()
    img.free()
    dl.free()
