"""Items without entries (behind the camera, beside the image) are left out of
the depth presort; the 64-bit key path keeps every item, so entries and images
of the two must be the same, also where no item or every item is left."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


# One workgroup's sort, the one without a scan, the one with; both digit widths.
@pytest.mark.parametrize("n", [1, 3000, 20_000, 200_000])
@pytest.mark.parametrize("digit", [8, 4])
def test_presort_without_culled_items_equals_sort64(gpu, n, digit):
    import splattar_amd as sa
    from splattar_amd import scenes
    w, h = 150, 90
    sc = scenes.make_scene(n, 0, -3.5, 0.5, n)
    sp = scenes.front_view(w, h)
    r = sa.Rasterizer(gpu, n, w, h, 64 * n)
    r.set_digit_bits(digit)
    forward = np.array([0.0, 0.0, 1.0])  # the camera is at z = -3
    kept = set()
    # Every surfel in front; about half behind the camera; a narrow view past
    # most of them; all behind.
    for shift, zoom in ((0.0, 1.0), (3.0, 1.0), (0.0, 8.0), (50.0, 1.0)):
        r.upload_scene((sc.positions - shift * forward).astype(np.float32), sc.scales, sc.quats, sc.opacities, sc.sh)
        cam = sa.Camera(sp.center, sp.quat, sp.focal * zoom, 0)
        outs = []
        for binning in (0, 1, 2):
            announce(f"dropped items n={n} digit={digit} shift={shift} zoom={zoom} binning={binning}")
            r.set_binning(binning)
            r.forward(cam, n)
            outs.append((r.entry_count(), r.out_color.read().copy(), r.out_aux.read().copy(), r.out_ncontrib.read().copy()))
        assert outs[0][0] == outs[1][0]
        for k in (1, 2, 3):
            assert np.array_equal(outs[0][k], outs[1][k]), k
        for k in (1, 2):
            assert np.array_equal(outs[2][k], outs[1][k]), k
        kept.add(outs[0][0])
    if n > 1:
        assert len(kept) > 2 and 0 in kept  # the cases do differ, and one has no entry
    r.close()
