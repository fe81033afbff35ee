"""Forward lists of 4x4-pixel sub-blocks: a record outside a sub-block's list
cannot reach its pixels, so the outputs equal those of the walk without
footprint tests, in which every sub-block lists every record, bit for bit."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


# Images of part of a sub-block, of one tile, ragged ones; lists around one
# and two 256-record batches; round, thin and vanishing surfels; opacities
# around the 1/255 below which a record has no footprint.
@pytest.mark.parametrize("size", [(1, 1), (16, 16), (3, 37), (131, 61)])
@pytest.mark.parametrize("n,thin,opacity", [(1, 1.0, 0.9), (255, 1.0, 0.02), (257, 1e-2, 0.5), (513, 1.0, 0.00394),
                                            (20_000, 1e-4, 0.3)])
def test_listed_records_are_all_that_reach_a_pixel(gpu, size, n, thin, opacity):
    import splattar_amd as sa
    from splattar_amd import scenes
    announce(f"sub-blocks: {size[0]}x{size[1]}, n {n}, thin {thin}")
    w, h = size
    rng = np.random.default_rng(n)
    sc = scenes.make_scene(n, 1, -3.5, 1.0, n)
    scales = sc.scales.copy()
    scales[:, n % 2] *= thin ** rng.uniform(0, 1, n).astype(np.float32)
    op = (opacity * rng.uniform(0.9, 1.1, n)).astype(np.float32)
    r = sa.Rasterizer(gpu, n, w, h, 64 * n + 4096)
    r.upload_scene(0.4 * sc.positions, scales, sc.quats, op, sc.sh)
    sp = scenes.front_view(w, h)
    cam = sa.Camera(sp.center, sp.quat, max(sp.focal, 20.0), 1)
    outs = []
    for cull, binning in ((False, 0), (True, 0), (True, 2)):
        r.set_culling(cull)
        r.set_binning(binning)
        r.forward(cam, n)
        outs.append([b.read().copy() for b in (r.out_color, r.out_aux, r.out_normal, r.out_ncontrib)])
    r.close()
    for binning, got in ((0, outs[1]), (2, outs[2])):
        # ncontrib counts along the tile's list, which tight binning shortens.
        for name, a, b in zip(("color", "aux", "normal", "ncontrib")[:4 - binning // 2], outs[0], got):
            assert np.array_equal(a, b), f"binning {binning}: {name}"
