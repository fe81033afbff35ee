"""Backward over long tile lists split over depth: a one-tile image gives each
record one contribution, so the gradients of the split walk must equal those
of the whole walk bit for bit (a segment continues from the stored walk state,
and the sums over the tile's pixels are the same)."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


def _gradients(gpu, monkeypatch, queue, n, opaque, aux, seed):
    import splattar_amd as sa
    from splattar_amd import scenes
    # Without the tile queue a workgroup walks its tile's list whole.
    monkeypatch.setenv("GS_TILE_QUEUE", "1" if queue else "0")
    rng = np.random.default_rng(seed)
    size = 16
    sc = scenes.make_scene(n, 1, -2.5, 0.5, seed)
    # Low opacities keep the pixels unsaturated; those below 1/255 occupy the
    # list without contributing.
    op = np.where(rng.random(n) < opaque, rng.uniform(0.005, 0.02, n), 0.001).astype(np.float32)
    r = sa.Rasterizer(gpu, n, size, size, max(4 * n, 64))
    r.upload_scene(0.4 * sc.positions, sc.scales, sc.quats, op, sc.sh)
    sp = scenes.front_view(size, size)
    r.set_lambda_dist(0.35 if aux else 0.0)
    r.dl_dcolor.write(rng.normal(size=(size, size, 4)).astype(np.float32))
    r.dl_dnormal.write(rng.normal(size=(size, size, 4)).astype(np.float32))
    r.forward(sa.Camera(sp.center, sp.quat, sp.focal, 1), n)
    r.backward(n, flags=0 if aux else sa._lib.GS_BWD_COLOR_ONLY)
    out = [b.read().copy() for b in (r.grad_pos, r.grad_scales, r.grad_quat, r.grad_opacity, r.grad_sh, r.grad_cam)]
    last = int(r.out_ncontrib.read().max())
    r.close()
    return out, last


# Lists around one, two and three segments of the smallest length (32), a list
# of many, and enough entries (over 6144 x 32) for longer segments.
@pytest.mark.parametrize("aux", [False, True])
@pytest.mark.parametrize("n,opaque", [(31, 1.0), (32, 1.0), (33, 1.0), (64, 1.0), (65, 1.0), (97, 1.0), (1500, 1.0),
                                      (250_000, 0.01)])
def test_split_lists_give_the_whole_walks_gradients(gpu, monkeypatch, n, opaque, aux):
    announce(f"segments: n {n}, aux {aux}")
    whole, last = _gradients(gpu, monkeypatch, False, n, opaque, aux, n)
    split, _ = _gradients(gpu, monkeypatch, True, n, opaque, aux, n)
    print(f"  last contributor at {last}")
    if n in (1500, 250_000):
        assert last > 640  # well past one segment
    for name, a, b in zip(("pos", "scales", "quat", "opacity", "sh", "cam"), whole, split):
        assert np.abs(a).max() > 0, name
        assert np.array_equal(a, b), f"{name}: {np.abs(a - b).max()}"
