"""Backward over long tile lists split over depth, with many tiles of two views
in one launch: split tiles beside whole ones, segments of several tiles in one
pool, tiles cut by the image's edges. A surfel that reaches at most two tiles of
a view gets at most two terms in each slot there, whose sum has no order, so the
gradients of the split walk equal those of the whole walk bit for bit."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

SIZES = [(83, 45), (61, 70)]


def _run(gpu, monkeypatch, queue, sc, counts, aux):
    import splattar_amd as sa
    from splattar_amd import scenes
    # Without the tile queue a workgroup walks its tile's list whole.
    monkeypatch.setenv("GS_TILE_QUEUE", "1" if queue else "0")
    rng = np.random.default_rng(5)
    w, h = max(s[0] for s in SIZES), max(s[1] for s in SIZES)
    r = sa.Rasterizer(gpu, sc.n, w, h, 32 * sc.n, 2)
    r.upload_scene(sc.positions, sc.scales, sc.quats, sc.opacities, sc.sh)
    r.set_binning(sa._lib.GS_BINNING_TIGHT)  # entries only where the footprint reaches
    r.set_lambda_dist(0.35 if aux else 0.0)
    r.dl_dcolor.write(rng.normal(size=r.dl_dcolor.shape).astype(np.float32))
    r.dl_dnormal.write(rng.normal(size=r.dl_dnormal.shape).astype(np.float32))
    specs = scenes.sphere_views(2, 11, SIZES)
    r.forward_batch([(sa.Camera(sp.center, sp.quat, sp.focal, 1), sp.width, sp.height, m)
                     for sp, m in zip(specs, counts)])
    dbg = r.debug()
    r.backward_batch(flags=0 if aux else sa._lib.GS_BWD_COLOR_ONLY)
    out = {k: getattr(r, k).read().copy() for k in ("grad_pos", "grad_scales", "grad_quat", "grad_opacity", "grad_sh")}
    r.close()
    return out, dbg


@pytest.mark.parametrize("aux", [False, True])
@pytest.mark.parametrize("counts", [(5000, 5000), (2500, 5000), (5000, 600)])
def test_split_lists_of_many_tiles(gpu, monkeypatch, counts, aux):
    from splattar_amd import scenes
    announce(f"segments of many tiles: counts {counts}, aux {aux}")
    n = max(counts)
    sc = scenes.make_scene(n, 1, -2.9, 0.4, 17)  # about a pixel: both hit branches
    rng = np.random.default_rng(17)
    # Three quarters in a part of the volume: lists of a few records and of
    # hundreds. Low opacities keep the pixels unsaturated.
    near = rng.random(n) < 0.75
    sc.positions[near] = sc.positions[near] * 0.45 + np.float32(0.3)
    sc.opacities[:] = rng.uniform(0.005, 0.02, n).astype(np.float32)
    whole, dbg = _run(gpu, monkeypatch, False, sc, counts, aux)
    split, _ = _run(gpu, monkeypatch, True, sc, counts, aux)
    tile = (dbg["sorted_keys"] >> np.uint64(32)).astype(np.int64)
    lens = np.bincount(tile)
    tiles0 = -(-SIZES[0][0] // 16) * -(-SIZES[0][1] // 16)
    seg = 64 if aux else 32  # the shortest segment: few entries here
    assert (lens[:tiles0] > 2 * seg).sum() >= 3 and (lens[tiles0:] > 2 * seg).sum() >= (3 if counts[1] == n else 0)
    assert ((lens > 0) & (lens <= seg)).sum() >= 3
    reached = np.bincount(dbg["sorted_payloads"], minlength=2 * n).reshape(2, n)
    sure = (reached <= 2).all(0)
    assert sure.mean() > 0.5
    for k in whole:
        a, b = whole[k].reshape(n, -1)[sure], split[k].reshape(n, -1)[sure]
        assert (np.abs(a).max(1) > 0).mean() > 0.3, k
        np.testing.assert_array_equal(b, a, err_msg=k)
