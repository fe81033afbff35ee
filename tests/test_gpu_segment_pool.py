"""The buffers of lists split over depth: allocated by the first backward that
splits, also under capture, and never by an object that only renders; tiles
that find no room in the pool are walked whole."""

import ctypes as C

import numpy as np
import pytest

from conftest import announce
from test_gpu_segment_tiles import SIZES, _run

pytestmark = pytest.mark.gpu


def _hip(name, *args):
    """A HIP call of the runtime that the library is linked to."""
    import splattar_amd as sa
    rc = getattr(sa.lib(), name)(*args)
    assert rc == 0, f"{name}: {rc}"


def _free_mib():
    _hip("hipDeviceSynchronize")
    free, total = C.c_size_t(), C.c_size_t()
    _hip("hipMemGetInfo", C.byref(free), C.byref(total))
    return free.value / 2**20


def _raster(gpu, n, size, seed):
    import splattar_amd as sa
    from splattar_amd import scenes
    rng = np.random.default_rng(seed)
    sc = scenes.make_scene(n, 1, -2.5, 0.5, seed)
    op = rng.uniform(0.005, 0.02, n).astype(np.float32)
    r = sa.Rasterizer(gpu, n, size, size, 64 * n)
    r.upload_scene(0.4 * sc.positions, sc.scales, sc.quats, op, sc.sh)
    r.dl_dcolor.write(rng.normal(size=r.dl_dcolor.shape).astype(np.float32))
    r.dl_dnormal.write(rng.normal(size=r.dl_dnormal.shape).astype(np.float32))
    sp = scenes.front_view(size, size)
    return r, sa.Camera(sp.center, sp.quat, sp.focal, 1)


def test_only_a_backward_allocates_segment_states(gpu):
    import splattar_amd as sa
    n, size = 10_000, 256
    r, cam = _raster(gpu, n, size, 1)  # the process's own first launches
    r.forward(cam, n)
    r.backward(n)
    r.close()
    free0 = _free_mib()
    announce("segment states: create and render")
    r, cam = _raster(gpu, n, size, 1)
    r.forward(cam, n)
    free1 = _free_mib()
    announce("segment states: colour backward")
    r.backward(n, flags=sa._lib.GS_BWD_COLOR_ONLY)
    free2 = _free_mib()
    announce("segment states: backward with depth and normals")
    r.backward(n)
    free3 = _free_mib()
    r.backward(n, flags=sa._lib.GS_BWD_COLOR_ONLY)
    r.backward(n)
    free4 = _free_mib()
    r.close()
    print(f"  MiB: rendering {free0 - free1:.0f}, colour {free1 - free2:.0f}, aux {free2 - free3:.0f}")
    # 256 tiles: 6609 segments of 256 pixels, 16 B a pixel and plane.
    plane = 6609 * 256 * 16 / 2**20
    assert free0 - free1 < 70  # parameters, images, 640k entries; 81 more with three planes
    assert plane <= free1 - free2 < 2 * plane
    assert 2 * plane <= free2 - free3 < 3 * plane
    assert free4 == free3


@pytest.mark.parametrize("mode", [0, 1, 2])  # global, thread-local, relaxed
@pytest.mark.parametrize("aux", [False, True])
def test_first_backward_may_be_captured(gpu, aux, mode):
    import splattar_amd as sa
    n, size = 1500, 16  # one tile: one term a slot, so equal bits
    flags = 0 if aux else sa._lib.GS_BWD_COLOR_ONLY
    grads = ("grad_pos", "grad_scales", "grad_quat", "grad_opacity", "grad_sh")
    r, cam = _raster(gpu, n, size, 2)
    r.forward(cam, n)
    r.backward(n, flags=flags)
    want = {k: getattr(r, k).read().copy() for k in grads}
    r.close()
    r, cam = _raster(gpu, n, size, 2)
    r.forward(cam, n)
    gpu.synchronize()
    announce(f"segment states: capture of the first backward, aux {aux}, mode {mode}")
    s, g, e = C.c_void_p(), C.c_void_p(), C.c_void_p()
    _hip("hipStreamCreateWithFlags", C.byref(s), 1)
    _hip("hipStreamBeginCapture", s, mode)
    try:
        r.backward(n, stream=s, flags=flags)
    finally:
        _hip("hipStreamEndCapture", s, C.byref(g))
    _hip("hipGraphInstantiate", C.byref(e), g, None, None, C.c_size_t(0))
    for replay in range(3):
        for k in grads:
            getattr(r, k).clear()
        gpu.synchronize()
        _hip("hipGraphLaunch", e, s)
        _hip("hipStreamSynchronize", s)
        for k in grads:
            np.testing.assert_array_equal(getattr(r, k).read(), want[k], err_msg=f"replay {replay}: {k}")
        # The object's own work between the replays: the other planes as well.
        r.forward(cam, n)
        r.backward(n)
        r.forward(cam, n)
        gpu.synchronize()
    _hip("hipGraphExecDestroy", e)
    _hip("hipGraphDestroy", g)
    _hip("hipStreamDestroy", s)
    r.close()


@pytest.mark.parametrize("aux", [False, True])
@pytest.mark.parametrize("pool", [1, 7, 40])
def test_tiles_without_room_are_walked_whole(gpu, monkeypatch, pool, aux):
    from splattar_amd import scenes
    n = 5000
    sc = scenes.make_scene(n, 1, -2.9, 0.4, 17)
    sc.positions[: 3 * n // 4] = sc.positions[: 3 * n // 4] * 0.45 + np.float32(0.3)
    sc.opacities[:] = np.random.default_rng(17).uniform(0.005, 0.02, n).astype(np.float32)
    announce(f"segment pool of {pool}, {len(SIZES)} views, aux {aux}")
    whole, dbg = _run(gpu, monkeypatch, False, sc, (n, n), aux)
    monkeypatch.setenv("GS_SEGMENT_POOL", str(pool))
    split, _ = _run(gpu, monkeypatch, True, sc, (n, n), aux)
    lens = np.bincount((dbg["sorted_keys"] >> np.uint64(32)).astype(np.int64))
    assert (lens // (64 if aux else 32)).sum() > 2 * pool  # more segments than the pool holds
    sure = (np.bincount(dbg["sorted_payloads"], minlength=2 * n).reshape(2, n) <= 2).all(0)
    for k in whole:
        np.testing.assert_array_equal(split[k].reshape(n, -1)[sure], whole[k].reshape(n, -1)[sure], err_msg=k)
