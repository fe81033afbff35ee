"""The work a user of this framework has it do, as cases that can be timed.

Training steps through `Trainer` (one captured graph per step, or plain
per-view steps), renders and gradients through `Rasterizer`, camera tracking
through `Tracker`, and the loss and binning operations on their own, over the
sizes of the benchmark configurations (10k surfels at 256 x 256 up to 1.25M
surfels over sixteen 720p frames) and odd sizes between them.

Scenes follow the benchmark's distributions: centres U[-1, 1]^3, log-normal
scales, uniform rotations, opacity sigmoid(N(0, 1)), colours U[0, 1], higher
SH bands N(0, 0.2); cameras look at the origin from a sphere of radius 3 with
a 60-degree field of view. Everything random comes from the seed.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import splattar_amd as sa
from splattar_amd._lib import GS_BWD_COLOR_ONLY, GS_BWD_NO_CAMERA

SH_C0 = 0.28209479177387814


# ------------------------------------------------------------------- cases

def _train(name, n, degree, views, width, height, mode="graph", sigma=0.5, mu=-5.0, uneven=False, growth=0.0):
    return {"name": name, "kind": "train", "n": n, "degree": degree, "views": views, "width": width,
            "height": height, "mode": mode, "mu": mu, "sigma": sigma, "uneven": uneven, "growth": growth}


def listed():
    return [
        # A preview-size fit (the 10k-surfel SH0 256 x 256 configuration): the
        # step is a chain of small kernels.
        _train("train_10k_256px", 10_000, 0, 1, 256, 256, mu=-4.0),
        # One full-HD view per step of a mid-size scene, the reference's own
        # per-iteration shape.
        _train("train_100k_1080p", 100_000, 3, 1, 1920, 1080),
        # A photo collection: eight views of uneven resolution per step.
        _train("train_100k_8_uneven", 100_000, 3, 8, 1920, 1080, uneven=True),
        # The headline workload: 1M heavy-tailed surfels, four 1080p views.
        _train("train_1m_4x1080p", 1_000_000, 3, 4, 1920, 1080, sigma=1.0),
        # A video: sixteen 720p frames over a growing scene in one step.
        _train("train_1250k_16x720p", 1_250_000, 3, 16, 1280, 720, growth=0.1),
        # Per-view steps without a graph (the reference's semantics) at an
        # odd image size.
        _train("plain_250k_2x1283x717", 250_000, 2, 2, 1283, 717, mode="plain"),
        # A viewer drawing a trained scene: forward only, every output.
        {"name": "render_300k_720p", "kind": "render", "n": 300_000, "degree": 3, "width": 1280, "height": 720,
         "mu": -5.0, "sigma": 0.7},
        # The renderer inside another program's loss: colour, depth and normal
        # gradients and the camera's, at a small odd size.
        {"name": "grads_20k_321x243", "kind": "grads", "n": 20_000, "degree": 3, "width": 321, "height": 243,
         "mu": -4.0, "sigma": 0.5},
        # Several views of one scene rendered and differentiated together
        # (colour losses of the caller's own).
        {"name": "batch_200k_6x640x360", "kind": "batch", "n": 200_000, "degree": 1, "views": 6, "width": 640,
         "height": 360, "mu": -5.0, "sigma": 0.5},
        # A SLAM front end aligning one frame to its map: twenty dependent
        # render / differentiate / pose-update iterations on a small room.
        {"name": "track_room_320px", "kind": "track", "per_side": 24, "width": 320, "height": 320,
         "iterations": 20},
        # The photometric loss alone, for a caller with its own renderer.
        {"name": "loss_1080p", "kind": "loss", "width": 1920, "height": 1080},
        # The tile binner alone: 64-bit keys, sorted, with tile ranges.
        {"name": "bin_200k_1080p", "kind": "bin", "n": 200_000, "width": 1920, "height": 1080, "spread": 3},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    # Training is most of the use.
    kind = rng.choice(["train", "train", "train", "train", "plain", "render", "grads", "batch", "track", "loss",
                       "bin"])
    width = _log_int(rng, 128, 1920)
    height = max(96, int(width * rng.uniform(0.5, 1.0)))
    degree = rng.choice([0, 1, 2, 3, 3])
    sigma = rng.choice([0.5, 0.5, 0.7, 1.0])
    if kind == "train":
        n = _log_int(rng, 5_000, 1_000_000)
        views = rng.choice([1, 1, 2, 4, 8, 16])
        while views > 1 and (n * views > 8_000_000 or width * height * views > 9_000_000):
            views //= 2
        c = _train("", n, degree, views, width, height, sigma=sigma, uneven=views > 1 and rng.random() < 0.3,
                   growth=0.1 if views > 1 and rng.random() < 0.3 else 0.0)
    elif kind == "plain":
        c = _train("", _log_int(rng, 5_000, 500_000), degree, rng.choice([1, 2]), width, height, mode="plain",
                   sigma=sigma)
    elif kind == "render":
        c = {"kind": kind, "n": _log_int(rng, 5_000, 1_000_000), "degree": degree, "width": width, "height": height,
             "mu": -5.0, "sigma": sigma}
    elif kind == "grads":
        c = {"kind": kind, "n": _log_int(rng, 2_000, 200_000), "degree": degree, "width": min(width, 1280),
             "height": min(height, 720), "mu": -4.5, "sigma": 0.5}
    elif kind == "batch":
        c = {"kind": kind, "n": _log_int(rng, 5_000, 400_000), "degree": degree, "views": rng.randint(2, 8),
             "width": min(width, 1280), "height": min(height, 720), "mu": -5.0, "sigma": sigma}
    elif kind == "track":
        c = {"kind": kind, "per_side": rng.randint(16, 96), "width": min(width, 640), "height": min(height, 480),
             "iterations": rng.randint(8, 24)}
    elif kind == "loss":
        c = {"kind": kind, "width": _log_int(rng, 128, 3840), "height": _log_int(rng, 128, 2160)}
    else:
        c = {"kind": kind, "n": _log_int(rng, 5_000, 500_000), "width": width, "height": height,
             "spread": rng.randint(0, 5)}
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ inputs

_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = sa.GpuContext(0)
    return _ctx


class _Buffer:
    """A framework buffer that torch can view in place; keeps its owner."""

    def __init__(self, owner, buf, shape):
        kind = {4: "<f4" if buf.dtype.kind == "f" else "<i4", 8: "<i8"}[buf.dtype.itemsize]
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (buf.ptr, False),
                                         "version": 2, "strides": None}


class _Handles:
    """Framework handles, closed when neither the state nor an output that
    views their buffers is left."""

    def __init__(self):
        self.list = []

    def __del__(self):
        if self.list:
            torch.cuda.synchronize()
        for h in reversed(self.list):
            h.close()


class _State:
    """What a program keeps between calls."""

    def __init__(self, case):
        self.case = case
        self.kind = case["kind"]
        self.handles = _Handles()
        self.out = None

    def own(self, handle):
        self.handles.list.append(handle)
        return handle

    def view(self, buf, shape=None):
        return torch.as_tensor(_Buffer(self.handles, buf, buf.shape if shape is None else shape), device="cuda")


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _scene(n, degree, mu, sigma, g):
    """Activated scene arrays on the host (what a program loads or keeps)."""
    dev = "cuda"
    pos = torch.rand(n, 3, generator=g, device=dev) * 2 - 1
    scales = torch.exp(torch.randn(n, 2, generator=g, device=dev) * sigma + mu)
    quats = torch.nn.functional.normalize(torch.randn(n, 4, generator=g, device=dev), dim=1)
    opac = torch.sigmoid(torch.randn(n, generator=g, device=dev))
    sh = torch.randn(n, (degree + 1) ** 2, 3, generator=g, device=dev) * 0.2
    sh[:, 0] = (torch.rand(n, 3, generator=g, device=dev) - 0.5) / SH_C0
    host = lambda t: t.float().cpu().numpy()  # noqa: E731
    return {"positions": host(pos), "scales": host(scales), "quats": host(quats), "opacities": host(opac),
            "sh": host(sh.reshape(n, -1))}


def _look_at_origin(eye):
    """Camera-to-world quaternion (xyzw), right-handed, y up, looking down -z."""
    eye = np.asarray(eye, float)
    f = -eye / np.linalg.norm(eye)
    r = np.cross(f, [0.0, 1.0, 0.0])
    r /= np.linalg.norm(r)
    m = np.stack([r, np.cross(r, f), -f], axis=1)
    # Eigenvector form (stable for every rotation).
    k = np.array([[m[0, 0] - m[1, 1] - m[2, 2], m[1, 0] + m[0, 1], m[2, 0] + m[0, 2], m[2, 1] - m[1, 2]],
                  [m[1, 0] + m[0, 1], m[1, 1] - m[0, 0] - m[2, 2], m[2, 1] + m[1, 2], m[0, 2] - m[2, 0]],
                  [m[2, 0] + m[0, 2], m[2, 1] + m[1, 2], m[2, 2] - m[0, 0] - m[1, 1], m[1, 0] - m[0, 1]],
                  [m[2, 1] - m[1, 2], m[0, 2] - m[2, 0], m[1, 0] - m[0, 1], m[0, 0] + m[1, 1] + m[2, 2]]])
    return np.linalg.eigh(k)[1][:, 3]


def _focal(height):
    return float(np.float32(0.5 * height / math.tan(math.radians(30.0))))


def _cameras(case, count, rng):
    """(Camera, width, height) of each view: poses on the sphere, or a slow
    walk (1 cm a frame) for the frames of a growing scene."""
    yaw, pitch = rng.uniform(0, 2 * math.pi), rng.uniform(-0.5, 0.5)
    out = []
    for k in range(count):
        w, h = case["width"], case["height"]
        if case.get("uneven"):
            h = int(rng.integers(max(96, h // 3), h + 1))
            w = max(96, int(round(h * case["width"] / case["height"])))
        if case.get("growth"):
            yaw, pitch = yaw + 0.01 / 3.0, pitch + 0.002
        else:
            yaw, pitch = rng.uniform(0, 2 * math.pi), rng.uniform(-math.pi / 3, math.pi / 3)
        eye = 3.0 * np.array([math.cos(pitch) * math.sin(yaw), math.sin(pitch), math.cos(pitch) * math.cos(yaw)])
        cam = sa.Camera(eye.astype(np.float32), _look_at_origin(eye).astype(np.float32), _focal(h),
                        case.get("degree", 0))
        out.append((cam, w, h))
    return out


def _counts(case):
    """Surfels that each view sees (a growing scene's frames see a prefix)."""
    n, v = case["n"], case.get("views", 1)
    if not case.get("growth"):
        return [n] * v
    base = n / (1.0 + case["growth"] * (v - 1))
    return [min(n, int(base * (1.0 + case["growth"] * k))) for k in range(v - 1)] + [n]


def _raster(state, case, views=1):
    n = case["n"]
    cap = min(max(64 * n, 1 << 16), (1 << 30) // (2 * views))
    return state.own(sa.Rasterizer(_context(), n, case["width"], case["height"], cap, views))


def _upload(r, sc):
    r.upload_scene(sc["positions"], sc["scales"], sc["quats"], sc["opacities"], sc["sh"])


def _prepare_train(state, case, g, rng):
    sc = _scene(case["n"], case["degree"], case["mu"], case["sigma"], g)
    views = _cameras(case, case["views"], rng)
    counts = _counts(case)
    jitter = torch.randn(case["n"], 3, generator=g, device="cuda").mul_(0.01).cpu().numpy()
    targets, entries = [], 0
    rasters = {}
    for (cam, w, h), m in zip(views, counts):
        if (w, h) not in rasters:
            for r in rasters.values():
                r.close()
            rasters = {(w, h): sa.Rasterizer(_context(), case["n"], w, h, min(64 * case["n"], 1 << 28))}
            rasters[(w, h)].upload_scene(sc["positions"] + jitter, sc["scales"], sc["quats"], sc["opacities"],
                                         sc["sh"])
        r = rasters[(w, h)]
        r.forward(cam, m)
        entries = max(entries, r.entry_count())
        targets.append(r.out_color.read().reshape(h, w, 4))
    for r in rasters.values():
        r.close()
    # The rates of a run's end: the scene stays where it is while it is timed.
    cfg = sa.TrainConfig(lam=0.2, dssim_scale=1.0, lr_pos=1.6e-6, lr_scales=5e-5, lr_quat=1e-5, lr_opacity=2.5e-4,
                         lr_sh=2.5e-5, max_views_per_step=case["views"], entries_per_view=(int(entries * 1.3) // 1024 + 1) * 1024)
    tr = state.own(sa.Trainer(_context(), cfg, sc, [(v[0], t, m) for v, t, m in zip(views, targets, counts)]))
    state.trainer = tr
    state.ids = list(range(case["views"]))
    state.mode = {"graph": tr.GRAPH, "batched": tr.BATCHED, "plain": tr.PLAIN}[case["mode"]]
    state.out = {"positions": state.view(tr.positions), "scales": state.view(tr.scales),
                 "quats": state.view(tr.quats), "opacities": state.view(tr.opacities), "sh": state.view(tr.sh)}
    if case["mode"] == "plain":  # plain steps leave the summed gradients behind
        state.out |= {"grad_pos": state.view(tr.grad_pos), "grad_scales": state.view(tr.grad_scales),
                      "grad_quat": state.view(tr.grad_quat), "grad_opacity": state.view(tr.grad_opacity),
                      "grad_sh": state.view(tr.grad_sh)}


def _prepare_raster(state, case, g, rng):
    sc = _scene(case["n"], case["degree"], case["mu"], case["sigma"], g)
    views = _cameras(case, case.get("views", 1), rng)
    state.raster = r = _raster(state, case, len(views))
    _upload(r, sc)
    state.views = views
    images = {"color": state.view(r.out_color), "ncontrib": state.view(r.out_ncontrib)}
    if case["kind"] != "batch":
        images |= {"aux": state.view(r.out_aux), "normal": state.view(r.out_normal)}
    state.out = images
    if case["kind"] == "render":
        return
    # dL/d(image) as a caller's own loss leaves it: rgb, depth in .w, normals.
    P = len(views) * case["width"] * case["height"]
    dl = torch.randn(P, 4, generator=g, device="cuda") / (3 * P)
    dn = torch.randn(P, 4, generator=g, device="cuda") / (3 * P)
    if case["kind"] == "batch":
        dl[:, 3] = 0
    dn[:, 3] = 0
    state.view(r.dl_dcolor, (P, 4)).copy_(dl)
    state.view(r.dl_dnormal, (P, 4)).copy_(dn)
    state.out = images | {"grad_pos": state.view(r.grad_pos), "grad_scales": state.view(r.grad_scales),
                          "grad_quat": state.view(r.grad_quat), "grad_opacity": state.view(r.grad_opacity),
                          "grad_sh": state.view(r.grad_sh)}
    if case["kind"] == "grads":
        state.out["grad_cam"] = state.view(r.grad_cam)


def _room(per_side, g, size=3.0):
    """Six inward-facing walls of per_side x per_side round opaque surfels."""
    step = 2.0 * size / (per_side - 1)
    a = np.linspace(-size, size, per_side)
    u, v = (x.ravel() for x in np.meshgrid(a, a, indexing="ij"))
    pos, quats = [], []
    h = math.sqrt(0.5)
    for axis in range(3):
        for sign in (1.0, -1.0):
            p = np.empty((u.size, 3))
            p[:, axis] = sign * size
            p[:, (axis + 1) % 3], p[:, (axis + 2) % 3] = u, v
            pos.append(p)
            # Rotations taking +z onto the wall's axis (disks: the sign is free).
            q = {0: [0, h, 0, h], 1: [h, 0, 0, h], 2: [0, 0, 0, 1]}[axis]
            quats.append(np.tile(q, (u.size, 1)))
    n = 6 * u.size
    rgb = 0.25 + 0.6 * torch.rand(n, 3, generator=g, device="cuda").cpu().numpy()
    return {"positions": np.concatenate(pos).astype(np.float32),
            "scales": np.full((n, 2), 0.75 * step, np.float32),
            "quats": np.concatenate(quats).astype(np.float32), "opacities": np.full(n, 0.95, np.float32),
            "sh": ((rgb - 0.5) / SH_C0).astype(np.float32)}


def _prepare_track(state, case, g, rng):
    sc = _room(case["per_side"], g)
    n = sc["positions"].shape[0]
    w, h = case["width"], case["height"]
    r = state.own(sa.Rasterizer(_context(), n, w, h, n * 64))
    _upload(r, sc)
    tr = state.own(sa.Tracker(_context(), r, w, h))
    truth_c = rng.uniform(-0.4, 0.4, 3)
    ang = rng.uniform(-0.6, 0.6)
    quat = lambda a: np.array([0.0, math.sin(a / 2), 0.0, math.cos(a / 2)], np.float32)  # noqa: E731
    r.forward(sa.Camera(truth_c.astype(np.float32), quat(ang), _focal(h), 0), n)
    tr.set_target(r.out_color.read())
    state.tracker, state.n = tr, n
    # Where the last frame left the camera: a few centimetres and a degree off.
    state.start = (truth_c + rng.uniform(-0.06, 0.06, 3)).astype(np.float32), quat(ang + 0.02), _focal(h)
    state.cfg = sa.TrackConfig(iterations=case["iterations"], patience=case["iterations"] + 1)


def _loss_inputs(case, seed):
    g = _generator(seed)
    w, h = case["width"], case["height"]
    # A smooth image and a render of it: noise on top.
    low = torch.rand(1, 4, max(2, h // 16), max(2, w // 16), generator=g, device="cuda")
    tgt = torch.nn.functional.interpolate(low, size=(h, w), mode="bilinear", align_corners=False)[0]
    tgt = tgt.permute(1, 2, 0).contiguous()
    img = (tgt + 0.05 * torch.randn(h, w, 4, generator=g, device="cuda")).contiguous()
    return img, tgt


def _prepare_loss(state, case, seed):
    w, h = case["width"], case["height"]
    ctx = _context()
    img, dl = (ctx.alloc(np.float32, (h, w, 4)) for _ in range(2))
    loss = sa.SsimLoss(ctx, w, h, 0.2, img, dl)

    class _Free:  # buffers of the caller's own, released after the loss
        def close(self):
            img.free()
            dl.free()

    state.own(_Free())
    state.loss = state.own(loss)
    a, b = _loss_inputs(case, seed)
    state.view(img).copy_(a)
    state.view(loss.target).copy_(b)
    state.out = {"dl": state.view(dl)}


def _prepare_bin(state, case, g):
    n, w, h = case["n"], case["width"], case["height"]
    tx, ty = -(-w // 16), -(-h // 16)
    # Every rect size equally often and a tenth of the items culled, so the
    # number of entries does not depend on the seed.
    k = torch.randperm(n, generator=g, device="cuda")
    m = case["spread"] + 1
    culled = k % 10 == 0
    ex, ey = (k // 10) % m, (k // (10 * m)) % m
    u = torch.rand(2, n, generator=g, device="cuda")
    cx, cy = (u[0] * (tx - ex)).long(), (u[1] * (ty - ey)).long()
    rects = torch.stack([cx, cy, cx + ex, cy + ey], 1).int()
    rects[culled] = torch.tensor([1, 1, 0, 0], device="cuda").int()
    depths = (2.0 + 2.0 * torch.rand(n, generator=g, device="cuda")).view(torch.int32)
    entries = int(((ex + 1) * (ey + 1))[~culled].sum())
    b = state.own(sa.TileBinner(_context(), n, entries + 1024, tx * ty))
    state.view(b.rects).copy_(rects)
    state.view(b.depths).copy_(depths)
    state.binner, state.n, state.tiles_x = b, n, tx
    keys, pays = b.sorted_keys(), b.sorted_entries()
    state.out = {"keys": state.view(keys, (entries,)), "items": state.view(pays, (entries,)),
                 "ranges": state.view(b.ranges), "count": state.view(b.entry_count())}


def prepare(case, seed):
    state = _State(case)
    g, rng = _generator(seed), np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "train":
        _prepare_train(state, case, g, rng)
    elif kind in ("render", "grads", "batch"):
        _prepare_raster(state, case, g, rng)
    elif kind == "track":
        _prepare_track(state, case, g, rng)
    elif kind == "loss":
        _prepare_loss(state, case, seed)
    elif kind == "bin":
        _prepare_bin(state, case, g)
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()
    return state


# -------------------------------------------------------------------- pass

def run(state):
    kind = state.kind
    if kind == "train":
        state.trainer.step(state.ids, mode=state.mode)
    elif kind == "render":
        state.raster.forward(state.views[0][0], state.case["n"])
    elif kind == "grads":
        state.raster.forward(state.views[0][0], state.case["n"])
        state.raster.backward(state.case["n"])
    elif kind == "batch":
        n = state.case["n"]
        state.raster.forward_batch([(cam, w, h, n) for cam, w, h in state.views])
        state.raster.backward_batch(flags=GS_BWD_COLOR_ONLY | GS_BWD_NO_CAMERA)
    elif kind == "track":
        center, quat, focal = state.start
        cam = sa.Camera(center, quat, focal, 0)
        rep = state.tracker.track(state.n, cam, 3.0, state.cfg)
        return {"residuals": np.array(rep.residuals, np.float32), "center": cam.center, "quat": cam.quat,
                "coverage": float(rep.coverage)}
    elif kind == "loss":
        state.loss.encode()
    else:
        state.binner.encode(state.n, state.tiles_x)
    return state.out


# -------------------------------------------------------------------- work

def work(case):
    """Compulsory traffic (each input read once, each output written once)
    and arithmetic of a pass. Per-pixel arithmetic counts about 20
    contributing surfels (the benchmark scenes' mean): 30 operations to
    evaluate and composite one, 80 more to differentiate it."""
    kind = case["kind"]
    P = case["width"] * case["height"] * case.get("views", 1)
    if case.get("uneven"):
        P *= 0.45
    S = 4 * (3 + 2 + 4 + 1 + 3 * (case.get("degree", 0) + 1) ** 2)
    if kind == "train":
        n, nv = case["n"], sum(_counts(case))
        # Parameters and two moments read and written, the activated copies
        # written; targets read.
        return {"bytes": 7 * S * n + 12 * P, "flops": P * (20 * 110 + 400) + nv * 600 + n * 900}
    if kind == "render":
        return {"bytes": S * case["n"] + 44 * P, "flops": P * 20 * 30 + case["n"] * 300}
    if kind in ("grads", "batch"):
        nv = case["n"] * case.get("views", 1)
        return {"bytes": 2 * S * case["n"] + (44 + 28) * P, "flops": P * 20 * 110 + nv * 600}
    if kind == "track":
        n = 6 * case["per_side"] ** 2
        # The map and the frame once per iteration, with the image between.
        return {"bytes": case["iterations"] * (S * n + 28 * P), "flops": case["iterations"] * (P * 8 * 110 + n * 600)}
    if kind == "loss":
        return {"bytes": 40 * P, "flops": 3 * P * 420}
    e = 0.9 * case["n"] * (1 + case["spread"] / 2.0) ** 2  # entries
    return {"bytes": 20 * case["n"] + 12 * e, "flops": 0}


# ------------------------------------------------------------ 64-bit values

def _exact_loss(case, seed):
    img, tgt = _loss_inputs(case, seed)
    taps = [0.26601818, 0.21300237, 0.10936069, 0.03599398, 0.00759866, 0.00102838]
    k = torch.tensor([np.float32(taps[abs(d)]) for d in range(-5, 6)], dtype=torch.float64, device="cuda")

    def blur(t):
        c = t.shape[0]
        t = torch.nn.functional.conv2d(t[None], k.view(1, 1, 1, 11).expand(c, 1, 1, 11), padding=(0, 5), groups=c)
        return torch.nn.functional.conv2d(t, k.view(1, 1, 11, 1).expand(c, 1, 11, 1), padding=(5, 0), groups=c)[0]

    x = img[..., :3].double().permute(2, 0, 1).contiguous().requires_grad_(True)
    y = tgt[..., :3].double().permute(2, 0, 1).contiguous()
    mx, my = blur(x), blur(y)
    vx, vy, vxy = blur(x * x) - mx * mx, blur(y * y) - my * my, blur(x * y) - mx * my
    ssim = ((2 * mx * my + 1e-4) * (2 * vxy + 9e-4)) / ((mx * mx + my * my + 1e-4) * (vx + vy + 9e-4))
    loss = 0.8 * (x - y).abs().mean() + 0.2 * 0.5 * (1 - ssim).mean()
    loss.backward()
    out = torch.zeros(case["height"], case["width"], 4, dtype=torch.float64, device="cuda")
    out[..., :3] = x.grad.permute(1, 2, 0)
    return {"dl": out}


def _sh_basis(degree, d):
    x, y, z = d.unbind(-1)
    b = [torch.full_like(x, SH_C0)]
    if degree >= 1:
        c1 = 0.48860251190291987
        b += [-c1 * y, c1 * z, -c1 * x]
    if degree >= 2:
        b += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z,
              0.31539156525252005 * (2 * z * z - x * x - y * y), -1.0925484305920792 * x * z,
              0.5462742152960396 * (x * x - y * y)]
    if degree >= 3:
        b += [-0.5900435899266435 * y * (3 * x * x - y * y), 2.890611442640554 * x * y * z,
              -0.4570457994644658 * y * (4 * z * z - x * x - y * y),
              0.3731763325901154 * z * (2 * z * z - 3 * x * x - 3 * y * y),
              -0.4570457994644658 * x * (4 * z * z - x * x - y * y), 1.445305721320277 * z * (x * x - y * y),
              -0.5900435899266435 * x * (x * x - 3 * y * y)]
    return torch.stack(b, -1)


def _rotation(q):
    x, y, z, w = (q / q.norm(dim=-1, keepdim=True)).unbind(-1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], -1).reshape(
                            *q.shape[:-1], 3, 3)


def _exact_raster(case, seed):
    """The forward model over every (surfel, pixel) pair in 64 bits, front to
    back in chunks of surfels; gradients by autograd."""
    n, w, h = case["n"], case["width"], case["height"]
    if n * w * h > 4e9:
        return None
    g, rng = _generator(seed), np.random.default_rng(seed)
    sc = _scene(n, case["degree"], case["mu"], case["sigma"], g)
    (cam, _, _), = _cameras(case, 1, rng)
    grads = case["kind"] == "grads"
    leaf = lambda a: torch.as_tensor(np.asarray(a, np.float64), device="cuda").requires_grad_(grads)  # noqa: E731
    pos, scales, quats, opac = (leaf(sc[k]) for k in ("positions", "scales", "quats", "opacities"))
    sh = leaf(sc["sh"].reshape(n, -1, 3))
    R = _rotation(torch.as_tensor(cam.quat.astype(np.float64), device="cuda")).float().double().requires_grad_(grads)
    C, f = leaf(cam.center), leaf(cam.focal)
    rel = pos - C
    c = rel @ R
    depth = -c[:, 2]
    axes = _rotation(quats)
    tu, tv = (axes[:, :, 0] * scales[:, :1]) @ R, (axes[:, :, 1] * scales[:, 1:]) @ R
    cx, cy = w * 0.5, h * 0.5
    px, py = cx + f * c[:, 0] / depth, cy - f * c[:, 1] / depth
    with torch.no_grad():
        rad = (3 * f * (tu.norm(dim=1) + tv.norm(dim=1)) / depth + 3).clamp(max=64)
        keep = (depth >= 0.05) & (px + rad >= 0) & (px - rad < w) & (py + rad >= 0) & (py - rad < h)
        tiles = lambda v, m: (v / 16).clamp(0, m - 1).floor()  # noqa: E731
        tx, ty = -(-w // 16), -(-h // 16)
        rect = torch.stack([tiles(px - rad, tx), tiles(py - rad, ty), tiles(px + rad, tx), tiles(py + rad, ty)], 1)
        order = torch.argsort(depth.float(), stable=True)
        order = order[keep[order]]
        ys, xs = torch.meshgrid(torch.arange(h, device="cuda"), torch.arange(w, device="cuda"), indexing="ij")
        xs, ys = xs.reshape(-1).double(), ys.reshape(-1).double()
        tile_x, tile_y = (xs / 16).floor(), (ys / 16).floor()
    M = torch.linalg.cross(tu, tv)
    A, B = torch.linalg.cross(tv, c), torch.linalg.cross(c, tu)
    Nt = -(M * c).sum(1)
    direction = rel / rel.norm(dim=1, keepdim=True)
    colour = (0.5 + (_sh_basis(case["degree"], direction)[:, :, None] * sh).sum(1)).clamp(min=0)
    nrm = M / M.norm(dim=1, keepdim=True)
    nrm = torch.where((nrm * c).sum(1, keepdim=True) > 0, -nrm, nrm)
    sx, sy = -(xs + 0.5 - cx) / f, (ys + 0.5 - cy) / f

    def chunk(T, M, A, B, Nt, px, py, depth, opac, colour, nrm, sx, sy, rect):
        dot = lambda v: v[:, :1] * sx + v[:, 1:2] * sy + v[:, 2:]  # noqa: E731
        D = dot(M)
        safe = D.abs() > 1e-12
        inv = torch.where(safe, 1.0 / torch.where(safe, D, torch.ones_like(D)), torch.zeros_like(D))
        u, v, t = dot(A) * inv, dot(B) * inv, Nt[:, None] * inv
        e_ray = torch.where(t > 0.05, -(u * u + v * v) * 0.5, torch.full_like(u, -1e30))
        e_scr = -((xs + 0.5 - px[:, None]) ** 2 + (ys + 0.5 - py[:, None]) ** 2)
        ray = e_ray >= e_scr
        a = (opac[:, None] * torch.exp(torch.where(ray, e_ray, e_scr))).clamp(max=0.995)
        t = torch.where(ray, t, depth[:, None].expand_as(t))
        inside = ((tile_x >= rect[:, :1]) & (tile_x <= rect[:, 2:3]) & (tile_y >= rect[:, 1:2]) &
                  (tile_y <= rect[:, 3:]))
        a = torch.where(inside & (a >= 1.0 / 255.0), a, torch.zeros_like(a))
        after = T * torch.cumprod(1 - a, 0)
        before = torch.cat([T[None], after[:-1]])
        live = before >= 1e-4
        wgt = torch.where(live, before * a, torch.zeros_like(a))
        T = T * torch.where(live, 1 - a, torch.ones_like(a)).prod(0)
        return T, wgt.T @ colour, wgt.sum(0), (wgt * t).sum(0), wgt.T @ nrm

    from torch.utils.checkpoint import checkpoint
    T = torch.ones(w * h, dtype=torch.float64, device="cuda")
    rgb, alpha, dep, normal = 0, 0, 0, 0
    for k in torch.split(order, 64):
        args = (T, M[k], A[k], B[k], Nt[k], px[k], py[k], depth[k], opac[k], colour[k], nrm[k], sx, sy, rect[k])
        T, drgb, dalpha, ddep, dnormal = checkpoint(chunk, *args, use_reentrant=False) if grads else chunk(*args)
        rgb, alpha, dep, normal = rgb + drgb, alpha + dalpha, dep + ddep, normal + dnormal
    zero = torch.zeros_like(T)
    image = lambda *p: torch.stack(p, 1).detach().reshape(h, w, 4)  # noqa: E731
    out = {"color": image(*rgb.unbind(1), alpha), "aux": image(T, dep, zero, zero),
           "normal": image(*normal.unbind(1), zero), "ncontrib": None}
    if not grads:
        return out
    P = w * h
    dl = (torch.randn(P, 4, generator=g, device="cuda") / (3 * P)).double()
    dn = (torch.randn(P, 4, generator=g, device="cuda") / (3 * P)).double()
    ((dl[:, :3] * rgb).sum() + (dl[:, 3] * dep).sum() + (dn[:, :3] * normal).sum()).backward()
    pad = lambda t, m: torch.nn.functional.pad(t.reshape(n, -1), (0, m - t.reshape(n, -1).shape[1]))  # noqa: E731
    out |= {"grad_pos": pad(pos.grad, 4), "grad_scales": scales.grad, "grad_quat": quats.grad,
            "grad_opacity": opac.grad, "grad_sh": pad(sh.grad, 48),
            "grad_cam": torch.cat([R.grad.T.reshape(9), C.grad, f.grad.reshape(1), torch.zeros(3).cuda().double()])}
    return out


def exact(case, seed):
    if case["kind"] == "loss":
        return _exact_loss(case, seed)
    if case["kind"] in ("render", "grads"):
        return _exact_raster(case, seed)
    # A training step's weights carry Adam's normalised updates and a track's
    # pose twenty of them: their arithmetic is the gradients', given above;
    # a binner's outputs are whole numbers.
    return None
