"""The work that programs built on this library have it do, as measurable cases.

A case is a dict of plain values; prepare() makes what a program holds before the call (a renderer
with its scene resident, camera and parameters; host records where the data comes from the host),
run() is one pass through the public entry points and returns its outputs, exact() the same outputs
from plain torch in 64 bits where that is affordable, work() the bytes and operations that a pass
cannot do without.

Kinds of passes:
  frame     rebuild the structure over a resident scene and render one frame; the frame stays on the
            device (zero-copy views) or is downloaded as the CPU framebuffer of a MegaMol view
  ingest    a new trajectory frame arrives as interleaved host records: upload, build, render, download
  denoised  rebuild, 1-sample ambient occlusion with features, denoise on the device
  refit     the spheres moved a little: new positions from a device buffer, refit, render
  progress  a still camera: frames of a progressive diffuse-bounce accumulation over a built scene
  series    timesteps x cameras in one batched call, results on the host
  train     one training step of the denoiser: loss and gradients of every parameter
"""
from __future__ import annotations

import math
from pathlib import Path

import numpy as np
import torch

from megamol_amd import _lib as L
from megamol_amd import denoiser as DN
from megamol_amd import scenes
from megamol_amd.renderer import ParticleList, SphereRenderer, look_at, params

WEIGHTS = Path(DN.__file__).resolve().parent / "weights" / "denoiser_fcc.bin"
MODES = {"lambert": L.MODE_LAMBERT, "ao": L.MODE_AO, "bounce": L.MODE_BOUNCE}
CROP_DEPTH = 400.0  # depth scale of the training crops


def listed():
    return [
        # interactive preview of a small data set: launches and latency, nothing else
        dict(name="preview_10k", kind="frame", scene="uniform", n=10_000, width=320, height=240, spp=1, mode="lambert",
             bits=30, accel=0, device=False),
        # playing a trajectory in a viewer: every frame comes from the host and goes back as an image,
        # at a window size that is no multiple of a tile
        dict(name="trajectory_250k", kind="ingest", n=250_007, width=1279, height=719, spp=1, mode="lambert", bits=30),
        # the 1M uniform cube at 1024 x 1024, primary rays and Lambert shading
        dict(name="uniform_1m", kind="frame", scene="uniform", n=1_000_000, width=1024, height=1024, spp=1,
             mode="lambert", bits=30, accel=0, device=True),
        # a still for a document: an odd-sized image with some samples per pixel
        dict(name="still_ao16_3m", kind="frame", scene="fcc", n=3_014_284, width=1000, height=621, spp=16, mode="ao",
             bits=30, accel=0, device=True),
        # 50M spheres at 1080p, ambient occlusion with 64 samples, rebuilt for the frame
        dict(name="plain_fcc50m", kind="frame", scene="fcc", n=49_948_672, width=1920, height=1080, spp=64, mode="ao",
             bits=30, accel=0, device=True),
        # the same scene, 1 sample and the denoiser
        dict(name="denoised_fcc50m", kind="denoised", n=49_948_672, width=1920, height=1080),
        # clustered particles (cosmology) at 4K: 63-bit codes, sub-pixel spheres
        dict(name="clusters_60m_4k", kind="frame", scene="clusters", n=60_000_000, width=3840, height=2160, spp=1,
             mode="ao", bits=63, accel=0, device=True),
        # the compact structure for scenes near the memory limit
        dict(name="treelets_8m", kind="frame", scene="clusters", n=8_000_000, width=1280, height=720, spp=1, mode="ao",
             bits=63, accel=1, device=True),
        # a simulation beside the renderer: positions move on the device, the tree is refitted
        dict(name="refit_4m", kind="refit", n=4_000_000, width=1280, height=720, spp=1, mode="ao", bits=30),
        # progressive refinement of a still view with diffuse bounces
        dict(name="progress_1m", kind="progress", n=1_000_000, width=801, height=600, spp=1, bounces=4, frames=4),
        # a time series rendered from several cameras per timestep in one call
        dict(name="series_8x500k", kind="series", n=500_000, timesteps=8, cameras=2, width=800, height=600, spp=1,
             mode="ao", bits=30, refit_period=4),
        # training the denoiser on 128 x 128 crops
        dict(name="train_16x128", kind="train", batch=16, height=128, width=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _image(rng, hi=2_000_000):
    h = _log(rng, 200, math.sqrt(hi / 1.78))
    return int(h * rng.uniform(1.0, 1.78)), h


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "ingest", "denoised", "refit", "progress", "series", "train"])
    if kind == "train":
        return dict(kind=kind, batch=_log(rng, 1, 16), height=rng.randint(24, 128), width=rng.randint(24, 128))
    if kind == "series":
        w, h = _image(rng, 800_000)
        return dict(kind=kind, n=_log(rng, 20_000, 500_000), timesteps=rng.randint(1, 8), cameras=rng.randint(1, 2),
                    width=w, height=h, spp=rng.choice([1, 1, 2]), mode=rng.choice(["ao", "lambert"]), bits=30,
                    refit_period=rng.randint(1, 4))
    w, h = _image(rng)
    if kind == "progress":
        return dict(kind=kind, n=_log(rng, 10_000, 1_000_000), width=w, height=h, spp=rng.choice([1, 1, 2]),
                    bounces=rng.randint(1, 4), frames=rng.randint(1, 4))
    if kind == "refit":
        return dict(kind=kind, n=_log(rng, 10_000, 4_000_000), width=w, height=h, spp=1,
                    mode=rng.choice(["ao", "lambert"]), bits=30)
    if kind == "ingest":
        return dict(kind=kind, n=_log(rng, 10_000, 1_000_000), width=w, height=h, spp=1, mode="lambert", bits=30)
    if kind == "denoised":
        return dict(kind=kind, n=4 * round((_log(rng, 500_000, 49_948_672) / 4) ** (1 / 3)) ** 3, width=w, height=h)
    scene = rng.choice(["uniform", "fcc", "clusters"])
    accel = 1 if scene == "clusters" and rng.random() < 0.4 else 0
    n = _log(rng, 10_000, 8_000_000 if accel else 40_000_000)
    if scene == "fcc":
        n = 4 * round((n / 4) ** (1 / 3)) ** 3
    spp = rng.choice([1, 1, 1, 2, 4, 12, 16, 64] if n < 4_000_000 and not accel else [1, 1, 4])
    return dict(kind="frame", scene=scene, n=n, width=w, height=h, spp=spp, mode=rng.choice(["ao", "lambert"]),
                bits=63 if scene == "clusters" else 30, accel=accel, device=rng.random() < 0.7)


# ---- scenes, made on the device ------------------------------------------------------------------


def _gen(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed) * 7919 + 17)


def _uniform(n, seed):
    """Spheres uniform in the unit cube; radius as in the 1M scene, scaled with the spacing."""
    g = _gen(seed)
    s = torch.empty(n, 4, device="cuda")
    s[:, :3] = torch.rand(n, 3, generator=g, device="cuda")
    s[:, 3] = 0.2 / n ** (1 / 3) * (0.5 + torch.rand(n, generator=g, device="cuda"))
    c = torch.rand(n, 4, generator=g, device="cuda")
    c[:, 3] = 1.0
    return s, c


def _fcc(n, seed):
    """Jittered FCC lattice coloured through the 256-entry transfer function."""
    cells = round((n / 4) ** (1 / 3))
    n = 4 * cells ** 3
    g = _gen(seed)
    j = torch.arange(cells, device="cuda", dtype=torch.float32)
    basis = torch.tensor([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]], device="cuda")
    grid = torch.stack(torch.meshgrid(j, j, j, indexing="ij"), -1).reshape(-1, 1, 3)
    s = torch.empty(n, 4, device="cuda")
    s[:, :3] = (grid + basis).reshape(-1, 3)
    s[:, :3] += torch.randn(n, 3, generator=g, device="cuda") * 0.05
    s[:, 3] = 0.35 + 0.15 * torch.rand(n, generator=g, device="cuda")
    tf = torch.from_numpy(scenes.transfer_function_256()).cuda()
    c = tf[(torch.rand(n, generator=g, device="cuda") * 255.999).long()]
    return s, c


def _clusters(n, seed):
    """Gaussian clusters with lognormal widths and radii, ordered by cluster."""
    g = _gen(seed)
    k = max(20, n // 50_000)
    box = 1e4 * (n / 5e8) ** (1 / 3)
    centre = torch.rand(k, 3, generator=g, device="cuda") * box
    sig = torch.exp(3.0 + 0.5 * torch.randn(k, generator=g, device="cuda"))
    a = torch.randint(0, k, (n,), generator=g, device="cuda").sort().values
    s = torch.empty(n, 4, device="cuda")
    s[:, :3] = centre[a] + torch.randn(n, 3, generator=g, device="cuda") * sig[a, None]
    s[:, 3] = torch.exp(-0.5 + 0.3 * torch.randn(n, generator=g, device="cuda"))
    c = torch.rand(k, 4, generator=g, device="cuda")[a]
    c[:, 3] = 1.0
    return s, c, box


def _box_series(n, seed):
    """Spheres of radius 0.5 uniform in a box at the density of the 4M series."""
    box = 200.0 * (n / 4e6) ** (1 / 3)
    g = _gen(seed)
    s = torch.empty(n, 4, device="cuda")
    s[:, :3] = torch.rand(n, 3, generator=g, device="cuda") * box
    s[:, 3] = 0.5
    c = torch.rand(n, 4, generator=g, device="cuda")
    c[:, 3] = 1.0
    return s, c, box, g


def _move(s, g):
    out = s.clone()
    out[:, :3] += torch.randn(len(s), 3, generator=g, device="cuda") * 0.05
    return out


def _orbit(box, seed, width, height, dist=1.9):
    rs = np.random.RandomState(int(seed) % (2 ** 31))
    a, e = rs.uniform(0, 2 * np.pi), rs.uniform(-0.3, 0.5)
    c = box / 2
    pos = (c + dist * box * math.cos(a) * math.cos(e), c + dist * box * math.sin(e), c + dist * box * math.sin(a) * math.cos(e))
    return look_at(pos, (c, c, c), (0, 1, 0), 40.0, width / height, 0.01 * box, 4 * dist * box)


def _set(r, s, c):
    """The device-resident scene into the renderer (copied on the device)."""
    torch.cuda.synchronize()
    L.check(r.ctx, r.lib.mmhrt_set_spheres_device(r.ctx, s.data_ptr(), c.data_ptr(), len(s), None))


# ---- frames on the device --------------------------------------------------------------------------


class _View:
    """Device memory of a renderer for torch.as_tensor. The tensor keeps this object, and with it the
    renderer that owns the memory, alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": shape, "typestr": typestr, "version": 3}


def _device_frame(r):
    """Zero-copy views of the last frame, complete when this returns."""
    r.sync()
    d = r.device_framebuffer()
    h, w = d.height, d.width
    view = lambda p, shape, t: torch.as_tensor(_View(r, p, shape, t), device="cuda")  # noqa: E731
    return dict(color=view(d.color, (h, w, 4), "<f4"), depth=view(d.depth, (h, w), "<f4"),
                hit_id=view(d.hit_id, (h, w), "<i4"), rgba8=view(d.rgba8, (h, w, 4), "|u1"))


# ---- prepare / run ---------------------------------------------------------------------------------


def _frame_scene(case, seed):
    w, h = case["width"], case["height"]
    if case["scene"] == "fcc":
        s, c = _fcc(case["n"], seed)
        return s, c, scenes.fcc_camera(round((len(s) / 4) ** (1 / 3)), width=w, height=h), 4.0
    if case["scene"] == "clusters":
        s, c, box = _clusters(case["n"], seed)
        return s, c, scenes.clusters_camera(box, width=w, height=h), 0.01 * box
    s, c = _uniform(case["n"], seed)
    return s, c, scenes.uniform_cube_camera(w, h), 0.1


def prepare(case, seed):
    k = case["kind"]
    st = dict(case=case)
    r = st["r"] = SphereRenderer(0)
    if k == "train":
        st["den"] = DN.Denoiser(r, seed=None)
        st["den"].load(str(WEIGHTS))
        st["feats"], st["target"] = _crops(case, seed)
        return st
    w, h = case["width"], case["height"]
    if k == "series":
        s, c, box, g = _box_series(case["n"], seed)
        steps = [s]
        for _ in range(case["timesteps"] - 1):
            steps.append(_move(steps[-1], g))
        r.set_timesteps(torch.stack(steps).cpu().numpy(), c.cpu().numpy())
        p = params(w, h, case["spp"], MODES[case["mode"]], ao_distance=4.0)
        st["jobs"] = [(t, _orbit(box, 1000 * seed + 10 * t + i, w, h), p) for t in range(case["timesteps"])
                      for i in range(case["cameras"])]
        return st
    if k == "ingest":
        s, c = _uniform(case["n"], seed)
        rec = np.zeros(case["n"], np.dtype([("xyz", "<f4", 3), ("rgba", "u1", 4)]))
        rec["xyz"] = s[:, :3].cpu().numpy()
        rec["rgba"] = (c * 255).to(torch.uint8).cpu().numpy()
        st["list"] = ParticleList(L.VERTDATA_FLOAT_XYZ, rec, L.COLDATA_UINT8_RGBA, rec, 16, 16, case["n"],
                                  global_radius=0.2 / case["n"] ** (1 / 3), col_offset=12)
        st["cam"] = scenes.uniform_cube_camera(w, h)
        st["p"] = params(w, h, case["spp"], MODES[case["mode"]])
        return st
    if k == "refit":
        s, c, box, g = _box_series(case["n"], seed)
        st["moved"], st["col"] = _move(s, g), c
        _set(r, s, c)
        r.build(L.BUILD_REBUILD, case["bits"])
        st["cam"] = _orbit(box, seed, w, h)
        st["p"] = params(w, h, case["spp"], MODES[case["mode"]], ao_distance=4.0)
    elif k == "progress":
        s, c = _uniform(case["n"], seed)
        s[:, 3] *= 2.0
        _set(r, s, c)
        r.build(L.BUILD_REBUILD, 30)
        st["cam"] = scenes.uniform_cube_camera(w, h)
        st["ps"] = [params(w, h, case["spp"], L.MODE_BOUNCE, max_bounces=case["bounces"], frame_idx=i, accumulate=1)
                    for i in range(case["frames"])]
    elif k == "denoised":
        s, c = _fcc(case["n"], seed)
        cells = round((len(s) / 4) ** (1 / 3))
        _set(r, s, c)
        st["cam"] = scenes.fcc_camera(cells, width=w, height=h)
        st["p"] = params(w, h, 1, L.MODE_AO, ao_distance=4.0, flags=L.FLAG_AUX, frame_idx=seed % 1000)
        st["den"] = DN.Denoiser(r, seed=None)
        st["den"].load(str(WEIGHTS))
        st["scale"] = 4.0 * cells
    else:
        s, c, st["cam"], ao = _frame_scene(case, seed)
        _set(r, s, c)
        r.set_option("accel", case["accel"])
        st["p"] = params(w, h, case["spp"], MODES[case["mode"]], ao_distance=ao)
    r.sync()
    return st


def run(st):
    case, r = st["case"], st["r"]
    k = case["kind"]
    if k == "train":
        loss, grads = st["den"].train_step(st["feats"], st["target"], CROP_DEPTH, apply=False, want_grads=True)
        return dict(loss=loss, grads=grads)
    if k == "series":
        out, _ = r.render_batch(st["jobs"], refit_period=case["refit_period"], bits=case["bits"])
        return dict(rgba8=[o[0] for o in out], depth=[o[1] for o in out])
    if k == "ingest":
        r.set_lists([st["list"]])
        r.build(L.BUILD_REBUILD, case["bits"])
        f = r.render(st["cam"], st["p"], outputs=("rgba8", "depth"))
        return dict(rgba8=f.rgba8, depth=f.depth)
    if k == "refit":
        L.check(r.ctx, r.lib.mmhrt_set_spheres_device(r.ctx, st["moved"].data_ptr(), st["col"].data_ptr(),
                                                      len(st["moved"]), None))
        r.build(L.BUILD_REFIT, case["bits"])
        r.render_async(st["cam"], st["p"])
        return _device_frame(r)
    if k == "progress":
        for p in st["ps"]:
            r.render_async(st["cam"], p)
        return _device_frame(r)
    if k == "denoised":
        r.build(L.BUILD_REBUILD, 30)
        r.render_async(st["cam"], st["p"])
        st["den"].denoise_frame(st["scale"])
        return _device_frame(r)
    r.build(L.BUILD_REBUILD, case["bits"])
    if case["device"]:
        r.render_async(st["cam"], st["p"])
        return _device_frame(r)
    f = r.render(st["cam"], st["p"], outputs=("rgba8", "depth", "color", "hit_id"))
    return dict(color=f.color, depth=f.depth, hit_id=f.hit_id, rgba8=f.rgba8)


# ---- what a pass cannot do without -----------------------------------------------------------------

NET_FLOPS = 171e3  # denoiser inference, per pixel


def work(case):
    k = case["kind"]
    if k == "train":
        px = case["batch"] * case["height"] * case["width"]
        return {"bytes": px * 36 + 4 * DN.param_count() * 2, "flops": 3 * NET_FLOPS * px}
    n, px = case["n"], case["width"] * case["height"]
    rays = px * case.get("spp", 1)
    if k == "series":
        f = case["timesteps"] * case["cameras"]
        return {"bytes": 16 * n * case["timesteps"] + 8 * px * f, "flops": 2 * rays * f * 50 * math.log2(n)}
    if k == "progress":
        return {"bytes": case["frames"] * px * 32, "flops": case["frames"] * rays * (1 + case["bounces"]) * 50 * math.log2(n)}
    if k == "ingest":
        return {"bytes": 16 * n + 8 * px, "flops": rays * 50 * math.log2(n)}
    fl = rays * (1 if case.get("mode") == "lambert" else 2) * 50 * math.log2(n)
    if k == "denoised":
        return {"bytes": 16 * n + 48 * px, "flops": fl + NET_FLOPS * px}
    return {"bytes": (32 if k == "refit" else 16) * n + 32 * px, "flops": fl}


# ---- the same outputs in 64 bits ---------------------------------------------------------------------


def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    if case["kind"] == "frame" and case["mode"] == "lambert" and case["spp"] == 1 and \
            case["n"] * case["width"] * case["height"] <= 2_000_000_000:
        return _exact_lambert(case, seed)
    return None


def _jitter(px, frame):
    """The two jitter numbers of sample 0 of each pixel: TEA with 16 rounds, then the LCG's low 24 bits."""
    m = np.uint64(0xFFFFFFFF)
    u = lambda v: np.uint64(v)  # noqa: E731
    a, b, s = px.astype(np.uint64), np.full(px.shape, frame, np.uint64), 0
    for _ in range(16):
        s = (s + 0x9E3779B9) & 0xFFFFFFFF
        a = (a + ((((b << u(4)) + u(0xA341316C)) & m) ^ ((b + u(s)) & m) ^ (((b >> u(5)) + u(0xC8013EA4)) & m))) & m
        b = (b + ((((a << u(4)) + u(0xAD90777D)) & m) ^ ((a + u(s)) & m) ^ (((a >> u(5)) + u(0x7E95761E)) & m))) & m
    out = []
    for _ in range(2):
        a = (a * u(1664525) + u(1013904223)) & m
        out.append((a & u(0xFFFFFF)).astype(np.float64) / 16777216.0)
    return out


def _exact_lambert(case, seed):
    """Every primary ray against every sphere, nearest hit, Lambert shading, pseudo depth."""
    s, c, cam, _ = _frame_scene(case, seed)
    s, c = s.double(), c.double()
    w, h = case["width"], case["height"]
    f8 = lambda v: np.array(v[:], np.float64)  # noqa: E731
    pos, front, up = f8(cam.position), f8(cam.direction), f8(cam.up)
    right = np.cross(front, up)
    th = math.tan(0.5 * cam.fovy) * 100.0
    rw = th * cam.aspect
    px = np.arange(w * h)
    jx, jy = _jitter(px, 0)
    u = -rw + 2 * rw * ((px % w) + jx) / w
    v = -(th - 2 * th * ((px // w) + jy) / h)
    d = 100.0 * front + u[:, None] * right + v[:, None] * up
    d = torch.from_numpy(d / np.linalg.norm(d, axis=1, keepdims=True)).cuda()
    o = torch.from_numpy(pos).cuda()
    oc = s[:, :3] - o
    cc = (oc * oc).sum(1) - s[:, 3] ** 2
    col = torch.zeros(w * h, 4, dtype=torch.float64, device="cuda")
    col[:, 3] = 1.0
    depth = torch.ones(w * h, dtype=torch.float64, device="cuda")
    zn, zf = cam.near_plane, cam.far_plane
    step = max(1, 40_000_000 // len(s))
    for i in range(0, w * h, step):
        di = d[i:i + step]
        b = di @ oc.T
        disc = b * b - cc
        t = torch.where(disc >= 0, b - disc.clamp(min=0).sqrt(), torch.inf)
        t = torch.where(t > 1e-6, t, torch.inf)
        t, k = t.min(1)
        hit = torch.isfinite(t)
        tt = torch.where(hit, t, 1.0)
        n = o + tt[:, None] * di - s[k, :3]
        n = n / n.norm(dim=1, keepdim=True)
        sh = 0.2 + 0.6 * (n * di).sum(1).abs()
        ci = torch.cat([c[k, :3] * sh[:, None], torch.ones_like(sh)[:, None]], 1)
        col[i:i + step] = torch.where(hit[:, None], ci, col[i:i + step])
        depth[i:i + step] = torch.where(hit, 0.5 * (-(2 * zf * zn) / (zf - zn) / tt + (zf + zn) / (zf - zn) + 1.0), 1.0)
    return dict(color=col.reshape(h, w, 4), depth=depth.reshape(h, w), hit_id=None, rgba8=None)


def _crops(case, seed):
    """Feature records and targets like the renderer's: patches of spheres on a background, one noisy
    visibility sample per pixel, the target the same surface under its mean visibility."""
    b, h, w = case["batch"], case["height"], case["width"]
    g = _gen(seed)
    rnd = lambda *s: torch.rand(*s, generator=g, device="cuda")  # noqa: E731
    up = lambda x: x.repeat_interleave(4, 1).repeat_interleave(4, 2)[:, :h, :w]  # noqa: E731
    hb, wb = (h + 3) // 4, (w + 3) // 4
    alb, mean, hit = up(0.1 + 0.9 * rnd(b, hb, wb, 3)), up(rnd(b, hb, wb)), up((rnd(b, hb, wb) > 0.15).float())
    t = up(100.0 + 250.0 * rnd(b, hb, wb)) * hit
    nrm = torch.randn(b, h, w, 3, generator=g, device="cuda")
    nrm = nrm / nrm.norm(dim=-1, keepdim=True) * hit[..., None]
    vis = (rnd(b, h, w) < mean).float() * hit
    f = torch.zeros(b, h, w, 12, device="cuda")
    f[..., 0:3] = alb * (vis * hit)[..., None]
    f[..., 3:6] = alb * hit[..., None]
    f[..., 6:9] = nrm
    f[..., 9] = t
    f[..., 10] = vis
    target = alb * (mean * hit)[..., None]
    return f.half().cpu().numpy(), target.float().cpu().numpy()


def _exact_train(case, seed):
    """Loss and gradients of the U-Net by autograd in 64 bits, each 3x3 convolution as nine products."""
    feats, target = _crops(case, seed)
    p, _ = DN.load_weights(str(WEIGHTS))
    f = torch.from_numpy(feats).cuda().double()
    target = torch.from_numpy(target).cuda().double()
    b, h, w, _ = f.shape
    hp, wp = (h + 7) // 8 * 8, (w + 7) // 8 * 8
    x = torch.zeros(b, hp, wp, 16, dtype=torch.float64, device="cuda")
    hit = (f[..., 9] > 0).double()
    x[:, :h, :w, 0] = f[..., 10]
    x[:, :h, :w, 1:4] = f[..., 3:6]
    x[:, :h, :w, 4:7] = f[..., 6:9]
    x[:, :h, :w, 7] = f[..., 9] / CROP_DEPTH * hit
    x[:, :h, :w, 8:11] = f[..., 0:3]
    x[:, :h, :w, 11] = hit
    par = torch.from_numpy(p).cuda().double().requires_grad_(True)
    layers, o = [], 0
    for _, c1, c2, co, relu in DN.LAYERS:
        m = 9 * (c1 + c2) * co
        layers.append((par[o:o + m].view(9, c1 + c2, co), par[o + m:o + m + co], relu))
        o += m + co

    def conv(i, x, skip=None):
        if skip is not None:
            x = torch.cat([skip, x.repeat_interleave(2, 1).repeat_interleave(2, 2)], -1)
        wt, bias, relu = layers[i]
        n, hh, ww, ci = x.shape
        q = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        y = bias
        for t in range(9):
            y = y + (q[:, t // 3:t // 3 + hh, t % 3:t % 3 + ww].reshape(-1, ci) @ wt[t]).view(n, hh, ww, -1)
        return y.relu() if relu else y

    pool = lambda v: v.view(v.shape[0], v.shape[1] // 2, 2, v.shape[2] // 2, 2, v.shape[3]).mean((2, 4))  # noqa: E731
    a1 = conv(1, conv(0, x))
    a3 = conv(3, conv(2, pool(a1)))
    a5 = conv(5, conv(4, pool(a3)))
    y = conv(7, conv(6, pool(a5)))
    y = conv(9, conv(8, y, a5))
    y = conv(11, conv(10, y, a3))
    y = conv(14, conv(13, conv(12, y, a1)))
    out = f[..., 3:6] * y[:, :h, :w, 0:1] + y[:, :h, :w, 1:4]
    out = torch.where(hit[..., None] > 0, out, torch.zeros((), dtype=torch.float64, device="cuda"))
    loss = ((out - target) ** 2).mean()
    loss.backward()
    return dict(loss=loss.detach(), grads=par.grad)
