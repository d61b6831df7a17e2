"""The work a user of this path tracer has it do, as cases that can be timed.

Five kinds of call, all through the public Python API:

  first_hit   ParallelRenderer.first_hit: ids and distances of the primary hits
              (picking, masks, geometry buffers);
  preview     reset, one sample per pixel at a time, then the 8-bit image: the loop
              of the command line and of an interactive viewer;
  render      reset, `spp` samples per pixel in one call, then the mean radiance (to
              the host, or to a tensor on the renderer's device);
  batch       render_batch: views of uneven size and sample count over several scenes;
  train       differentiable rendering of the L2 image loss with respect to every
              material's albedo and emission, forward and backward: `how` = "torch"
              (torch_render and autograd, each sample's radiance kept by the forward
              pass) or "adjoint" (ParallelRenderer.adjoint, nothing kept).

Scenes: the Cornell box fixture (36 triangles), the displaced-sphere scenes
(10,000 to 1,024,006 triangles), the closed Cornell-like box of displaced spheres
(97,292 triangles, 16 materials) and the textured terrain (here 2.8 million
triangles). A scene is built once per process, as a program keeps it; the camera,
the random numbers, and for `train` the parameters and the target come from the seed.
"""
from __future__ import annotations

import functools
import math
import random

import numpy as np
import torch

import cudart_amd as ca
from cudart_amd import torch_render
from cudart_amd import workloads as W

SCENES = ("cornell", "mixed", "spheres1m", "cornell100k", "terrain")
TERRAIN = "grid=700;instances=600;textures=16;texsize=512"
TRIANGLES = {"cornell": 36, "spheres1m": 1_024_006, "cornell100k": 97_292, "terrain": 2_800_000}


def listed():
    return [
        # Picking in a small window: one call, microseconds of device work.
        {"name": "first_hit_cornell_256", "kind": "first_hit", "scene": "cornell", "tris": 36, "w": 256, "h": 256},
        # Geometry buffers of an odd-sized view of the million-triangle scene.
        {"name": "first_hit_1m_1271x713", "kind": "first_hit", "scene": "spheres1m", "tris": 1_024_006, "w": 1271,
         "h": 713},
        # An interactive viewer whose camera has just moved: one sample per pixel at the
        # command line's default size, default integrator.
        {"name": "preview_cornell_640x480_1", "kind": "preview", "scene": "cornell", "tris": 36, "w": 640, "h": 480,
         "spp": 1, "depth": 6, "wave": False},
        # The command line's defaults (640x480, ten passes of one sample) on an ordinary scene.
        {"name": "preview_100k_640x480_10", "kind": "preview", "scene": "mixed", "tris": 100_000, "w": 640, "h": 480,
         "spp": 10, "depth": 6, "wave": False},
        # The Cornell fixture as it is checked and benchmarked: a small whole image.
        {"name": "wave_cornell_256_16", "kind": "render", "scene": "cornell", "tris": 36, "w": 256, "h": 256, "spp": 16,
         "depth": 5, "wave": True, "device": False},
        # The default integrator in one call, an odd size.
        {"name": "mega_1m_961x541_8", "kind": "render", "scene": "spheres1m", "tris": 1_024_006, "w": 961, "h": 541,
         "spp": 8, "depth": 8, "wave": False, "device": False},
        # A draft frame of the million-triangle scene, image to the host.
        {"name": "wave_1m_1280x720_16", "kind": "render", "scene": "spheres1m", "tris": 1_024_006, "w": 1280, "h": 720,
         "spp": 16, "depth": 8, "wave": True, "device": False},
        # The headline workload: a final frame, kept on the GPU for what comes after it.
        {"name": "wave_1m_1080p_128", "kind": "render", "scene": "spheres1m", "tris": 1_024_006, "w": 1920, "h": 1080,
         "spp": 128, "depth": 8, "wave": True, "device": True},
        # The largest image: textured terrain at 4K, a few samples per pixel.
        {"name": "wave_terrain_4k_6", "kind": "render", "scene": "terrain", "tris": 2_800_000, "w": 3840, "h": 2160,
         "spp": 6, "depth": 8, "wave": True, "device": True},
        # A data set's views: 12 uneven views of three scenes in one call.
        {"name": "batch_12_views", "kind": "batch", "scene": "mixed", "tris": 150_000, "scenes": 3, "views": 12,
         "side": 512, "spp": 64, "depth": 8},
        # One optimisation step at the size the gradients are checked on.
        {"name": "train_512_64", "kind": "train", "scene": "cornell100k", "tris": 97_292, "w": 512, "h": 512, "spp": 64,
         "depth": 6, "how": "torch"},
        # The smallest optimisation step, ragged, through the C ABI's one-call form.
        {"name": "train_adjoint_125x93_8", "kind": "train", "scene": "cornell100k", "tris": 97_292, "w": 125, "h": 93,
         "spp": 8, "depth": 6, "how": "adjoint"},
    ]


def _log(rng: random.Random, lo: float, hi: float) -> int:
    """A whole number in [lo, hi], spread over its logarithm."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choice(["first_hit", "preview", "render", "render", "render", "batch", "train"])
    scene = rng.choice(["cornell", "mixed", "mixed", "spheres1m", "cornell100k", "terrain"])
    if kind == "batch":
        scene = "mixed"
    if kind == "train":
        scene = "cornell100k"
    tris = _log(rng, 10_000, 500_000) if scene == "mixed" else TRIANGLES[scene]
    c = {"kind": kind, "scene": scene, "tris": tris}
    if kind == "batch":
        return c | {"scenes": rng.randint(1, 4), "views": rng.randint(2, 16), "side": _log(rng, 64, 640),
                    "spp": _log(rng, 4, 64), "depth": rng.randint(5, 8)}
    w = _log(rng, 96, 1920)
    h = max(16, min(1080, round(w * rng.uniform(0.5, 1.0))))
    c |= {"w": w, "h": h}
    if kind == "first_hit":
        return c
    most = {"preview": 4e6, "render": 6e7, "train": 1.6e7}[kind]  # paths
    wave = rng.random() < 0.6
    if kind == "render" and not wave:
        most = 1e7
    top = {"preview": 10, "render": 128, "train": 64}[kind]
    c["spp"] = _log(rng, 1, max(1, min(top, most // (w * h))))
    c["depth"] = rng.randint(4, 8)
    if kind == "train":
        return c | {"how": rng.choice(["torch", "adjoint"])}
    c["wave"] = wave
    return c | {"device": rng.random() < 0.5} if kind == "render" else c


# --- what a program has in hand ---------------------------------------------

@functools.lru_cache(maxsize=12)
def _scene(kind: str, tris: int, which: int = 0):
    """(mesh, Scene) of a kind; `which` gives other scenes of the same size."""
    if kind == "cornell":
        mesh = W.cornell().mesh
    elif kind == "mixed":
        mesh = ca.Mesh.generate("mixed", f"tris={tris}", W.SEED + 101 * which)
    elif kind == "spheres1m":
        mesh = W.spheres1m().mesh
    elif kind == "cornell100k":
        mesh = W.cornell100k(seed=W.SEED + which).mesh
    elif kind == "terrain":
        mesh = W.large(params=TERRAIN).mesh
    else:
        raise ValueError(kind)
    return mesh, ca.Scene(mesh)


def _camera(kind: str, rng: np.random.Generator, w: int, h: int):
    up = (0.0, 1.0, 0.0)
    if kind == "cornell":
        eye = np.array([2.2, 0.548, 0.0]) + rng.uniform(-0.05, 0.05, 3)
        return ca.camera_look_at(eye, (0.0, 0.548, 0.0), up, 39.3, w, h)
    if kind == "cornell100k":
        eye = np.array([0.0, 5.0, 18.0]) + rng.uniform(-0.5, 0.5, 3)
        return ca.camera_look_at(eye, (0.0, 5.0, 0.0), up, 40.0, w, h)
    th = rng.uniform(0.0, 2.0 * math.pi)
    if kind == "terrain":
        return ca.camera_look_at((110.0 * math.sin(th), 35.0, 110.0 * math.cos(th)), (0.0, 0.0, 0.0), up, 50.0, w, h)
    eye = (35.0 * math.sin(th), 12.0 + 4.0 * math.cos(3.0 * th), 35.0 * math.cos(th))
    return ca.camera_look_at(eye, (0.0, 8.0, 0.0), up, 45.0, w, h)


def _rng(seed: int) -> np.random.Generator:
    return np.random.Generator(np.random.Philox(key=seed))


def _views(case):
    """(scene, side, samples per pixel, view) of a batch: sides from a quarter of the
    largest up, an eighth to all of the samples. The case alone decides them, so that
    every seed's images have the same sizes."""
    rng = _rng(case["side"] * 1000 + case["views"])
    return [(v % case["scenes"], int(rng.integers(max(16, case["side"] // 4), case["side"] + 1)),
             max(1, int(case["spp"] * rng.choice([0.125, 0.25, 0.5, 1.0]))), v) for v in range(case["views"])]


def prepare(case, seed):
    rng = _rng(seed)
    key = int(rng.integers(1, 1 << 31))  # the renderer's random numbers
    kind, s = case["kind"], dict(case)
    if kind == "batch":
        jobs = []
        for which, side, spp, v in _views(case):
            scene = _scene("mixed", max(10_000, case["tris"] >> which), which)[1]
            jobs.append(ca.BatchJob(scene, _camera("mixed", rng, side, side), spp, v + 1))
        return s | {"jobs": jobs, "config": ca.default_config(max_depth=case["depth"], seed=key)}
    w, h = case["w"], case["h"]
    # Training sets the scene's materials, so its scene is its own.
    mesh, scene = _scene(case["scene"], case["tris"], 1 if kind == "train" else 0)
    cam = _camera(case["scene"], rng, w, h)
    s |= {"mesh": mesh, "camera": cam, "key": key}
    if kind == "train":
        materials = mesh.materials
        kd = np.array([list(m.kd) for m in materials], np.float32)
        em = np.array([m.ka[0] for m in materials], np.float32)
        target_kd = np.clip(kd + rng.uniform(-0.1, 0.1, kd.shape), 0.05, 0.95).astype(np.float32)
        common = dict(camera=cam, max_depth=case["depth"])
        for m in range(len(materials)):
            scene.set_material_params(m, target_kd[m], float(em[m]))
        t = ca.ParallelRenderer(scene, w, h, case["spp"], seed=key ^ 0x7A5C3E1,
                                integrator=ca.INTEGRATOR_WAVEFRONT, **common)
        t.render(case["spp"])
        s["target"] = t.radiance()
        t.close()
        s["kd"], s["em"], s["scene_handle"] = kd, em, scene
        if case["how"] == "torch":
            s["albedo"] = torch.from_numpy(kd).cuda().requires_grad_(True)
            s["emission"] = torch.from_numpy(em).cuda().requires_grad_(True)
            s["target"] = torch.from_numpy(s["target"]).cuda()
            s["renderer"] = ca.ParallelRenderer(scene, w, h, case["spp"], seed=key, keep_samples=1,
                                                integrator=ca.INTEGRATOR_WAVEFRONT, **common)
        else:
            s["renderer"] = ca.ParallelRenderer(scene, w, h, case["spp"], seed=key, **common)
        return s
    cfg = dict(max_depth=case.get("depth", 6), seed=key)
    if case.get("wave"):
        cfg["integrator"] = ca.INTEGRATOR_WAVEFRONT
    s["renderer"] = ca.ParallelRenderer(scene, w, h, case.get("spp", 1), camera=cam, **cfg)
    if case.get("device"):
        s["image"] = torch.zeros(h, w, 3, device="cuda")
    return s


# --- one pass ------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "batch":
        images, _ = ca.render_batch(s["jobs"], s["config"])
        return images
    r = s["renderer"]
    if kind == "first_hit":
        tri, mat, t = r.first_hit(0)
        return {"triangle": tri, "material": mat, "t": t}
    if kind == "preview":
        r.reset()
        for _ in range(s["spp"]):
            r.renderOneSamplePerPixel()
        return r.copyImageBytes()
    if kind == "render":
        r.reset()
        r.render(s["spp"])
        if not s["device"]:
            return r.radiance()
        r.radiance_to(s["image"].data_ptr())
        return s["image"]
    if s["how"] == "torch":
        image = torch_render.render(s["albedo"], s["emission"], r, s["spp"], hess=2.0 / s["target"].numel())
        loss = ((image - s["target"]) ** 2).mean()
        d_albedo, d_emission = torch.autograd.grad(loss, [s["albedo"], s["emission"]])
        return {"image": image.detach(), "albedo": d_albedo, "emission": d_emission}
    scene = s["scene_handle"]
    for m in range(len(s["kd"])):
        scene.set_material_params(m, s["kd"][m], float(s["em"][m]))
    d_albedo, d_emission, loss = r.adjoint(s["target"], s["spp"])
    return {"albedo": d_albedo, "emission": d_emission, "loss": loss}


# --- what a pass cannot do without ----------------------------------------------

def _path_work(tris: int, paths: float, depth: int):
    """Scene bytes, and operations of `paths` paths: about 3.1 rays per path were
    counted at depth 8 on the open scenes, two per vertex in the closed boxes; a ray
    visits about 1.3 log4(triangles) four-wide nodes (4 children: 6 fused
    multiply-adds and 6 minima or maxima each) and tests about five triangles (some
    50 operations each); a vertex takes some 400 (random numbers, shading, light)."""
    closed = tris in (TRIANGLES["cornell"], TRIANGLES["cornell100k"])
    rays = paths * (2.0 * depth - 1.0 if closed else min(3.1, 2.0 * depth - 1.0))
    nodes = 1.3 * max(1.0, math.log(tris, 4.0))
    flops = rays * (nodes * 4 * 18 + 5 * 50) + rays / 2 * 400
    return tris * (48 + 64 + 16), flops


def work(case):
    kind, tris = case["kind"], case["tris"]
    if kind == "batch":
        nbytes = sum(max(10_000, tris >> k) * 128 for k in range(min(case["scenes"], case["views"])))
        flops = 0.0
        for which, side, spp, _ in _views(case):
            nbytes += 12 * side * side
            flops += _path_work(max(10_000, tris >> which), side * side * spp, case["depth"])[1]
        return {"bytes": nbytes, "flops": flops}
    px = case["w"] * case["h"]
    if kind == "first_hit":
        nodes = 1.3 * max(1.0, math.log(tris, 4.0))
        return {"bytes": tris * 64 + 12 * px, "flops": px * (nodes * 4 * 18 + 5 * 50 + 150)}
    scene, flops = _path_work(tris, px * case["spp"], case["depth"])
    if kind == "train":  # each vertex once for the image and once for the gradient
        return {"bytes": scene + 24 * px, "flops": 2 * flops}
    return {"bytes": scene + (4 if kind == "preview" else 12) * px, "flops": flops}


# --- the same in 64 bits ------------------------------------------------------------
# Brute force over all triangles in torch, for what that can do within seconds:
# primary hits, and whole images of the Cornell box (diffuse and emissive materials).

def _philox(c, k0, k1):
    """Philox4x32-10 (Salmon et al., 2011) of four int64 tensors of 32-bit words."""
    mask = 0xFFFFFFFF
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
        halves = []
        for word, mul in ((c[0], 0xD2511F53), (c[2], 0xCD9E8D57)):
            lo, hi = (word & 0xFFFF) * mul, (word >> 16) * mul  # each below 2^48
            total = lo + ((hi & 0xFFFF) << 16)
            halves.append((total & mask, ((hi >> 16) + (total >> 32)) & mask))
        (lo0, hi0), (lo1, hi1) = halves
        c = [hi1 ^ c[1] ^ k0, lo1, hi0 ^ c[3] ^ k1, lo0]
    return [(x >> 8).double() * 2.0 ** -24 for x in c]


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True)


class _Exact:
    def __init__(self, mesh, camera, seed):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        a = mesh.arrays()
        f = lambda x: torch.as_tensor(np.asarray(x, np.float64), device=self.dev)  # noqa: E731
        p = f(a.positions)
        self.v1, self.e1, self.e2 = p[:, 0], p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
        self.nrm = f(a.normals)
        self.mid = torch.as_tensor(a.material_ids.astype(np.int64), device=self.dev)
        self.area = 0.5 * torch.linalg.cross(self.e1, self.e2).norm(dim=1)
        self.bsdf = torch.tensor([m.bsdf for m in a.materials], device=self.dev)
        self.kd = f([list(m.kd) for m in a.materials])
        self.emit = 3.0 * f([list(m.ka) for m in a.materials])
        self.lights = torch.nonzero(self.bsdf[self.mid] == ca.EMISSIVE)[:, 0]
        self.light_area = self.area[self.lights].sum()
        self.cam, self.seed = camera, seed

    def block(self, pixel, sample, b):
        zero = torch.zeros_like(pixel)
        return _philox([pixel, sample, zero + b, zero], self.seed & 0xFFFFFFFF, 0)

    def rays(self, pixel, sample):
        c, u = self.cam, self.block(pixel, sample, 0)
        tent = lambda r: torch.where(r < 1, r.clamp(max=1).sqrt() - 1, 1 - (2 - r).clamp(min=0).sqrt())  # noqa: E731
        ni = ((pixel % c.xpixels) + tent(2 * u[0])) / c.xpixels - 0.5
        nj = 0.5 - (torch.div(pixel, c.xpixels, rounding_mode="floor") + tent(2 * u[1])) / c.ypixels
        vec = lambda x: torch.tensor(list(x), dtype=torch.float64, device=self.dev)  # noqa: E731
        d = vec(c.dir) + vec(c.right) * (c.fov * c.aspect * ni)[:, None] + vec(c.up) * (c.fov * nj)[:, None]
        return vec(c.eye).expand(len(pixel), 3), _unit(d)

    def test(self, o, d, tri):
        """Moeller-Trumbore of rays (n, 3) against triangles (m,): distances (n, m), inf
        where there is no hit, and the barycentric coordinates. The triangles' dot and
        cross products are written as matrix products of the rays."""
        v1, e1, e2 = self.v1[tri], self.e1[tri], self.e2[tri]
        n = torch.linalg.cross(e1, e2)
        # det = e1 . (d x e2) = -d . (e1 x e2); with T = o - v1, u det = T . (d x e2) =
        # d . (e2 x T), v det = d . (T x e1), t det = e2 . (T x e1) = T . (e1 x e2)
        det = -(d @ n.T)
        m = torch.linalg.cross(o, d)  # d . (e2 x o) = e2 . m
        u = m @ e2.T - d @ torch.linalg.cross(e2, v1).T
        v = d @ torch.linalg.cross(e1, v1).T - m @ e1.T
        t = o @ n.T - (v1 * n).sum(1)
        u, v, t = u / det, v / det, t / det
        ok = (det.abs() >= 1e-5) & (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1) & (t > 1e-5)
        return torch.where(ok, t, torch.full_like(t, math.inf)), u, v

    def closest(self, o, d):
        n = len(o)
        best = torch.full((n,), math.inf, dtype=torch.float64, device=self.dev)
        rec = torch.full((n,), -1, dtype=torch.int64, device=self.dev)
        bu, bv = torch.zeros_like(best), torch.zeros_like(best)
        step = max(1, min(len(self.v1), 40_000_000 // max(1, n)))
        for k in range(0, len(self.v1), step):
            tri = torch.arange(k, min(k + step, len(self.v1)), device=self.dev)
            t, u, v = self.test(o, d, tri)
            tt, i = t.min(dim=1)
            better = tt < best
            at = i[:, None]
            best = torch.where(better, tt, best)
            rec = torch.where(better, tri[i], rec)
            bu = torch.where(better, u.gather(1, at)[:, 0], bu)
            bv = torch.where(better, v.gather(1, at)[:, 0], bv)
        return best, rec, bu, bv

    def normal(self, rec, u, v):
        n = self.nrm[rec]
        return _unit(n[:, 0] * (1 - u - v)[:, None] + n[:, 1] * u[:, None] + n[:, 2] * v[:, None])

    def radiance(self, pixel, sample, depth, rr_start=3):
        """The estimator's radiance of each pixel-sample."""
        out = torch.zeros(len(pixel), 3, dtype=torch.float64, device=self.dev)
        live = torch.arange(len(pixel), device=self.dev)
        o, d = self.rays(pixel, sample)
        mask, old = torch.ones_like(out), torch.zeros_like(out)  # old: the last sampled direction
        for b in range(depth):
            t, rec, u, v = self.closest(o, d)
            sky = torch.tensor([0.0, 0.025, 0.05], dtype=torch.float64, device=self.dev)
            miss = rec < 0
            out[live[miss]] += mask[miss] * sky
            hit = ~miss
            live, o, d, mask, old = live[hit], o[hit], d[hit], mask[hit], old[hit]
            t, rec, u, v = t[hit], rec[hit], u[hit], v[hit]
            mat = self.mid[rec]
            if b == 0:
                out[live] += mask * self.emit[mat]
            n = self.normal(rec, u, v)
            pos = o + d * t[:, None] + n * 5e-6
            ra, rb = (self.block(pixel[live], sample[live], k + 2 * b) for k in (1, 2))
            diffuse = self.bsdf[mat] == ca.DIFFUSE
            phi, r2 = 2 * math.pi * ra[1], ra[2]
            ey = torch.tensor([0.0, 1.0, 0.0], dtype=torch.float64, device=self.dev)
            axis = torch.where((n[:, :1].abs() > 0.1), ey, ey[[1, 0, 2]])
            uu = _unit(torch.linalg.cross(axis, n))
            vv = torch.linalg.cross(n, uu)
            new = _unit(uu * (phi.cos() * r2.sqrt())[:, None] + vv * (phi.sin() * r2.sqrt())[:, None]
                        + n * (1 - r2).sqrt()[:, None])
            weight = self.kd[mat] * ((new * n).sum(1) * 2)[:, None]
            old = torch.where(diffuse[:, None], new, old)
            mask = torch.where(diffuse[:, None], mask * weight, mask)
            light = self.lights[(ra[3] * (len(self.lights) - 1e-5)).long()]
            lu, lv = rb[0], rb[1]
            fold = lu + lv >= 1
            lu, lv = torch.where(fold, 1 - lu, lu), torch.where(fold, 1 - lv, lv)
            point = self.v1[light] + self.e1[light] * lu[:, None] + self.e2[light] * lv[:, None]
            so, sd = pos + n * 1e-5, _unit(point - pos)
            ts, srec, su, sv = self.closest(so, sd)
            seen = diffuse & (rec != light) & (srec == light)
            cos = (self.normal(light, su, sv) * sd).sum(1).abs()
            direct = self.emit[self.mid[light]] * (self.area[light] / (ts * ts) * cos)[:, None]
            out[live] += torch.where(seen[:, None], mask * direct, torch.zeros_like(mask))
            o, d = pos + old * 1e-5, old
            if b >= rr_start:
                p = mask.max(dim=1).values
                keep = rb[2] <= p
                live, o, d, mask, old = live[keep], o[keep], d[keep], mask[keep] / p[keep][:, None], old[keep]
            # A ray with no direction (a light seen by the camera) hits nothing: the sky.
            if len(live) == 0:
                break
        return out


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("first_hit", "render"):
        return None  # bytes, or gradients and images of scenes too large for brute force
    px, spp = case["w"] * case["h"], case.get("spp", 1)
    if kind == "first_hit" and px * case["tris"] > 2.5e10:
        return None
    if kind == "render" and (case["scene"] != "cornell" or px * spp * case["depth"] > 4e7):
        return None
    rng = _rng(seed)
    key = int(rng.integers(1, 1 << 31))
    mesh = _scene(case["scene"], case["tris"])[0]
    e = _Exact(mesh, _camera(case["scene"], rng, case["w"], case["h"]), key)
    if kind == "first_hit":
        out = []
        for part in torch.arange(px, device=e.dev).split(16384):
            out.append(e.closest(*e.rays(part, torch.zeros_like(part)))[0])
        t = torch.cat(out).cpu().numpy()
        return {"triangle": None, "material": None,
                "t": np.where(np.isinf(t), np.finfo(np.float32).max, t).reshape(case["h"], case["w"])}
    image = torch.zeros(px, 3, dtype=torch.float64, device=e.dev)
    pixels = torch.arange(px, device=e.dev)
    for part in pixels.split(262_144):
        for k in range(spp):
            image[part] += e.radiance(part, torch.full_like(part, k), case["depth"])
    return (image / spp).cpu().numpy().reshape(case["h"], case["w"], 3)
