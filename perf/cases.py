"""The work a program has this library do, as measurable cases.

Each case is one call (or the few calls a program makes together) through the
package's public entry points, at a size of this repository's own workloads:

* build: the LBVH of a set of triangle boxes, with its refit (`GpuBvh`).
* raycast: one closest-hit or any-hit ray a pixel of a view (`Tracer.raycast_on`).
* frame: samples of a path-traced view of one triangle tree (`Tracer.sample`).
* batch: many small scenes rendered in one launch (`Batch.render`).
* pose, forest: new vertices and matrices for a scene of rigid bodies, and a
  frame of it (`Tracer.repose_on`, `reinstance`, `sample`).
* world: one substep of the rigid-body `World`, poses taken to the host.
* denoise: the a-trous denoiser over a traced frame (`Tracer.denoise`).
* infer, train: the learned denoiser (`Kpcn`).
"""
import functools
import math

import numpy as np
import torch

import phiray_amd as P
from phiray_amd import kpcn as K
from phiray_amd import scenes as S


@functools.lru_cache(maxsize=None)
def _gpu():
    gpu = P.Gpu.new(0)
    if gpu is None:
        raise RuntimeError("no HIP device")
    return gpu


# ---- the cases ---------------------------------------------------------------
def listed():
    return [
        # The small tree of an interactive edit: launches and latency count.
        {"name": "build_10007", "kind": "build", "n": 10_007, "leaf": 4, "into_own_arrays": True},
        # The benchmark scene's tree, built again over moved geometry.
        {"name": "build_1310724", "kind": "build", "n": 1_310_724, "leaf": 4, "into_own_arrays": False},
        # Visibility queries: one pinhole ray a pixel of a 256 x 256 view.
        {"name": "raycast_65536", "kind": "raycast", "n": 65_536, "w": 256, "h": 256, "any_hit": False},
        # One sample of a 720p viewport while the user looks around.
        {"name": "preview_720p_1spp", "kind": "frame", "spheres": 16, "level": 4, "w": 1280, "h": 720, "spp": 1},
        # The final frame of the benchmark scene, 1.31M triangles.
        {"name": "frame_1080p_64spp", "kind": "frame", "spheres": 64, "level": 5, "w": 1920, "h": 1080, "spp": 64},
        # Many unrelated scenes of uneven size in one launch (data generation).
        {"name": "batch_32x256x256_16spp", "kind": "batch", "scenes": 32, "w": 256, "h": 256, "spp": 16},
        # A physics substep's new pose for 1,024 bodies, 3.9M triangles.
        {"name": "pose_1024", "kind": "pose", "bodies": 1024},
        # The frame after it, 4 samples at 720p.
        {"name": "forest_720p_4spp", "kind": "forest", "bodies": 1024, "w": 1280, "h": 720, "spp": 4},
        # The physics substep itself.
        {"name": "world_1024", "kind": "world", "bodies": 1024},
        # A noisy 1080p frame cleaned for display.
        {"name": "denoise_1080p", "kind": "denoise", "w": 1920, "h": 1080, "spp": 4},
        # The learned denoiser on the same size of frame.
        {"name": "infer_1080p", "kind": "infer", "b": 1, "w": 1920, "h": 1080},
        # One Adam step of its training, 8 crops of 512 x 512.
        {"name": "train_8x512", "kind": "train", "b": 8, "w": 512, "h": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["build", "raycast", "frame", "batch", "pose", "forest", "world", "denoise", "infer", "train"])
    if kind == "build":
        n = _log_int(rng, 1_000, 1_310_724)
        return {"kind": kind, "n": n, "leaf": rng.choice([1, 4]), "into_own_arrays": n <= P.STATIC_BUILD_MAX and rng.random() < 0.5}
    if kind == "raycast":
        return {"kind": kind, "n": _log_int(rng, 1_000, 200_000), "w": _log_int(rng, 16, 1024), "h": _log_int(rng, 16, 1024),
                "any_hit": rng.random() < 0.3}
    if kind == "frame":
        return {"kind": kind, "spheres": _log_int(rng, 2, 64), "level": rng.choice([2, 3, 4]), "w": _log_int(rng, 64, 1920),
                "h": _log_int(rng, 64, 1080), "spp": _log_int(rng, 1, 16)}
    if kind == "batch":
        return {"kind": kind, "scenes": _log_int(rng, 2, 32), "w": _log_int(rng, 32, 256), "h": _log_int(rng, 32, 256),
                "spp": _log_int(rng, 1, 16)}
    if kind == "pose":
        return {"kind": kind, "bodies": _log_int(rng, 16, 1024)}
    if kind == "forest":
        return {"kind": kind, "bodies": _log_int(rng, 16, 1024), "w": _log_int(rng, 64, 1280), "h": _log_int(rng, 64, 720),
                "spp": _log_int(rng, 1, 4)}
    if kind == "world":
        return {"kind": kind, "bodies": _log_int(rng, 16, 1900)}
    if kind == "denoise":
        return {"kind": kind, "w": _log_int(rng, 64, 1920), "h": _log_int(rng, 64, 1080), "spp": rng.choice([1, 2, 4, 8])}
    if kind == "infer":
        return {"kind": kind, "b": rng.choice([1, 2]), "w": _log_int(rng, 64, 1920), "h": _log_int(rng, 64, 1080)}
    return {"kind": kind, "b": rng.choice([1, 2, 4, 8]), "w": _log_int(rng, 32, 512), "h": _log_int(rng, 32, 512)}


# ---- device arrays as tensors --------------------------------------------------
class _Span:
    def __init__(self, owner, ptr, words, typestr):
        self.owner = owner  # the tensor keeps this object, and so the memory, alive
        self.__cuda_array_interface__ = {"shape": (words,), "typestr": typestr, "data": (ptr, False), "version": 2}


def _tensor(owner, handle, words, dtype=torch.int32):
    """`words` 4-byte words of a device array of `owner`'s, in place."""
    lib = P.lib()
    if words * 4 > lib.phr_array_len(handle) * lib.phr_array_elem(handle):
        raise ValueError("more words than the array holds")
    span = _Span(owner, int(lib.phr_array_device_ptr(handle)), int(words), "<f4" if dtype == torch.float32 else "<i4")
    return torch.as_tensor(span, device="cuda")


def _device_floats(gpu, values):
    """A GpuArray holding a CUDA float tensor's values."""
    a = P.GpuArray.zeroed(gpu, np.float32, values.numel())
    gpu.wait()
    _tensor(a, a._h, values.numel(), torch.float32).copy_(values.reshape(-1))
    torch.cuda.synchronize()
    return a


def _image(tr):
    """The planes a frame leaves: linear sums, first-hit guides, counts."""
    w, h = tr.size
    n = w * h
    px = _tensor(tr, P.lib().phr_tracer_image(tr._h), P.PX_LEN * n + 1)
    f = px.view(torch.float32)
    return {"pixel": px[:n], "radiance": f[n:4 * n], "display": f[4 * n:7 * n], "guides": f[7 * n:14 * n],
            "count": px[31 * n:32 * n]}


# ---- inputs --------------------------------------------------------------------
@functools.lru_cache(maxsize=2)
def _bodies(n):
    """The rigid-body scene's geometry: n bodies, a ground plane and a lamp."""
    builder, worlds = S.bodies_scene(n)
    return builder.arrays(), worlds


def _turned(base, worlds, rng):
    """The bodies' matrices after a small turn and move each."""
    n = len(worlds)
    a = rng.uniform(-0.1, 0.1, n)
    r = np.zeros((n, 4, 4))
    r[:, 0, 0], r[:, 0, 1], r[:, 1, 0], r[:, 1, 1] = np.cos(a), -np.sin(a), np.sin(a), np.cos(a)
    r[:, 2, 2] = r[:, 3, 3] = 1.0
    m = worlds.astype(np.float64).copy()
    m[:, :3, :3] = (r @ m)[:, :3, :3]
    m[:, :3, 3] += rng.uniform(-0.02, 0.02, (n, 3))
    out = base.copy()
    out[:n] = m.transpose(0, 2, 1).reshape(n, 16).astype(np.float32)
    return out


def _frames(b, h, w, seed):
    """Frames like a render at a few samples (smooth albedo, noisy light with
    fireflies, unit normals, some misses), and their smooth targets."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    y = torch.linspace(0, 1, h, device="cuda")[None, :, None, None]
    x = torch.linspace(0, 1, w, device="cuda")[None, None, :, None]
    tone = torch.tensor([1.0, 0.8, 0.6], device="cuda")
    ph = torch.rand(b, 1, 1, 3, generator=g, device="cuda") * 6.0
    light = (0.5 + 0.4 * torch.sin(6 * x + 3 * y + ph)) * tone
    alb = 0.5 + 0.3 * torch.sin(40 * x + ph.flip(-1)) * torch.cos(30 * y + ph)
    target = light * alb
    noise = -torch.log(torch.rand(b, h, w, 1, generator=g, device="cuda").clamp_min(1e-6))
    nrm = torch.randn(b, h, w, 3, generator=g, device="cuda") * 0.2 + torch.tensor([0.0, 0.0, 1.0], device="cuda")
    nrm = nrm / nrm.norm(dim=-1, keepdim=True)
    depth = 2.0 + x + y + 0.1 * torch.rand(b, h, w, 1, generator=g, device="cuda")
    miss = torch.rand(b, h, w, 1, generator=g, device="cuda") < 0.02
    depth = torch.where(miss, torch.full_like(depth, -1.0), depth)
    fr = torch.cat([target * noise, alb.expand(b, h, w, 3), nrm, depth], -1)
    return fr.contiguous(), target.expand(b, h, w, 3).contiguous()


def _rays(case):
    rays = S.pinhole_rays(case["w"], case["h"])
    rays["tmax"] = 10.0  # the scene lies within 3
    return rays


def _spheres(case, seed):
    return S.spheres_scene(spheres=case["spheres"], level=case["level"], seed=seed)


def _tuned(tr):
    """The build the tracer's autotune keeps for one tree on this GPU."""
    tr.set_path_regen(P.Tracer.PATH_SPLIT)
    tr.set_path_waves(4)
    tr.set_samples(1 << 30)
    return tr


def prepare(case, seed):
    gpu, kind = _gpu(), case["kind"]
    st = {"kind": kind, "case": case, "gpu": gpu}
    if kind == "build":
        n = case["n"]
        boxes = S.corner_boxes(S.lbvh_scene(n, seed)[0])
        prims = P.GpuArray.from_(gpu, boxes)
        st["prims"] = prims
        if case["into_own_arrays"]:
            st["nodes"] = P.GpuArray.zeroed(gpu, P.NODE, 2 * n - 1)
            st["order"], st["depth"] = P.GpuArray.zeroed(gpu, np.uint32, n), P.GpuArray.zeroed(gpu, np.uint32, 1)
            st["out"] = [_tensor(st["nodes"], st["nodes"]._h, 8 * (2 * n - 1)), _tensor(st["order"], st["order"]._h, n), _tensor(st["depth"], st["depth"]._h, 1)]
        else:
            st["bvh"] = P.GpuBvh.build_on(gpu, prims, case["leaf"])
            b = st["bvh"]
            st["out"] = [_tensor(b, P.lib().phr_bvh_nodes(b._h), 8 * (2 * n - 1)), _tensor(b, P.lib().phr_bvh_order(b._h), n)]
    elif kind == "raycast":
        corners, _ = S.lbvh_scene(case["n"], seed)
        st["tr"] = P.Tracer.new(gpu, S.tris_from_corners(corners), 4)
        rays = _rays(case)
        st["rays"] = P.GpuArray.from_(gpu, rays)
        st["hits"] = P.GpuArray.zeroed(gpu, P.HIT, len(rays))
        words = _tensor(st["hits"], st["hits"]._h, 5 * len(rays)).view(-1, 5)
        fl = words.view(torch.float32)
        st["out"] = {"t": fl[:, 0], "tri": words[:, 1], "uv": fl[:, 2:4], "inst": words[:, 4]}
    elif kind == "frame":
        st["tr"] = _tuned(P.Tracer.new(gpu, _spheres(case, seed), 4))
        st["cam"] = S.path_camera(case["w"], case["h"], rr_from=3)
    elif kind == "batch":
        tris, lo = S.batch_tris(case["scenes"], seed=seed)
        b = P.Batch(gpu, tris, lo)
        b.set_path(4, 1 if case["scenes"] % 8 == 0 else 0)
        b.set_path_build(P.Tracer.PATH_SPLIT)
        st["batch"] = b
        st["cam"] = S.cloud_camera(case["w"], case["h"], rr_from=3)
        st["px"] = np.zeros((case["scenes"], 4 * case["w"] * case["h"]), dtype=np.uint32)
    elif kind in ("pose", "forest"):
        (v, f, m, me, ins), worlds = _bodies(case["bodies"])
        rng = np.random.default_rng(seed)
        tr = P.Tracer.from_scene(gpu, v, f, m, me, ins, 4)
        tr.set_samples(1 << 30)
        tr.set_path_waves(4)
        moved = v.copy()
        moved["p"][:, :3] *= np.float32(1.0 + 0.02 * rng.random())
        st["tr"], st["verts"] = tr, P.GpuArray.from_(gpu, moved)
        st["worlds"] = _turned(ins["world"], worlds, rng)
        if kind == "pose":
            lib = P.lib()
            st["out"] = [_tensor(tr, x, lib.phr_array_len(x) * lib.phr_array_elem(x) // 4)
                         for x in (lib.phr_tracer_nodes(tr._h), lib.phr_tracer_instances(tr._h))]
        else:
            st["cam"] = S.path_camera(case["w"], case["h"], eye=(0.0, -16.0, 9.0), target=(0.0, 0.0, 1.5), rr_from=3)
            assert tr.repose_on(st["verts"]) and tr.reinstance(st["worlds"])
    elif kind == "world":
        n = case["bodies"]
        world = P.World(gpu)
        world.configure(substeps=1, iterations=10)
        spread = 12.0 * math.sqrt(n / 1024.0)
        ground = world.add_box((spread, spread, 0.5))
        world.add_body(kind=P.PASSIVE, shape=ground, x=(0.0, 0.0, -0.5), friction=1.0)
        for d in S.bodies_defs(n, seed=seed, spread=spread, heights=(1.0, 10.0)):
            r = float(d["r"])
            shape = world.add_box((r, r, r)) if d["shape"] == "box" else world.add_sphere(r)
            world.add_body(shape=shape, x=d["x"], q=d["q"], scale=(r, r, r))
        st["world"] = world
    elif kind == "denoise":
        tr = _tuned(P.Tracer.new(gpu, S.spheres_scene(spheres=16, level=3, seed=seed), 4))
        tr.sample(S.path_camera(case["w"], case["h"], rr_from=3), case["w"], case["h"], case["spp"])
        st["tr"], st["out"] = tr, _image(tr)
    elif kind in ("infer", "train"):
        b, w, h = case["b"], case["w"], case["h"]
        fr, tg = _frames(b, h, w, seed)
        st["frames"] = _device_floats(gpu, fr)
        if kind == "infer":
            st["net"] = P.Kpcn(gpu, K.load(K.WEIGHTS))
            st["image"] = P.GpuArray.zeroed(gpu, np.float32, b * w * h * 3)
            st["out"] = _tensor(st["image"], st["image"]._h, b * w * h * 3, torch.float32)
        else:
            st["net"] = P.Kpcn(gpu, K.init_params(seed % 1000))
            st["targets"] = _device_floats(gpu, tg)
    return st


def _sampled(st):
    st["tr"].sample(st["cam"], st["case"]["w"], st["case"]["h"], st["case"]["spp"])
    if "out" not in st:  # the image is made by the first sample and stays
        st["out"] = _image(st["tr"])
    return st["out"]


def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "build":
        if case["into_own_arrays"]:
            P.GpuBvh.build_static(st["gpu"], st["prims"], st["nodes"], st["order"], st["depth"], case["leaf"])
        else:
            st["bvh"].rebuild_async()
        return st["out"]
    if kind == "raycast":
        st["tr"].raycast_on(st["rays"], st["hits"], case["any_hit"])
        return st["out"]
    if kind == "frame":
        return _sampled(st)
    if kind == "batch":
        b, px = st["batch"], st["px"]
        b.render(st["cam"], case["w"], case["h"], case["spp"])
        for k in range(case["scenes"]):  # each scene's packed pixels and linear sums, to the host
            P._check(P.lib().phr_batch_px(b._h, k, 0, px.shape[1], P._ptr(px[k])), "Batch px")
        n = case["w"] * case["h"]
        return {"pixel": px[:, :n].view(np.int32), "radiance": px[:, n:].view(np.float32)}
    if kind == "pose":
        assert st["tr"].repose_on(st["verts"]) and st["tr"].reinstance(st["worlds"])
        return st["out"]
    if kind == "forest":
        return _sampled(st)
    if kind == "world":
        st["world"].step(1.0 / 60.0 / 8.0)
        poses, bodies = st["world"].poses(), st["world"].bodies()
        return {"poses": poses, "x": bodies["x"], "q": bodies["q"], "v": bodies["v"], "w": bodies["w"]}
    if kind == "denoise":
        st["tr"].denoise(keep=False)
        return {k: st["out"][k] for k in ("radiance", "display", "pixel")}
    if kind == "infer":
        st["net"].infer(st["frames"], case["b"], case["w"], case["h"], st["image"])
        return st["out"]
    st["net"].train_step(st["frames"], st["targets"], case["b"], case["w"], case["h"], 1e-4, want_loss=False)
    return st["net"].grads()


# ---- what a pass cannot do without ---------------------------------------------
FLOP_PX = 155_000.0  # the network's multiply-adds a pixel, times two


def work(case):
    kind = case["kind"]
    px = case.get("w", 0) * case.get("h", 0)
    if kind == "build":
        # Boxes in; order and about one 32-byte node a box out.
        return {"bytes": case["n"] * (32 + 4 + 32), "flops": case["n"] * 60}
    if kind == "raycast":
        return {"bytes": case["n"] * (36 + 32) + px * (32 + 20), "flops": px * 26 * 30}
    if kind == "frame":
        # About 2.7 rays a sample, 26 box steps and 3.5 triangle tests a ray.
        tris = case["spheres"] * 20 * 4 ** case["level"]
        return {"bytes": tris * (36 + 32) + px * 4 * 22, "flops": px * case["spp"] * 2.7 * (26 * 30 + 3.5 * 50)}
    if kind == "batch":
        return {"bytes": case["scenes"] * (37_500 * (36 + 32) + px * 4 * 22),
                "flops": case["scenes"] * px * case["spp"] * 2.7 * (26 * 30 + 3.5 * 50)}
    if kind == "pose":
        # 3,800 triangles a body: vertices in, their nodes written.
        return {"bytes": case["bodies"] * 3_800 * (16 + 32 + 32), "flops": case["bodies"] * 3_800 * 40}
    if kind == "forest":
        return {"bytes": case["bodies"] * 3_800 * (36 + 32) + px * 4 * 22,
                "flops": px * case["spp"] * 3.7 * (30 * 30 + 3.5 * 50)}
    if kind == "world":
        # 3 pairs a body, 4 points a pair, 10 iterations of a projection.
        return {"bytes": case["bodies"] * (64 * 2 + 48 + 64), "flops": case["bodies"] * 3 * 4 * 10 * 200}
    if kind == "denoise":
        # Radiance, albedo, normal, depth, counts in; radiance, display, pixel out.
        return {"bytes": px * 4 * (3 + 3 + 3 + 1 + 2 + 3 + 3 + 1), "flops": px * 4 * 25 * 40}
    n = case["b"] * px
    if kind == "infer":
        return {"bytes": n * (40 + 12), "flops": n * FLOP_PX}
    return {"bytes": n * (40 + 12) + 337_801 * 4 * 7, "flops": n * FLOP_PX * 3}


def tolerance(case):
    kind = case["kind"]
    if kind in ("build", "pose"):
        return "exact"  # node words and slot orders
    if kind == "raycast":
        return {"rel": 3e-5, "max": 1e-3, "differ": 0.0}
    if kind in ("frame", "batch", "forest"):
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-4}  # packed bytes may round apart
    if kind == "world":
        return {"rel": 1e-3, "max": 4e-2}  # velocities are position differences over 1/480 s
    if kind == "denoise":
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-2}
    if kind == "infer":
        return {"rel": 1e-2, "max": 0.4}
    return {"rel": 2e-2, "max": 0.8}


# ---- the same in 64 bits ---------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "raycast" and case["n"] * case["w"] * case["h"] <= 1.5e10 and not case["any_hit"]:
        return _exact_raycast(case, seed)
    if kind == "denoise":
        return _exact_denoise(case, seed)
    if kind == "infer":
        fr, _ = _frames(case["b"], case["h"], case["w"], seed)
        return _net(_layers(K.load(K.WEIGHTS)), fr.double()).reshape(-1)
    if kind == "train" and case["b"] * case["w"] * case["h"] <= 8 * 512 * 512:
        fr, tg = _frames(case["b"], case["h"], case["w"], seed)
        ls = [(w.requires_grad_(True), b.requires_grad_(True)) for w, b in _layers(K.init_params(seed % 1000))]
        y, t = _net(ls, fr.double()), tg.double()
        torch.mean((y - t) ** 2 / (t * t + 0.01)).backward()
        return torch.cat([g for w, b in ls for g in (w.grad.reshape(-1), b.grad)]).cpu().numpy()
    return None


def _exact_raycast(case, seed):
    """Every triangle against every ray (Moller and Trumbore's test)."""
    c = torch.tensor(S.lbvh_scene(case["n"], seed)[0], device="cuda").double()
    rays = _rays(case)
    o, dirs = torch.tensor(rays["o"][0].copy(), device="cuda").double(), torch.tensor(rays["d"].copy(), device="cuda").double()
    e1, e2, s = c[:, 1] - c[:, 0], c[:, 2] - c[:, 0], o - c[:, 0]
    # With one origin each triangle's terms are linear in the direction.
    nrm, q = torch.cross(e1, e2, dim=1), torch.cross(s, e1, dim=1)
    a = torch.stack([-nrm, torch.cross(e2, s, dim=1), q])  # det, u, v numerators over d
    tn = (e2 * q).sum(1)
    far = torch.full((), float("inf"), device="cuda", dtype=torch.float64)
    t_out, uv = torch.empty(len(dirs), device="cuda", dtype=torch.float64), torch.zeros(len(dirs), 2, device="cuda", dtype=torch.float64)
    for lo in range(0, len(dirs), 1024):
        d = dirs[lo:lo + 1024]
        det, u, v = (d @ m.T for m in a)
        u, v, t = u / det, v / det, tn / det
        t = torch.where((u >= 0) & (v >= 0) & (u + v <= 1) & (t > 0), t, far)
        best, k = t.min(1)
        hit = torch.isfinite(best)
        i = torch.arange(len(d), device="cuda")
        t_out[lo:lo + 1024] = torch.where(hit, best, torch.tensor(float(rays["tmax"][0]), device="cuda", dtype=torch.float64))
        # The library's u, v are the weights of the second and third corner.
        uv[lo:lo + 1024] = torch.where(hit[:, None], torch.stack([u[i, k], v[i, k]], 1), 0.0)
    return {"t": t_out, "tri": None, "uv": uv, "inst": None}


def _exact_denoise(case, seed):
    """Four a-trous passes (5 x 5 B3 spline taps at spacing 1, 2, 4, 8) over
    the light without its albedo, guided by first-hit albedo, normal, depth
    and the light itself; the first pass clamps fireflies."""
    st = prepare(case, seed)
    torch.cuda.synchronize()
    w, h = case["w"], case["h"]
    n = w * h
    px = _tensor(st["tr"], P.lib().phr_tracer_image(st["tr"]._h), P.PX_LEN * n + 1).clone()
    f = px.view(torch.float32).double()
    cnt = px[31 * n:32 * n].double().clamp_min(1.0).reshape(h, w, 1)
    rad, alb = f[n:4 * n].reshape(h, w, 3) / cnt, f[7 * n:10 * n].reshape(h, w, 3) / cnt
    x = alb.clamp(0, 1)
    alb = torch.where(x <= 0.0031308, x * 12.92, 1.055 * x.clamp_min(1e-300) ** (1 / 2.4) - 0.055)
    nrm = f[10 * n:13 * n].reshape(h, w, 3) + 1e-9
    nrm = nrm / nrm.norm(dim=-1, keepdim=True)
    dep = f[13 * n:14 * n].reshape(h, w, 1) / cnt
    col = rad / alb.clamp_min(0.05)
    lw = torch.tensor([0.2126, 0.7152, 0.0722], device="cuda", dtype=torch.float64)

    def luma(c):
        return (c * lw).sum(-1, keepdim=True)

    def at(img, dy, dx, fill=0.0):
        out = torch.full_like(img, fill)
        ys, xs = slice(max(0, -dy), min(h, h - dy)), slice(max(0, -dx), min(w, w - dx))
        yt, xt = slice(max(0, dy), min(h, h + dy)), slice(max(0, dx), min(w, w + dx))
        if ys.start < ys.stop and xs.start < xs.stop:
            out[ys, xs] = img[yt, xt]
        return out

    one = torch.ones_like(dep)
    for step in (1, 2, 4, 8):
        mid = col
        if step == 1:
            ring = [(dy, dx) for dy in (-1, 0, 1) for dx in (-1, 0, 1) if dy or dx]
            cs = [at(col, *o) for o in ring]
            near = sum(at(one, *o) for o in ring)
            top = torch.stack([luma(c) for c in cs]).amax(0).clamp_min(0.0)
            mid = torch.where((near > 0) & (luma(col) > 1.5 * top + 0.05), sum(cs) / near.clamp_min(1.0), col)
        lc, total, weight = luma(mid), torch.zeros_like(col), torch.zeros_like(dep)
        for dy in range(-2, 3):
            for dx in range(-2, 3):
                o = (dy * step, dx * step)
                tap = mid if dy == 0 and dx == 0 else at(col, *o)
                dj = at(dep, *o)
                dn = (1.0 - (nrm * at(nrm, *o)).sum(-1, keepdim=True)).clamp_min(0.0)
                da = (at(alb, *o) - alb).norm(dim=-1, keepdim=True)
                dd = (dj - dep).abs() / dep.abs().clamp_min(1e-3)
                dl = (luma(tap) - lc).abs() / (0.08 + lc)
                k = (0.375, 0.25, 0.0625)[abs(dx)] * (0.375, 0.25, 0.0625)[abs(dy)]
                s = k * torch.exp(-dn * 64 - da * 8 - dd * 40 - dl * dl * 7)
                s = s * at(one, *o) * ((dj < 0) == (dep < 0))
                total, weight = total + tap * s, weight + s
        col = torch.where(weight > 0, total / weight.clamp_min(1e-300), mid)
    met = 1.0 - f[33 * n:34 * n].reshape(h, w, 1) / cnt
    lin = torch.where(met > 0.5 / cnt, col * alb.clamp_min(0.05), torch.zeros_like(col))
    return {"radiance": (lin * cnt).reshape(-1), "display": None, "pixel": None}


def _layers(params):
    """(weights [9, cout, cin], bias) a layer, in 64 bits."""
    out = []
    for ws, bs, (cout, cin) in K.layer_slices():
        out.append((torch.tensor(params[ws].reshape(9, cout, cin), device="cuda").double(),
                    torch.tensor(params[bs], device="cuda").double()))
    return out


def _net(ls, fr):
    """The network over frames [b, h, w, 10]: the denoised radiance."""
    b, h, w, _ = fr.shape
    hp, wp = (h + 7) // 8 * 8, (w + 7) // 8 * 8
    base = fr[..., 3:6].clamp_min(0.05)
    light = fr[..., :3] / base
    z = fr[..., 9:]
    z = torch.where(z < 0, torch.full_like(z, -1.0), z / (1.0 + z))
    x = torch.cat([torch.log1p(light.clamp_min(0.0)), fr[..., 3:9], z, torch.zeros(b, h, w, 6, device=fr.device, dtype=fr.dtype)], -1)
    x = x[:, torch.arange(hp, device=fr.device).clamp_max(h - 1)][:, :, torch.arange(wp, device=fr.device).clamp_max(w - 1)]

    def conv(i, x):
        wt, bias = ls[i]
        _, hh, ww, c = x.shape
        p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        y = bias
        for t in range(9):
            y = y + (p[:, t // 3:t // 3 + hh, t % 3:t % 3 + ww].reshape(-1, c) @ wt[t].T)
        y = y.reshape(b, hh, ww, -1)
        return y if i == 10 else torch.relu(y)

    def pool(x):
        return (x[:, ::2, ::2] + x[:, 1::2, ::2] + x[:, ::2, 1::2] + x[:, 1::2, 1::2]) * 0.25

    def up(x):
        return x.repeat_interleave(2, 1).repeat_interleave(2, 2)

    a0 = conv(1, conv(0, x))
    a1 = conv(3, conv(2, pool(a0)))
    a2 = conv(5, conv(4, pool(a1)))
    d2 = conv(7, torch.cat([up(conv(6, pool(a2))), a2], -1))
    d1 = conv(8, torch.cat([up(d2), a1], -1))
    d0 = conv(9, torch.cat([up(d1), a0], -1))
    k = torch.softmax(conv(10, d0)[:, :h, :w, :25], -1)
    ys, xs = torch.arange(h, device=fr.device), torch.arange(w, device=fr.device)
    out = torch.zeros_like(light)
    for t in range(25):
        tap = light[:, (ys + t // 5 - 2).clamp(0, h - 1)][:, :, (xs + t % 5 - 2).clamp(0, w - 1)]
        out = out + k[..., t:t + 1] * tap
    return base * out
