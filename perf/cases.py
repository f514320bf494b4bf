"""Cases for timing the framework's public entry points on one GPU.

A case is one call (or the few calls) that a program which traces rays or renders images makes
again and again: a flat batch of rays cast against a device scene, a batch of environment
samples or densities, some bounces of a resident render followed by the preview image, the same
for a batch of jobs or with the path guide, and a scene rebuilt on the device. Meshes and images are
procedural, so a seed chooses the rays, the RNG states, the render's random sequence or the
displacement of a mesh; scenes, lanes and buffers are prepared once and kept, as such a program
does.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from raccoongpurender_amd import _lib, render_scenes, render_workloads, scenes
from raccoongpurender_amd import guide as guiding
from raccoongpurender_amd.render import build_lane

FAR = 16.0  # far clip of the flat ray batches: beyond the meshes (radius about 1.15)


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # secondary rays of a large render as one flat batch: the ray-cast benchmark's own sizes
        dict(name="cast_incoherent", kind="cast", rays="incoherent", level=8, count=4194304, variant="stackless",
             block=0),
        # camera rays of one HD frame (one thread per ray, the launch for coherent rays)
        dict(name="cast_primary_1080p", kind="cast", rays="primary", level=8, count=1920 * 1080, variant="threaded",
             block=256),
        # a mid-size mesh and an odd number of rays through the threaded tables
        dict(name="cast_threaded_ragged", kind="cast", rays="incoherent", level=6, count=1000003, variant="threaded",
             block=0),
        # picking or visibility queries: a few thousand rays on a small mesh, where latency counts
        dict(name="cast_small", kind="cast", rays="incoherent", level=4, count=4097, variant="stackless", block=0),
        # next-event directions for a frame's worth of vertices under a large sky
        dict(name="env_sample_six_axis", kind="env_sample", width=2048, height=1024, count=4194301, normals=True),
        # densities of BSDF-sampled directions, a small map and an odd count
        dict(name="env_pdf_uniform", kind="env_pdf", width=512, height=256, count=1000003, normals=False),
        # the full-render workload: HD, 2 million triangles, every material, 2^22 resident paths
        dict(name="render_1080p", kind="render", scene="full", width=1920, height=1080, paths=1 << 22, steps=4,
             graph=False, variant="stackless", block=64),
        # an interactive Cornell box, its bounces replayed from a captured graph
        dict(name="render_cornell_graph", kind="render", scene="cornell", width=256, height=256, paths=1 << 18,
             steps=16, graph=True, variant="stackless", block=256),
        # a thumbnail with few paths, one bounce a call: launches dominate
        dict(name="render_thumbnail", kind="render", scene="materials", width=67, height=45, paths=4096, steps=1,
             graph=False, variant="threaded", block=256),
        # several small jobs in one wavefront, their images read back
        dict(name="batch_previews", kind="batch", jobs=8, side=160, paths=32768, steps=8),
        # guided rendering that trains its network while it renders
        dict(name="render_guided", kind="guided", scene="materials", width=640, height=480, paths=1 << 20, steps=8,
             capacity=1 << 16),
        # a mesh that changes: its tree rebuilt on the device, the scene uploaded, a batch cast
        dict(name="rebuild_and_cast", kind="rebuild", rays="incoherent", level=7, leaf=4, bins=16, count=262144,
             variant="stackless", block=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("cast", "cast", "cast", "env_sample", "env_pdf", "render", "render", "batch", "guided", "rebuild"))
    if kind == "cast":
        return dict(kind=kind, rays=rng.choice(("incoherent", "incoherent", "primary")), level=rng.randint(3, 8),
                    count=_log_int(rng, 1000, 4000000), variant=rng.choice(("stackless", "stackless", "threaded")),
                    block=rng.choice((0, 64, 256)))
    if kind in ("env_sample", "env_pdf"):
        h = _log_int(rng, 32, 1024)
        return dict(kind=kind, width=2 * h, height=h, count=_log_int(rng, 300000, 4000000),
                    normals=rng.choice((True, False)))
    if kind == "render":
        w = _log_int(rng, 64, 1280)
        return dict(kind=kind, scene=rng.choice(("cornell", "materials", "full")), width=w,
                    height=max(32, int(w * rng.uniform(0.5, 1.0))), paths=_log_int(rng, 4096, 1 << 21),
                    steps=rng.randint(1, 8), graph=rng.choice((True, False)),
                    variant=rng.choice(("stackless", "threaded")), block=rng.choice((64, 128, 256)))
    if kind == "batch":
        return dict(kind=kind, jobs=rng.randint(2, 12), side=_log_int(rng, 64, 256), paths=_log_int(rng, 1024, 65536),
                    steps=rng.randint(2, 12))
    if kind == "guided":
        w = _log_int(rng, 96, 800)
        return dict(kind=kind, scene=rng.choice(("cornell", "materials")), width=w, height=max(64, int(0.75 * w)),
                    paths=_log_int(rng, 16384, 1 << 20), steps=rng.randint(2, 8), capacity=1 << rng.randint(14, 17))
    return dict(kind=kind, rays="incoherent", level=rng.randint(3, 7), leaf=rng.choice((1, 2, 4, 8)),
                bins=rng.choice((8, 16, 32)), count=_log_int(rng, 1000, 1000000),
                variant=rng.choice(("stackless", "threaded")), block=rng.choice((0, 64, 256)))


# ---------------------------------------------------------------- what a program has in hand
@functools.lru_cache(maxsize=None)
def _context():
    return _lib.Context(0)


@functools.lru_cache(maxsize=None)
def _mesh(level):
    return scenes.displaced_icosphere(level=level)


@functools.lru_cache(maxsize=None)
def _sky(width, height):
    return render_scenes.sky_envmap(width, height)


@functools.lru_cache(maxsize=None)
def _full():
    return render_workloads.full_render_scene()


def _scene_dict(name, width, height):
    if name == "full":
        sd = dict(_full())
    elif name == "cornell":
        sd = dict(render_scenes.cornell_box(width, height), max_depth=5)
    else:
        sd = dict(render_scenes.material_test_scene(width, height, env_size=(256, 128)), max_depth=8)
    sd["camera"] = dict(sd["camera"], width=width, height=height)
    return sd


class _Buffer:
    """A torch tensor as the device buffer of an entry point."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _unit(n, g):
    v = torch.randn(n, 3, device="cuda", generator=g, dtype=torch.float64)
    return v / v.norm(dim=1, keepdim=True)


def _rays(case, seed):
    """The case's rays, n x 8 floats (origin, far clip, direction, 0): incoherent ones start
    uniformly in the mesh's box with uniform directions; primary ones go row by row through a
    jittered pixel of a frame seen from distance 3."""
    n, g = case["count"], _generator(seed)
    rays = torch.zeros(n, 8, device="cuda")
    rays[:, 3] = FAR
    if case["rays"] == "incoherent":
        v, _ = _mesh(case["level"])
        lo = torch.from_numpy(v.min(0)).to("cuda")
        hi = torch.from_numpy(v.max(0)).to("cuda")
        rays[:, 0:3] = lo + (hi - lo) * torch.rand(n, 3, device="cuda", generator=g)
        rays[:, 4:7] = _unit(n, g).float()
    else:
        w = max(1, int(math.sqrt(n * 16.0 / 9.0)))
        h = (n + w - 1) // w
        i = torch.arange(n, device="cuda")
        j = torch.rand(n, 2, device="cuda", generator=g, dtype=torch.float64)
        half = math.tan(math.radians(22.5))
        x = ((i % w + j[:, 0]) / w * 2.0 - 1.0) * half * w / h
        y = (1.0 - (torch.div(i, w, rounding_mode="floor") + j[:, 1]) / h * 2.0) * half
        d = torch.stack([x, y, -torch.ones_like(x)], 1)
        rays[:, 2] = 3.0
        rays[:, 4:7] = (d / d.norm(dim=1, keepdim=True)).float()
    return rays


def _bent(case, seed):
    """The case's mesh in another pose."""
    v, f = _mesh(case["level"])
    a = np.random.default_rng(seed).uniform(-0.05, 0.05, 3)
    return np.ascontiguousarray(v * (1.0 + np.sin(v[:, [1, 2, 0]] * 3.0) * a), np.float32), f


def _lane(ctx, case, seed):
    sd = _scene_dict(case["scene"], case["width"], case["height"])
    wf = build_lane(ctx, sd, case["paths"], seed=seed)
    wf.set_launch(case.get("variant", "stackless"), case.get("block", 64), wf.get_launch()[2])
    c = sd["camera"]
    cam = _lib.camera_look_at(c["eye"], c["target"], c["up"], c["fov"], c["width"], c["height"], c["lens_radius"])
    return wf, cam


def prepare(case, seed):
    ctx = _context()
    kind = case["kind"]
    if kind == "cast":
        v, f = _mesh(case["level"])
        scene = _lib.Scene(ctx, _lib.BVH(v, f))
        hits = torch.zeros(case["count"], 4, device="cuda")
        return dict(case=case, scene=scene, rays=_Buffer(_rays(case, seed)), hits=_Buffer(hits))
    if kind in ("env_sample", "env_pdf"):
        n, g = case["count"], _generator(seed)
        env = _lib.Envmap(ctx, _sky(case["width"], case["height"]))
        normals = _Buffer(_unit(n, g).float().contiguous()) if case["normals"] else None
        if kind == "env_pdf":
            return dict(case=case, env=env, normals=normals, dirs=_Buffer(_unit(n, g).float().contiguous()),
                        out=_Buffer(torch.zeros(n, device="cuda")))
        states = torch.randint(-(1 << 31), 1 << 31, (n, 4), device="cuda", generator=g, dtype=torch.int64)
        return dict(case=case, env=env, normals=normals, states=_Buffer(states.to(torch.int32)),
                    out=_Buffer(torch.zeros(n, 4, device="cuda")))
    if kind in ("render", "guided"):
        wf, cam = _lane(ctx, case, seed)
        state = dict(case=case, lane=wf,
                     image=_Buffer(torch.zeros(case["width"] * case["height"], 6, device="cuda", dtype=torch.int16)))
        if kind == "guided":
            v = wf._keep[0].points
            state["guide"] = guiding.Guide(ctx, scene_lo=v.min(0) - 1e-3, scene_hi=v.max(0) + 1e-3,
                                           capacity=case["capacity"], seed=1 + seed % 1000)
            guiding.attach(wf, state["guide"])
        wf.initialize(cam)
        if case.get("graph"):
            wf.graph_capture(case["steps"])
        return state
    if kind == "batch":
        jobs, keep = [], []
        for name in ("materials", "cornell"):
            sd = _scene_dict(name, 64, 64)
            bvh = _lib.BVH(sd["points"], sd["indices"])
            keep.append((sd, _lib.Scene(ctx, bvh), _lib.Materials(ctx, sd["materials"]), _lib.Envmap(ctx, sd["env"])))
        for k in range(case["jobs"]):
            sd, scene, mats, env = keep[k % 2]
            c, w = sd["camera"], case["side"] + 24 * (k % 3)
            cam = _lib.camera_look_at(c["eye"], c["target"], c["up"], c["fov"], w, case["side"], c["lens_radius"])
            jobs.append(_lib.BatchJob(scene, mats, env, cam, case["paths"], seed=seed + 7919 * k))
        return dict(case=case, batch=_lib.Batch(ctx, jobs, max_depth=8), keep=keep)
    points, f = _bent(case, seed)
    hits = torch.zeros(case["count"], 4, device="cuda")
    return dict(case=case, ctx=ctx, points=points, indices=f, rays=_Buffer(_rays(case, seed)), hits=_Buffer(hits))


# ---------------------------------------------------------------- one pass
def _image(buffer):
    """The half-float means and sample counts of an intermediate image, as views of its buffer."""
    return {"mean": buffer.tensor.view(torch.float16)[:, :3], "count": buffer.tensor.view(torch.int32)[:, 2]}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("cast", "rebuild"):
        if kind == "rebuild":
            bvh = _lib.BVH(state["points"], state["indices"], max_leaf=case["leaf"], bins=case["bins"],
                           device=state["ctx"])
            state["scene"] = _lib.Scene(state["ctx"], bvh)
        state["scene"].extension_ray_cast(case["variant"], state["rays"], state["hits"], case["count"], case["block"])
        h = state["hits"].tensor
        return {"prim": h.view(torch.int32)[:, 0], "t": h[:, 1], "u": h[:, 2], "v": h[:, 3]}
    if kind == "env_sample":
        state["env"].sample_device(state["states"], state["out"], case["count"], state["normals"])
        return {"states": state["states"].tensor, "sample": state["out"].tensor}
    if kind == "env_pdf":
        state["env"].pdf_device(state["dirs"], state["out"], case["count"], state["normals"])
        return state["out"].tensor
    if kind == "render":
        lane = state["lane"]
        if case["graph"]:
            lane.graph_launch(1)
        else:
            lane.step(case["steps"])
        lane.intermediate(state["image"])
        return _image(state["image"])
    if kind == "guided":
        lane = state["lane"]
        lane.step(case["steps"])
        trained = guiding.train_pass(lane, case["capacity"] // 2)
        lane.intermediate(state["image"])
        return dict(_image(state["image"]), trained=trained, weights=state["guide"].params())
    batch = state["batch"]
    batch.step(case["steps"])
    return [batch.job_accumulation(k) for k in range(case["jobs"])]


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind in ("cast", "rebuild"):
        # rays in, hits out, the scene's nodes and primitives once (or the part that few rays
        # reach); a descent of the tree's depth with two box tests a node, three triangle tests
        n, tris = case["count"], 20 * 4 ** case["level"]
        per_ray = math.log2(tris)
        w = dict(bytes=48.0 * n + min(112.0 * tris, 64.0 * per_ray * n), flops=n * (per_ray * 2 * 22 + 3 * 50))
        if kind == "rebuild":
            # vertices and indices in, the scene's tables out; a sweep over the primitives a level
            w["bytes"] += tris * (6.0 + 12.0 + 2 * 64.0 + 48.0 + 8.0 + 12.0)
            w["flops"] += tris * math.log2(tris) * 60.0
        return w
    if kind in ("env_sample", "env_pdf"):
        n = case["count"]
        if kind == "env_sample":
            return dict(bytes=n * (100.0 if case["normals"] else 76.0), flops=n * 100.0)
        return dict(bytes=n * (44.0 if case["normals"] else 20.0), flops=n * 100.0)
    if kind in ("render", "guided"):
        # per path and bounce: ray, path, hit and shading records and the RNG state read and
        # written once; per pixel the sums and the preview; the traversal as in a cast
        n, px = case["paths"] * case["steps"], case["width"] * case["height"]
        depth = {"full": 21.0, "cornell": 12.0, "materials": 10.0}[case["scene"]]
        w = dict(bytes=n * 176.0 + px * 28.0, flops=n * (depth * 2 * 22 + 3 * 50 + 400))
        if kind == "guided":
            w["flops"] += 37e3 * n * 0.5 + 111e3 * case["capacity"]
            w["bytes"] += 64.0 * case["capacity"]
        return w
    n, px = case["jobs"] * case["paths"] * case["steps"], case["jobs"] * case["side"] * (case["side"] + 24)
    return dict(bytes=n * 176.0 + px * 32.0, flops=n * (11 * 2 * 22 + 3 * 50 + 400))


# ---------------------------------------------------------------- the same in 64 bits
def _exact_cast(case, seed):
    v, f = _bent(case, seed) if case["kind"] == "rebuild" else _mesh(case["level"])
    if case["count"] * len(f) > 6e8:
        return None  # every ray against every triangle would take too long
    rays = _rays(case, seed).double()
    p = torch.from_numpy(v).to("cuda").double()[torch.from_numpy(f.astype(np.int64)).to("cuda")]
    v0, e1, e2 = p[:, 0], p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    step = max(1, int(2e7) // len(f))
    t, u, w = [], [], []
    for at in range(0, len(rays), step):
        o, d = rays[at:at + step, None, 0:3], rays[at:at + step, None, 4:7]
        pv = torch.linalg.cross(d, e2[None])
        inv = 1.0 / (e1 * pv).sum(-1)
        tv = o - v0
        uu = (tv * pv).sum(-1) * inv
        qv = torch.linalg.cross(tv, e1[None].expand_as(tv))
        ww = (d * qv).sum(-1) * inv
        tt = (e2 * qv).sum(-1) * inv
        ok = (uu >= 0) & (ww >= 0) & (uu + ww <= 1) & (tt >= 0) & (tt <= FAR)
        best, k = torch.where(ok, tt, torch.full_like(tt, math.inf)).min(1)
        hit = torch.isfinite(best)
        t.append(torch.where(hit, best, torch.full_like(best, FAR)))
        u.append(torch.where(hit, uu.gather(1, k[:, None])[:, 0], torch.zeros_like(best)))
        w.append(torch.where(hit, ww.gather(1, k[:, None])[:, 0], torch.zeros_like(best)))
    return {"prim": None, "t": torch.cat(t), "u": torch.cat(u), "v": torch.cat(w)}


def _exact_pdf(case, seed):
    """Selection probability over solid angle of each direction's texel (mixed by the squared
    normal over the axis-weighted tables where normals are given)."""
    n, g, W, H = case["count"], _generator(seed), case["width"], case["height"]
    nrm = _unit(n, g).float().double() if case["normals"] else None
    d = _unit(n, g).float().double()
    rgb = torch.from_numpy(_sky(W, H)).to("cuda").double()
    theta = torch.arange(H + 1, device="cuda", dtype=torch.float64) * (math.pi / H)
    sr = (theta[:-1].cos() - theta[1:].cos()) * (2.0 * math.pi / W)
    tc = (theta[:-1] + theta[1:]) * 0.5
    pc = 2.0 * math.pi - (torch.arange(W, device="cuda", dtype=torch.float64) + 0.5) * (2.0 * math.pi / W)
    lum = (0.2126 * rgb[..., 0] + 0.7152 * rgb[..., 1] + 0.0722 * rgb[..., 2]) * sr[:, None]
    centre = [tc.sin()[:, None] * pc.sin(), tc.cos()[:, None].expand(H, W), tc.sin()[:, None] * pc.cos()]

    def table(weight):
        p = lum * weight
        return (p / p.sum() / sr[:, None]).reshape(-1)

    th = torch.atan2((d[:, 2] ** 2 + d[:, 0] ** 2).sqrt(), d[:, 1])
    ph = torch.atan2(d[:, 0], d[:, 2])
    ix = torch.floor((1.0 - ph / (2.0 * math.pi)) * W).long() % W
    iy = torch.floor(th / math.pi * H).long().clamp(0, H - 1)
    at = iy * W + ix
    if nrm is None:
        return table(torch.ones_like(lum))[at]
    pdf = torch.zeros(n, device="cuda", dtype=torch.float64)
    for k in range(3):
        plus, minus = table(centre[k].clamp(min=0.0))[at], table((-centre[k]).clamp(min=0.0))[at]
        pdf += nrm[:, k] ** 2 * torch.where(nrm[:, k] > 0, plus, minus)
    return pdf


def exact(case, seed):
    if case["kind"] in ("cast", "rebuild"):
        return _exact_cast(case, seed)
    if case["kind"] == "env_pdf":
        return _exact_pdf(case, seed)
    # drawn directions and rendered images follow from integer random numbers and discrete
    # choices along each path
    return None
