"""What this renderer is measured on: passes through its Python binding (cwp) as programs make them.

A case is one of six kinds of work, over the sizes and options its users have:

* frame  - one wavefront pass of a still image (Renderer.render): the legacy or the full integrator, any BVH layout and
           triangle test, square, wide and odd image sizes, 1 to 256 samples per pixel in flight. The image stays on the
           device (accum_device), or is read back to the host as the batch command line does (host = 1).
* view   - one frame of the interactive viewer: the camera moves, a few samples are rendered into a cleared
           accumulation, and the display transform gives the 8-bit image on the host.
* anim   - one frame of a two-level animation: the instances' transforms change, the TLAS is rebuilt on the GPU, the
           frame is rendered.
* rays   - explicit rays in device memory against a resident scene (baking, visibility queries): closest hits, any-hit
           queries, or one after the other.
* build  - a BVH over triangle boxes in device memory: the H-PLOC build and its collapse to a compressed BVH8.
* jobs   - a stream of render jobs through the job server, images fetched at the end.

Needs a GPU. torch is imported before cwp, so that both use one HIP runtime.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuda-wavefront-pathtracer_amd"))
import cwp  # noqa: E402

# the sun and sky of the benchmark frames (bench.py)
LIGHTING = ["--sun_to", "0.608749", "-0.42625", "0.669131", "--sun_rgb", "3", "3", "3", "--sun_angle", "0.526",
            "--sky", "0.3", "0.38", "0.5"]


def listed():
    return [
        # The benchmark's headline frame: 118 k triangles, 256 samples per pixel in flight, 8 bounces, the first
        # bounce's continuations sorted. The largest still image.
        frame("frame-720p-256spp", w=1280, h=720, spp=256, bounces=8, sort=2, filter="box"),
        # The published diffuse configuration of the renderer this one follows: BVH2, 4 bounces.
        frame("frame-720p-bvh2", w=1280, h=720, spp=64, bounces=4, bvh=2, filter="box"),
        # The command line's defaults (512 x 512, 64 samples in flight, 8 bounces, BVH8), with the watertight test that
        # a user takes who cannot have cracks.
        frame("frame-512-watertight", w=512, h=512, spp=64, bounces=8, tri="watertight"),
        # A small still image read back to the host: 1,024 boxes, 256 x 256, 16 samples, 4 bounces.
        frame("frame-256-boxes-host", scene="boxes", w=256, h=256, spp=16, bounces=4, host=1),
        # The full material integrator (OpenPBR-subset materials, emitters, environment map, MIS) at the benchmark's size.
        frame("frame-720p-full", w=1280, h=720, spp=64, bounces=8, full=1, filter="box"),
        # The same with texture and normal maps on an odd, smaller image.
        frame("frame-639x361-textured", w=639, h=361, spp=16, bounces=6, full=1, tex=512),
        # The smallest calls: one sample per pixel of a small odd image while the camera moves.
        view("view-321x181-1spp", scene="boxes", w=321, h=181, spp=1, bounces=4),
        # An ordinary viewer frame: 720p, 16 samples (the README's viewer command).
        view("view-720p-16spp", scene="terrain", w=1280, h=720, spp=16, bounces=8),
        # The two-level scene: 1,001 instances of 6 meshes, every transform new each frame.
        anim("anim-1000-720p", instances=1000, w=1280, h=720, spp=16, bounces=8),
        # Baking: four million incoherent rays from the surfaces, closest hits and then visibility.
        rays("rays-4M-surface", n=(1 << 22) + 1, origin="surface", query="both"),
        # A BVH over a two-million-triangle heightfield (the published build size).
        build("build-2M", grid=1005),
        # A mixed stream of small and middling jobs over four scenes.
        jobs("jobs-24", scenes=4, jobs=24, side=512),
    ]


def frame(name=None, scene="terrain", grid=242, w=512, h=512, spp=64, bounces=8, bvh=8, tri="woop", sort=0, filter="bh",
          full=0, tex=0, host=0):
    return named(name, kind="frame", scene=scene, grid=grid, w=w, h=h, spp=spp, bounces=bounces, bvh=bvh, tri=tri, sort=sort,
                 filter=filter, full=full, tex=tex, host=host)


def view(name=None, scene="terrain", grid=242, w=512, h=512, spp=1, bounces=8, bvh=8, tri="woop"):
    return named(name, kind="view", scene=scene, grid=grid, w=w, h=h, spp=spp, bounces=bounces, bvh=bvh, tri=tri, sort=0,
                 filter="bh", full=0, tex=0)


def anim(name=None, instances=1000, w=1280, h=720, spp=16, bounces=8):
    return named(name, kind="anim", instances=instances, w=w, h=h, spp=spp, bounces=bounces)


def rays(name=None, scene="terrain", grid=242, n=1 << 20, origin="surface", query="closest", bvh=8, tri="woop"):
    return named(name, kind="rays", scene=scene, grid=grid, n=n, origin=origin, query=query, bvh=bvh, tri=tri)


def build(name=None, grid=1005):
    return named(name, kind="build", grid=grid)


def jobs(name=None, scenes=4, jobs=24, side=512, full=0):
    return named(name, kind="jobs", scenes=scenes, jobs=jobs, side=side, full=full)


def named(name, **case):
    return dict(case, name=name) if name else case


def draw(rng):
    """A case of the listed ones' ranges: sizes over their logarithm, odd ones among them."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def size(lo, hi):
        w = log(lo, hi)
        return w, max(16, int(w * rng.choice((1.0, 0.5625, 0.75, rng.uniform(0.4, 1.3)))))

    kind = rng.choices(("frame", "view", "anim", "rays", "build", "jobs"), (45, 15, 10, 12, 10, 8))[0]
    if kind == "frame":
        w, h = size(96, 1280)
        full = rng.random() < 0.35
        spp = min(log(1, 256), max(1, (1280 * 720 * (64 if full else 192)) // (w * h)))
        bvh = rng.choices((8, 4, 2), (70, 10, 20))[0]
        return frame(scene=rng.choices(("terrain", "boxes"), (70, 30))[0], grid=log(40, 400), w=w, h=h, spp=spp,
                     bounces=rng.randint(2, 8), bvh=bvh, tri=rng.choices(("woop", "watertight", "mt"), (70, 20, 10))[0],
                     sort=2 if rng.random() < 0.25 else 0, filter=rng.choice(("bh", "box")), full=int(full),
                     tex=256 if full and rng.random() < 0.4 else 0, host=int(rng.random() < 0.3))
    if kind == "view":
        w, h = size(160, 1280)
        return view(scene=rng.choice(("terrain", "boxes")), grid=log(40, 400), w=w, h=h, spp=log(1, 16),
                    bounces=rng.randint(2, 8))
    if kind == "anim":
        w, h = size(160, 1280)
        return anim(instances=log(10, 2000), w=w, h=h, spp=log(1, 16), bounces=rng.randint(2, 8))
    if kind == "rays":
        return rays(scene=rng.choice(("terrain", "boxes")), grid=log(40, 400), n=log(1000, 1 << 22) | 1,
                    origin=rng.choice(("surface", "camera")), query=rng.choice(("closest", "any", "both")),
                    tri=rng.choice(("woop", "watertight")))
    if kind == "build":
        return build(grid=log(30, 1005))
    return jobs(scenes=rng.randint(2, 4), jobs=rng.randint(4, 24), side=log(64, 512), full=int(rng.random() < 0.3))


# ---------------------------------------------------------------------------------------------------------- preparing
class _Device:
    """a device buffer of the library as an array for torch.as_tensor (no copy); the tensor keeps this record, and with
    it the buffer's owner, alive"""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 2}


def scene_args(case, seed):
    """the pt options of a case's scene: the terrain, the materials and the maps are made from the seed"""
    a = ["--gen", case["scene"], "--gen_seed", str(1 + seed % 100003)] + LIGHTING
    if case["scene"] == "terrain":
        a += ["--gen_grid", str(case["grid"])]
    if case.get("full"):
        a += ["--gen_materials", str(1 + seed % 97), "--gen_env", "1024,512,2,%d" % (1 + seed % 89)]
        if case["tex"]:
            a += ["--gen_textures", str(case["tex"])]
    return a


def setup_of(case, seed):
    a = scene_args(case, seed) + ["--variant", "bvh%d" % case["bvh"], "--tri", case["tri"], "--seed", str(seed % (1 << 30))]
    if case["kind"] in ("frame", "view"):
        a += ["--width", str(case["w"]), "--height", str(case["h"]), "--batch", str(case["spp"]), "--spp", str(case["spp"]),
              "--bounces", str(case["bounces"]), "--sort", str(case["sort"]), "--filter", case["filter"]]
    else:
        a += ["--width", "64", "--height", "64", "--batch", "1", "--bounces", "1"]
    return cwp.Setup(a)


def query_rays(case, seed, setup, device):
    """n rays of 8 floats (origin, tmin, direction, tmax) on `device`: cosine-distributed directions from random points of the
    surfaces, or a pinhole camera above the scene; tmax is the scene's size"""
    g = torch.Generator().manual_seed(seed)
    n = case["n"]
    v = torch.from_numpy(setup.array(cwp.ARR_VERTICES))
    f = torch.from_numpy(setup.array(cwp.ARR_TRIANGLES).astype(np.int64))
    lo, hi = v.amin(0), v.amax(0)
    reach = float((hi - lo).norm())
    u = torch.rand((n, 4), generator=g)
    if case["origin"] == "surface":
        t = f[torch.randint(len(f), (n,), generator=g)]
        a, b, c = v[t[:, 0]], v[t[:, 1]], v[t[:, 2]]
        s = u[:, :1].sqrt()
        p = a * (1 - s) + b * (s * (1 - u[:, 1:2])) + c * (s * u[:, 1:2])
        nrm = torch.nn.functional.normalize(torch.linalg.cross(b - a, c - a), dim=1)
        nrm = torch.where(nrm[:, 2:] < 0, -nrm, nrm)
        z = 1 - 2 * u[:, 2:3]
        ph = 2 * math.pi * u[:, 3:4]
        r = (1 - z * z).clamp_min(0).sqrt()
        d = torch.nn.functional.normalize(nrm * 1.0001 + torch.cat([r * ph.cos(), r * ph.sin(), z], 1), dim=1)
        o = p + nrm * (1e-4 * reach)
    else:
        side = int(math.ceil(math.sqrt(n)))
        k = torch.arange(n)
        x, y = ((k % side) + u[:, 0]) / side - 0.5, ((k // side) + u[:, 1]) / side - 0.5
        eye = torch.tensor([0.5 * float(lo[0] + hi[0]), float(lo[1]) - 0.3, float(hi[2]) + 0.5])
        look = torch.nn.functional.normalize((lo + hi) * 0.5 - eye, dim=0)
        right = torch.nn.functional.normalize(torch.linalg.cross(look, torch.tensor([0.0, 0.0, 1.0])), dim=0)
        up = torch.linalg.cross(right, look)
        d = torch.nn.functional.normalize(look + x[:, None] * right + y[:, None] * up, dim=1)
        o = eye.expand(n, 3)
    out = torch.cat([o, torch.zeros(n, 1), d, torch.full((n, 1), reach)], 1).float().contiguous()
    return out.to(device)


def heightfield_boxes(grid, seed, device):
    """the triangle boxes (lo, hi: 4 floats each) of a noisy heightfield of 2 (grid - 1)^2 triangles"""
    g = torch.Generator(device=device).manual_seed(seed)
    xs = torch.linspace(0.0, 1.0, grid, device=device)
    z = 0.05 * torch.randn((grid, grid), generator=g, device=device)
    v = torch.stack([xs.expand(grid, grid), xs[:, None].expand(grid, grid), z], 2)
    a, b, c, d = v[:-1, :-1], v[:-1, 1:], v[1:, :-1], v[1:, 1:]
    t = torch.stack([torch.stack([a, b, d], 2), torch.stack([a, d, c], 2)], 2).reshape(-1, 3, 3)
    pad = torch.zeros((t.shape[0], 1), device=device)
    return torch.cat([t.amin(1), pad], 1).contiguous(), torch.cat([t.amax(1), pad], 1).contiguous()


def job_list(case, seed):
    r = np.random.default_rng((case["scenes"], case["jobs"], case["side"]))   # the stream's mix is the case's, its noise the seed's
    sides = [s for s in (case["side"] // 4, case["side"] // 2, case["side"]) if s >= 16]
    return [(int(r.integers(case["scenes"])), int(r.choice(sides)), int(r.choice(sides)), int(r.choice((4, 16, 64))), 6,
             (seed * 1000 + k) % (1 << 30)) for k in range(case["jobs"])]


class State:
    pass


def prepare(case, seed):
    s = State()
    s.case = case
    kind = case["kind"]
    if kind in ("frame", "view"):
        s.setup = setup_of(case, seed)
        s.r = cwp.Renderer(s.setup)
        s.image = torch.as_tensor(_Device(s.r, s.r.accum_device(), (case["h"], case["w"], 4)), device="cuda")
        if kind == "view":
            s.params = s.setup.params()
            rng = np.random.default_rng(seed)
            for k in range(3):
                s.params.pos[k] += float(rng.uniform(-0.02, 0.02))
            s.pixels = cwp.DeviceArray(case["w"] * case["h"] * 4)
    elif kind == "anim":
        s.setup = cwp.Setup(["--gen", "instances", "--gen_instances", str(case["instances"]), "--gen_seed", str(1 + seed % 100003),
                             "--width", str(case["w"]), "--height", str(case["h"]), "--batch", str(case["spp"]),
                             "--spp", str(case["spp"]), "--bounces", str(case["bounces"]), "--filter", "box",
                             "--morton_bits", "30", "--seed", str(seed % (1 << 30))] + LIGHTING)
        s.r = cwp.Renderer(s.setup)
        s.frame = seed % 50
        s.image = torch.as_tensor(_Device(s.r, s.r.accum_device(), (case["h"], case["w"], 4)), device="cuda")
    elif kind == "rays":
        s.setup = setup_of(case, seed)
        s.r = cwp.Renderer(s.setup)
        s.rays = query_rays(case, seed, s.setup, "cuda")
        s.hits = torch.empty((case["n"], 4), dtype=torch.float32, device="cuda")
        s.any = torch.empty((case["n"], 4), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
    elif kind == "build":
        s.lo, s.hi = heightfield_boxes(case["grid"], seed, "cuda")
        s.n = len(s.lo)
        s.nodes = torch.zeros((s.n, 20), dtype=torch.int32, device="cuda")   # the tree fills the first rows
        s.prims = torch.empty(s.n, dtype=torch.int32, device="cuda")
        s.builder = Builder(s.n)
        torch.cuda.synchronize()
    else:
        s.server = cwp.Server(variant=8, bounces=6, full=case["full"], max_paths=1 << 24)
        for k in range(case["scenes"]):
            a = ["--gen", "terrain", "--gen_grid", str(60 + 80 * k), "--gen_seed", str(1 + (seed + k) % 100003), "--width", "64",
                 "--height", "64", "--bounces", "6", "--filter", "box", "--gen_boxes", "64"] + LIGHTING
            if case["full"]:
                a += ["--gen_materials", str(1 + k), "--gen_env", "512,256,2,%d" % (1 + k)]
            s.server.add_scene(cwp.Setup(a))
        s.jobs = job_list(case, seed)
        for j in s.jobs:
            s.server.submit(*j[:5], seed=j[5])
        s.server.preload()
    return s


class Builder:
    """a builder handle of the C interface, with its scratch memory"""

    def __init__(self, capacity):
        self.h = cwp.ctypes.c_void_p()
        cwp._check(cwp.lib().cwp_hploc_create(capacity, cwp.ctypes.byref(self.h)))

    def __del__(self):
        if self.h:
            cwp.lib().cwp_hploc_destroy(self.h)
            self.h = None


# ------------------------------------------------------------------------------------------------------------ running
def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "frame":
        s.r.render(case["spp"])
        return s.r.accum() if case["host"] else s.image
    if kind == "view":
        s.r.set_params(s.params)
        s.r.render(case["spp"])
        return s.r.display(case["spp"], 0.0, "aces", out=s.pixels)
    if kind == "anim":
        s.r.set_frame(s.frame)
        s.r.render(case["spp"])
        return s.image
    if kind == "rays":
        out = {}
        for any_hit, hits in ((0, s.hits), (1, s.any)):
            if case["query"] in (("closest", "both"), ("any", "both"))[any_hit]:
                s.r.trace_ptr(s.rays.data_ptr(), case["n"], any_hit, hits.data_ptr())
                if any_hit:   # which triangle an any-hit query names is the traversal's choice
                    out["seen"] = hits.view(torch.int32)[:, 3] < 0
                else:
                    out["hit"], out["triangle"] = hits[:, :3], hits.view(torch.int32)[:, 3]
        return out
    if kind == "build":
        L, c = cwp.lib(), cwp.ctypes
        root, nodes, count, depth = c.c_int(), c.c_void_p(), c.c_int(), c.c_int()
        cwp._check(L.cwp_hploc_build(s.builder.h, s.lo.data_ptr(), s.hi.data_ptr(), s.n, None, c.byref(root)))
        cwp._check(L.cwp_hploc_nodes(s.builder.h, c.byref(nodes)))
        cwp._check(L.cwp_cwbvh_from_hploc(nodes, s.n, s.nodes.data_ptr(), c.byref(count), s.prims.data_ptr(), c.byref(depth), None))
        return {"nodes": s.nodes, "count": count.value, "prims": s.prims, "depth": depth.value}
    s.server.clear_jobs()
    ids = [s.server.submit(*j[:5], seed=j[5]) for j in s.jobs]
    s.server.run()
    return [s.server.image(i) for i in ids]


# ------------------------------------------------------------------------------------------------------------ what it needs
RAYS_PER_PATH = 4.2        # closest and shadow rays of a path on these scenes (the benchmark's frames: 4.1 to 5.0)
FLOPS_PER_RAY = 1400.0     # about 8 wide-node visits of 8 boxes at 20 operations, and 3 triangles at 40


def work(case):
    kind = case["kind"]
    tris = {"boxes": 12290, "terrain": 2 * (case.get("grid", 2) - 1) ** 2 + 2400}.get(case.get("scene"), 0)
    scene = tris * (48 + 16 + 80 / 4.5)
    if kind in ("frame", "view", "anim"):
        if kind == "anim":
            scene = 300e3 * 82 + case["instances"] * 112
        paths = case["w"] * case["h"] * case["spp"]
        return {"bytes": scene + case["w"] * case["h"] * (20 if kind == "view" else 16), "flops": paths * RAYS_PER_PATH * FLOPS_PER_RAY}
    if kind == "rays":
        q = 2 if case["query"] == "both" else 1
        return {"bytes": scene + case["n"] * q * 48, "flops": case["n"] * q * FLOPS_PER_RAY}
    if kind == "build":
        n = 2 * (case["grid"] - 1) ** 2
        return {"bytes": n * (32 + 4 + 80 / 4.5), "flops": n * 600.0}
    each = case["side"] ** 2 * (1 / 16 + 1 / 4 + 1) / 3 * 28   # the mean job: sides and sample counts uniform
    return {"bytes": case["jobs"] * each / 28 * 16, "flops": case["jobs"] * each * RAYS_PER_PATH * FLOPS_PER_RAY}


def tolerance(case):
    kind = case["kind"]
    if kind in ("frame", "anim", "jobs"):
        # A change of rounding sends a path past an edge now and then: single pixels change, the rest to 32-bit rounding.
        # Against 64 bits a small frame is 1.1e-3 off.
        return {"rel": 5e-3, "max": 0.9}
    if kind == "view":
        return {"differ": 2e-3}
    if kind == "rays":
        return {"rel": 1e-4, "max": 0.9, "differ": 1e-4}
    return "exact"


# ------------------------------------------------------------------------------------------------------------ 64 bits
PAIRS = 4e10   # ray-triangle pairs that fit the time


class Brute:
    """closest hits of rays against every triangle, in 64 bits: each triangle is the affine map that takes it to the unit
    triangle, so a ray's plane distance and barycentric coordinates are products of small matrices"""

    def __init__(self, setup):
        v = torch.from_numpy(setup.array(cwp.ARR_VERTICES)).double().cuda()
        f = torch.from_numpy(setup.array(cwp.ARR_TRIANGLES).astype(np.int64)).cuda()
        a, e1, e2 = v[f[:, 0]], v[f[:, 1]] - v[f[:, 0]], v[f[:, 2]] - v[f[:, 0]]
        nrm = torch.linalg.cross(e1, e2)
        fine = (nrm * nrm).sum(1) > 0
        m = torch.stack([e1, e2, nrm], 2)
        m[~fine] = torch.eye(3, dtype=torch.float64, device="cuda")
        inv = torch.linalg.inv(m)
        w = -(inv @ a[:, :, None])[:, :, 0]
        w[~fine, 2] = float("nan")
        self.rows = [inv[:, k].T.contiguous() for k in range(3)]   # 3 x triangles
        self.w = [w[:, k].contiguous() for k in range(3)]
        self.normal = torch.nn.functional.normalize(nrm, dim=1)
        self.n = len(f)

    def closest(self, o, d, tmin, tmax):
        t, u, v = tmax.clone(), torch.zeros_like(tmax), torch.zeros_like(tmax)
        tri = torch.full((len(o),), -1, dtype=torch.int64, device="cuda")
        step = max(1, (1 << 26) // self.n)
        for i in range(0, len(o), step):
            oo, dd = o[i:i + step], d[i:i + step]
            tt = -(torch.mm(oo, self.rows[2]) + self.w[2]) / torch.mm(dd, self.rows[2])
            uu = torch.mm(oo, self.rows[0]) + self.w[0] + tt * torch.mm(dd, self.rows[0])
            vv = torch.mm(oo, self.rows[1]) + self.w[1] + tt * torch.mm(dd, self.rows[1])
            ok = (tt > tmin) & (tt < tmax[i:i + step, None]) & (uu >= 0) & (vv >= 0) & (uu + vv <= 1)
            best, k = torch.where(ok, tt, torch.inf).min(1)
            hit = torch.isfinite(best)
            g = k[:, None]
            t[i:i + step] = torch.where(hit, best, t[i:i + step])
            u[i:i + step] = torch.where(hit, uu.gather(1, g)[:, 0], 0.0)
            v[i:i + step] = torch.where(hit, vv.gather(1, g)[:, 0], 0.0)
            tri[i:i + step] = torch.where(hit, k, -1)
        return t, u, v, tri


def hash32(x):
    x = x & 0xffffffff
    x = ((x ^ (x >> 16)) * 0x7feb352d) & 0xffffffff
    x = ((x ^ (x >> 15)) * 0x846ca68b) & 0xffffffff
    return x ^ (x >> 16)


def uniform(pix, smp, depth, dim, seed):
    inner = hash32(torch.tensor(((depth * 8 + dim) * 0xC2B2AE3D ^ seed) & 0xffffffff, device="cuda"))
    mid = hash32(((smp * 0x85EBCA77) & 0xffffffff) ^ inner)
    return (hash32(((pix * 0x9E3779B1) & 0xffffffff) ^ mid) >> 8).double() / 16777216.0


def around(axis, x, y, z):
    """x, y, z in the orthonormal basis of Duff et al. (2017) around unit vectors `axis`"""
    s = torch.where(axis[:, 2] >= 0, 1.0, -1.0)
    a = -1.0 / (s + axis[:, 2])
    c = axis[:, 0] * axis[:, 1] * a
    t = torch.stack([1 + s * axis[:, 0] ** 2 * a, s * c, -s * axis[:, 0]], 1)
    b = torch.stack([c, s + axis[:, 1] ** 2 * a, -axis[:, 1]], 1)
    return torch.nn.functional.normalize(t * x[:, None] + b * y[:, None] + axis * z[:, None], dim=1)


def path_trace(case, setup):
    """the diffuse path tracer in 64 bits: sun and sky, one shadow ray and one cosine-distributed bounce per hit"""
    p, K = setup.params(), case["spp"]
    brute = Brute(setup)
    albedo = float(setup.array(cwp.ARR_ALBEDO)[0, 0])
    i = torch.arange(p.w * p.h * K, device="cuda")
    pix, smp, seed = i // K, i % K, p.seed
    vec = lambda a: torch.tensor(list(a), dtype=torch.float64, device="cuda")   # noqa: E731
    u0, u1 = uniform(pix, smp, 0, 0, seed), uniform(pix, smp, 0, 1, seed)
    if p.filter_bh:
        tab = vec(p.ftab)

        def jitter(u):
            k = (u * 64).long().clamp_max(63)
            return tab[k] + (u * 64 - k) * (tab[k + 1] - tab[k])
        u0, u1 = jitter(u0), jitter(u1)
    else:
        u0, u1 = u0 - 0.5, u1 - 0.5
    x, y = (pix % p.w + 0.5 + u0 - p.px) / p.fx, -(pix // p.w + 0.5 + u1 - p.py) / p.fy
    d = torch.nn.functional.normalize(vec(p.ax) * x[:, None] + vec(p.ay) * y[:, None] - vec(p.az), dim=1)
    o = vec(p.pos).expand_as(d)
    L = torch.zeros(len(i), 3, dtype=torch.float64, device="cuda")
    T, tmin, far = 1.0, float(p.near_t), 1e30
    for depth in range(p.max_bounce + 2):
        t, _, _, tri = brute.closest(o, d, tmin, torch.full((len(i),), far, dtype=torch.float64, device="cuda"))
        miss = tri < 0
        L[i[miss]] += T * vec(p.sky)
        if depth > p.max_bounce:
            break
        i, pix, smp, o, d, t, tri = (q[~miss] for q in (i, pix, smp, o, d, t, tri))
        n = brute.normal[tri]
        n = torch.where((n * d).sum(1, keepdim=True) > 0, -n, n)
        po = o + d * t[:, None] + n * p.eps
        u2, u3 = uniform(pix, smp, depth + 1, 2, seed), uniform(pix, smp, depth + 1, 3, seed)
        cz = 1 - u2 * (1 - p.sun_cos)
        sz = (1 - cz * cz).clamp_min(0).sqrt()
        to = around(vec(p.sun_to).expand_as(n), sz * torch.cos(2 * math.pi * u3), sz * torch.sin(2 * math.pi * u3), cz)
        cl = (n * to).sum(1)
        k = cl > 0
        _, _, _, blocked = brute.closest(po[k], to[k], 0.0, torch.full((int(k.sum()),), far, dtype=torch.float64, device="cuda"))
        L[i[k]] += torch.where(blocked < 0, T * albedo * cl[k] / math.pi, 0.0)[:, None] * vec(p.sun_e)
        u0, u1 = uniform(pix, smp, depth + 1, 0, seed), uniform(pix, smp, depth + 1, 1, seed)
        r = u0.sqrt()
        d = around(n, r * torch.cos(2 * math.pi * u1), r * torch.sin(2 * math.pi * u1), (1 - u0).sqrt())
        k = (d * n).sum(1) > 0
        i, pix, smp, o, d = (q[k] for q in (i, pix, smp, po, d))
        T, tmin = T * albedo, 0.0
        if not len(i):
            break
    image = torch.zeros(p.h, p.w, 4, dtype=torch.float64, device="cuda")
    image[..., :3] = L.view(p.h, p.w, K, 3).sum(2)
    return image


def exact(case, seed):
    kind = case["kind"]
    tris = 12290 if case.get("scene") == "boxes" else 2 * (case.get("grid", 2) - 1) ** 2 + 2400
    if kind == "rays" and case["query"] != "any" and case["n"] * tris <= PAIRS:
        setup = setup_of(case, seed)
        q = query_rays(case, seed, setup, "cuda").double()
        t, u, v, _ = Brute(setup).closest(q[:, :3].contiguous(), q[:, 4:7].contiguous(), 0.0, q[:, 7].contiguous())
        return dict({"hit": torch.stack([t, u, v], 1), "triangle": None}, **({"seen": None} if case["query"] == "both" else {}))
    if kind == "frame" and not case["full"] and case["w"] * case["h"] * case["spp"] * 2 * (case["bounces"] + 2) * tris <= PAIRS:
        return path_trace(case, setup_of(case, seed))
    return None   # path tracing at these sizes takes minutes in 64 bits; boxes, bytes and orders are compared exactly
