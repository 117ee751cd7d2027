"""GPU parity tests of two-level scenes (TLAS over instances rebuilt by the GPU H-PLOC builder each frame, as a BVH2 or,
over BVH8 BLASes, collapsed on the GPU into a compressed BVH8; BLAS per mesh) against the oracle's two-level traversal
and renderer (BVH2 TLAS, as the reference's travInst), and against the flattened scene."""
import math

import numpy as np
import pytest

import cwp
import pyoracle as po

pytestmark = pytest.mark.gpu

ARGS = ["--gen", "instances", "--gen_small", "1", "--gen_instances", "120", "--width", "96", "--height", "64"]


def psnr(a, b):
    def srgb(x):
        x = np.clip(x, 0, 1)
        return np.where(x <= 0.0031308, 12.92 * x, 1.055 * np.power(x, 1 / 2.4) - 0.055)
    mse = float(np.mean((srgb(a.astype(np.float64)) - srgb(b.astype(np.float64))) ** 2))
    return 99.0 if mse == 0 else 10 * math.log10(1.0 / mse)


def oracle_scene(s, frame, tri_test=1):
    v = s.info["variant"]
    sc = po.Scene(v, tri_test, s.array(cwp.ARR_NODES), s.array(cwp.ARR_WOOP), s.array(cwp.ARR_CORNERS),
                  s.array(cwp.ARR_ALBEDO))
    sc.set_instances(s.instances(frame), s.array(cwp.ARR_MESH_BOXES))
    return sc


def scene_rays(s, n, seed):
    p = s.params()
    rng = np.random.default_rng(seed)
    out = []
    for k in range(n):
        o, d = po.camera_ray(p, int(rng.integers(p.w * p.h)), int(rng.integers(256)))
        out.append(np.concatenate([o, [0.0], d, [1e30]]))
    cam = np.array(out, np.float32)
    o = rng.uniform([-12, -12, -1], [12, 12, 3], (n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32); d /= np.linalg.norm(d, axis=1, keepdims=True)
    rnd = np.concatenate([o, np.zeros((n, 1)), d, np.full((n, 1), 1e30)], 1).astype(np.float32)
    return np.concatenate([cam, rnd])


@pytest.mark.parametrize("variant,tri,tlas", [("bvh8", "woop", "bvh8"), ("bvh8", "woop", "bvh2"),
                                              ("bvh8", "watertight", "bvh8"), ("bvh2", "watertight", "bvh2"),
                                              ("bvh4", "mt", "bvh2")])
def test_two_level_trace_matches_oracle(variant, tri, tlas):
    print("case", variant, tri, tlas, flush=True)
    s = cwp.Setup(ARGS + ["--variant", variant, "--tri", tri, "--tlas", tlas])
    r = cwp.Renderer(s)
    sc = oracle_scene(s, 0, {"mt": 0, "woop": 1, "watertight": 2}[tri])
    rays = scene_rays(s, 20000, 3)
    g, gi = r.trace_inst(rays)
    o, oi = sc.trace_inst(rays)
    gt, ot = g[:, 3].view(np.int32), o[:, 3].view(np.int32)
    assert (ot >= 0).mean() > 0.3
    agree = ((gt == ot) & (gi == oi)).mean()
    assert agree >= 0.9999, agree
    both = (gt == ot) & (ot >= 0)
    assert (np.abs(g[both, 0] - o[both, 0]) / np.abs(o[both, 0])).max() <= 1e-5
    ga, _ = r.trace_inst(rays, any_hit=True)
    assert ((ga[:, 3].view(np.int32) >= 0) == (gt >= 0)).mean() >= 0.9999


def test_tlas_rebuilt_per_frame_matches_oracle():
    s = cwp.Setup(ARGS)
    r = cwp.Renderer(s)
    rays = scene_rays(s, 8000, 5)
    for f in (1, 7, 59):
        ms = r.set_frame(f)
        assert ms > 0
        g, gi = r.trace_inst(rays)
        o, oi = oracle_scene(s, f).trace_inst(rays)
        assert ((g[:, 3].view(np.int32) == o[:, 3].view(np.int32)) & (gi == oi)).mean() >= 0.9999
    with pytest.raises(cwp.CwpError, match="BLAS root"):
        bad = s.instances(0)
        bad.view(np.int32)[3, 24] += 1
        r.set_instances(bad)


@pytest.mark.parametrize("morton,tlas", [(0, "bvh8"), (30, "bvh8"), (30, "bvh2")])
def test_full_size_two_level_scene_matches_oracle(morton, tlas):
    """The two-level configuration at full size: 5 meshes of 1.3k-200k triangles and a ground, 1,001 instances with
    their transforms redrawn per frame, the TLAS rebuilt on the GPU with adaptive or 30-bit Morton keys (as a BVH2 or
    a compressed BVH8); closest-hit triangle and instance ids of 16,000 rays against the oracle's two-level traversal
    at 3 frames."""
    print("case full-size two-level morton=%d tlas=%s" % (morton, tlas), flush=True)
    s = cwp.Setup(["--gen", "instances", "--width", "96", "--height", "64", "--morton_bits", str(morton), "--tlas", tlas])
    assert s.info["num_instances"] >= 1000
    r = cwp.Renderer(s)
    rays = scene_rays(s, 8000, 11)
    for f in (0, 17, 59):
        assert r.set_frame(f) > 0
        g, gi = r.trace_inst(rays)
        o, oi = oracle_scene(s, f).trace_inst(rays)
        gt, ot = g[:, 3].view(np.int32), o[:, 3].view(np.int32)
        assert (ot >= 0).mean() > 0.3
        agree = ((gt == ot) & (gi == oi)).mean()
        assert agree >= 0.9999, (f, agree)
        both = (gt == ot) & (ot >= 0)
        assert (np.abs(g[both, 0] - o[both, 0]) / np.abs(o[both, 0])).max() <= 1e-5
    r.close()


def test_two_level_render_matches_oracle_and_flattened():
    spp, batch, bounces = 8, 8, 4
    extra = ["--batch", str(batch), "--bounces", str(bounces), "--spp", str(spp)]
    s = cwp.Setup(ARGS + extra)
    r = cwp.Renderer(s)
    st = r.render(spp)
    img = r.accum()[..., :3] / spp
    j = r.frame_json(st)
    assert j["instances"] == s.info["num_instances"] and j["tlas_ms"] > 0 and j["tlas"] == "bvh8"
    acc, ost = oracle_scene(s, 0).render(s.params(), spp, batch=batch, bounces=bounces)
    assert psnr(img, acc[..., :3] / spp) >= 50.0
    assert st["rays_closest"] == pytest.approx(ost[0], rel=1e-3)
    # the same geometry flattened into world space: equal up to transform rounding
    f = cwp.Setup(ARGS + extra + ["--flatten", "1"])
    rf = cwp.Renderer(f)
    rf.render(spp)
    assert psnr(img, rf.accum()[..., :3] / spp) >= 45.0
    # a BVH2 TLAS finds the same closest hits (only exact ties between instances may resolve differently)
    b = cwp.Renderer(cwp.Setup(ARGS + extra + ["--tlas", "bvh2"]))
    st2 = b.render(spp)
    assert b.frame_json(st2)["tlas"] == "bvh2"
    assert psnr(img, b.accum()[..., :3] / spp) >= 60.0
    assert st2["rays_closest"] == pytest.approx(st["rays_closest"], rel=1e-4)


@pytest.mark.parametrize("count", [1, 2, 3, 9])
def test_wide_tlas_over_few_instances(count):
    """Compressed BVH8 TLAS over 1-9 instances (a single leaf as the root, a root with a few leaf slots): trace ids
    against the oracle"""
    print("case wide TLAS over %d instances" % count, flush=True)
    s = cwp.Setup(ARGS)
    r = cwp.Renderer(s)
    inst = s.instances(0)[:count].copy()
    r.set_instances(inst)
    rays = scene_rays(s, 4000, 13)
    g, gi = r.trace_inst(rays)
    sc = po.Scene(s.info["variant"], 1, s.array(cwp.ARR_NODES), s.array(cwp.ARR_WOOP), s.array(cwp.ARR_CORNERS),
                  s.array(cwp.ARR_ALBEDO))
    sc.set_instances(inst, s.array(cwp.ARR_MESH_BOXES))
    o, oi = sc.trace_inst(rays)
    gt, ot = g[:, 3].view(np.int32), o[:, 3].view(np.int32)
    assert (ot >= 0).any()
    assert ((gt == ot) & (gi == oi)).mean() >= 0.9999
    r.close()


@pytest.mark.parametrize("tri,stack,tail,count", [("woop", 8, 0, 30), ("woop", 8, 2, 30), ("woop", 32, 64, 9),
                                                  ("watertight", 16, 12, 64), ("mt", 8, 12, 2)])
def test_overlapping_instances(tri, stack, tail, count):
    """Instances that all overlap, so that TLAS leaves name several at once, their rest waits on the stack while a BLAS is
    traversed, and waves hand such traversals off: triangle and instance ids of closest hits against the oracle, any
    hits, and the image without hand-off, bit for bit (a ray's visiting order depends on neither)."""
    print("case overlapping", tri, stack, tail, count, flush=True)
    args = ARGS + ["--tri", tri, "--stack", str(stack), "--batch", "4", "--bounces", "3"]
    s = cwp.Setup(args + ["--tail", str(tail)])
    inst = s.instances(0)[:count].copy()
    fwd, inv = inst[:, 12:24].reshape(-1, 3, 4), inst[:, :12].reshape(-1, 3, 4)
    fwd[:, :, 3] = np.random.default_rng(count).uniform(-0.3, 0.3, (count, 3))   # all around the origin
    inv[:, :, 3] = -np.einsum("nij,nj->ni", inv[:, :, :3].astype(np.float64), fwd[:, :, 3].astype(np.float64))
    r = cwp.Renderer(s)
    r.set_instances(inst)
    sc = po.Scene(s.info["variant"], {"mt": 0, "woop": 1, "watertight": 2}[tri], s.array(cwp.ARR_NODES), s.array(cwp.ARR_WOOP),
                  s.array(cwp.ARR_CORNERS), s.array(cwp.ARR_ALBEDO))
    sc.set_instances(inst, s.array(cwp.ARR_MESH_BOXES))
    rays = scene_rays(s, 4000, 17)
    g, gi = r.trace_inst(rays)
    o, oi = sc.trace_inst(rays)
    gt, ot = g[:, 3].view(np.int32), o[:, 3].view(np.int32)
    assert (ot >= 0).mean() > 0.02
    assert ((gt == ot) & (gi == oi)).mean() >= 0.999
    assert np.array_equal(r.trace_inst(rays, any_hit=True)[0][:, 3].view(np.int32) >= 0, gt >= 0)
    r.render(4)
    plain = cwp.Renderer(cwp.Setup(args + ["--tail", "0", "--persistent", "0"]))
    plain.set_instances(inst)
    plain.render(4)
    np.testing.assert_array_equal(r.accum(), plain.accum())


@pytest.mark.parametrize("tri,tlas,n", [("woop", "bvh8", 16384), ("woop", "bvh8", 16385), ("watertight", "bvh8", 60001),
                                        ("mt", "bvh8", 40000), ("woop", "bvh2", 40001)])
def test_two_level_queries_of_more_rays_than_lanes(tri, tlas, n):
    """With one workgroup per CU (16,384 lanes on 256 CUs) idle lanes take new rays beside lanes inside a BLAS (BVH8 TLAS;
    a BVH2 TLAS goes round by round): hits and instance ids bit for bit those of the full grid, which has a lane for
    every ray here, and the oracle's on all but grazing rays."""
    print("case", tri, tlas, n, flush=True)
    args = ARGS + ["--tri", tri, "--tlas", tlas]
    s = cwp.Setup(args)
    few, full = (cwp.Renderer(cwp.Setup(args + ["--blocks_per_cu", b])) for b in ("1", "0"))
    few.set_frame(0)
    full.set_frame(0)
    rng = np.random.default_rng(n)
    d = rng.normal(size=(n, 3))
    d[:n // 3] = np.abs(d[:n // 3]) * [1, 1, -1]   # like rays first: the waves' first chunks are traced whole
    rays = np.concatenate([rng.uniform([-12, -12, -1], [12, 12, 3], (n, 3)), np.zeros((n, 1)),
                           d / np.linalg.norm(d, axis=1, keepdims=True),
                           np.where(rng.random((n, 1)) < 0.3, rng.uniform(1, 10, (n, 1)), 1e30)], 1).astype(np.float32)
    (g, gi), (f, fi) = few.trace_inst(rays), full.trace_inst(rays)
    np.testing.assert_array_equal(g.view(np.uint32), f.view(np.uint32))
    np.testing.assert_array_equal(gi, fi)
    hit = g[:, 3].view(np.int32) >= 0
    assert 0.2 < hit.mean() < 0.95 and np.array_equal(gi >= 0, hit)
    a, ai = few.trace_inst(rays, any_hit=True)
    np.testing.assert_array_equal(a[:, 3].view(np.int32) >= 0, hit)
    np.testing.assert_array_equal(ai >= 0, hit)
    o, oi = oracle_scene(s, 0, {"mt": 0, "woop": 1, "watertight": 2}[tri]).trace_inst(rays)
    assert ((g[:, 3].view(np.int32) == o[:, 3].view(np.int32)) & (gi == oi)).mean() >= 0.999


@pytest.mark.parametrize("full", [False, True])
def test_two_level_queues_equal_whole_paths(full):
    """The queue kernels of two-level scenes, with one workgroup per CU (the counters hand most chunks out, to other
    partitions' waves too) and the full grid, against whole paths in one launch: images and ray counts bit for bit, on two
    frames. A frame of the full integrator with more paths than whole-path launches take uses them by itself."""
    print("case two-level queues", full, flush=True)
    extra = ["--gen_materials", "2", "--gen_env", "64,32,1.5,2"] if full else []
    keys = ("rays_closest", "rays_shadow", "rays_miss", "rays_cont", "shadow_unoccluded", "camera_miss")

    def frames(args, spp, n=2):
        r = cwp.Renderer(cwp.Setup(args))
        out = []
        for f in range(n):
            r.set_frame(f)
            st = r.render(spp, f * spp)
            out.append((r.accum(), [st[k] for k in keys], st["shadow_launches"]))
        r.close()
        return out

    args = ARGS[:-4] + ["--width", "211", "--height", "157", "--batch", "8", "--bounces", "4", "--graph", "0"] + extra
    whole = frames(args, 8)
    assert whole[0][2] == 0
    for o in (["--persistent", "0"], ["--persistent", "0", "--blocks_per_cu", "1"]):
        for (a, n, launches), (b, m, _) in zip(frames(args + o, 8), whole):
            assert launches == 6
            np.testing.assert_array_equal(a, b)
            assert n == m
    if full:
        args = ARGS[:-4] + ["--width", "1001", "--height", "701", "--batch", "3", "--bounces", "2", "--graph", "0"] + extra
        (a, n, launches), = frames(args, 3, 1)
        (b, m, _), = frames(args + ["--tail", "12"], 3, 1)
        assert launches == 4
        np.testing.assert_array_equal(a, b)
        assert n == m


FULL = ARGS + ["--gen_materials", "2", "--gen_env", "64,32,1.5,2", "--bounces", "3"]


def full_oracle(s, frame):
    i = s.info
    sc = po.Scene(i["variant"], i["tri_test"], s.array(cwp.ARR_NODES), s.array(cwp.ARR_WOOP), s.array(cwp.ARR_CORNERS),
                  s.array(cwp.ARR_ALBEDO))
    sc.set_instances(s.instances(frame), s.array(cwp.ARR_MESH_BOXES))
    sc.set_full(s.array(cwp.ARR_MATERIALS), s.array(cwp.ARR_ORDER), i["sun_on"], i["light_mode"], i["rr"], i["rr_depth"],
                i["gd_energy"], i["env_uniform"], s.array(cwp.ARR_ENV_TEX), i["env_w"], i["env_h"], i["env_rot_deg"])
    sc.set_inst_emitters(s.array(cwp.ARR_MESH_TRIS), s.array(cwp.ARR_ORDER))
    return sc


@pytest.mark.parametrize("variant", ["bvh8", "bvh2"])
def test_two_level_full_integrator_matches_oracle(variant):
    """materials, per-frame world emitters and an environment on a two-level scene: >= 50 dB against the oracle for
    two frames (TLAS and emitters rebuilt), counters within 1 %"""
    print("case", variant, flush=True)
    s = cwp.Setup(FULL + ["--variant", variant, "--batch", "16", "--spp", "16"])
    assert s.info["full"] == 1 and s.info["num_emitters"] > 0
    r = cwp.Renderer(s)
    for f in (0, 9):
        r.set_frame(f)
        st = r.render(16)
        img = r.accum()[..., :3] / 16
        acc, ost = full_oracle(s, f).render(s.params(), 16, batch=16, bounces=3)
        assert psnr(img, acc[..., :3] / 16) >= 50.0, (variant, f)
        assert st["rays_closest"] == pytest.approx(ost[0], rel=1e-2)
        assert st["rays_shadow"] == pytest.approx(ost[1], rel=1e-2)


def test_two_level_full_requires_the_frame_emitters():
    s = cwp.Setup(FULL + ["--batch", "4", "--spp", "4"])
    r = cwp.Renderer(s)
    em, cdf, mlp = s.emitters(0)
    bad = em.copy()
    bad[0, 1, 3] = np.array([99], np.int32).view(np.float32)[0]   # material id out of range
    with pytest.raises(cwp.CwpError, match="material id"):
        r.set_emitters(bad, cdf, mlp)
    with pytest.raises(cwp.CwpError, match="instanced emitters"):
        r.set_emitters(em[:-1], cdf[:-1], mlp)
    r.set_emitters(em, cdf, mlp)
    r.render(4)
