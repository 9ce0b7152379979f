"""The work this library is timed on, through its public entry points.

Each case is one pass of something a program does with the library: a viewer's frame, a rendered image,
an acceleration structure rebuilt for moved shapes, ray queries, a batch of scenes, served requests.
Sizes come from the benchmark workloads (Cornell spheres 256x256, the 65,538-shape soup at 512x512, the
327,692-shape icosphere at 1024x768, many scenes of 10^3..10^6 triangles, request streams) and from the
tests (ragged frames, trees of a few hundred shapes), with odd sizes among them.

Kinds
  frame    one image of `spp` samples over a prepared tree (LBVH, restructured LBVH, SAH or mean-split KD,
           or none), from fixed per-pixel seeds
  viewer   one progressive 1-spp pass: the running mean and the seeds carry over from pass to pass
  animate  the scene's LBVH rebuilt (and restructured) from its shapes, then one image
  build    an LBVH rebuilt from device-resident shapes; its exported trees and sorted order
  batch    many scenes rebuilt in one batched build, then one image of each in one batched render
  serve    requests submitted to a render server, ticked to completion, results copied to the host
  drawframe  one RadianceGPU call with the reference's argument list over the caller's own BVH / KD arrays
  queries  closest-hit and any-hit queries of arbitrary rays
"""
from __future__ import annotations

import math

import numpy as np
import torch

import ptgpu_pc_amd as pt
from ptgpu_pc_amd import lib, scenes
from ptgpu_pc_amd.layout import SHAPE_DTYPE

_CTX = None


def _ctx():
    global _CTX
    if _CTX is None:
        torch.cuda.init()
        _CTX = pt.Context(0)
    return _CTX


def listed():
    return [
        # the reference's built-in Cornell spheres without an acceleration structure (its default scene)
        {"name": "cornell_frame", "kind": "frame", "scene": "cornell", "n": 9, "accel": "none", "treelet": 0, "w": 256,
         "h": 256, "spp": 4, "depth": 5},
        # an interactive viewer on a small model (the reference's own scene has 326 shapes): smallest call
        {"name": "viewer_small", "kind": "viewer", "scene": "mesh", "n": 332, "accel": "bvh", "treelet": 0, "w": 97,
         "h": 61, "spp": 1, "depth": 6},
        # the triangle soup of the headline benchmark, one image
        {"name": "soup_frame", "kind": "frame", "scene": "soup", "n": 65538, "accel": "bvh", "treelet": 0, "w": 512,
         "h": 512, "spp": 8, "depth": 5},
        # the displaced icosphere in a closed box, restructured tree, a final-quality image: the largest render
        {"name": "mesh_frame", "kind": "frame", "scene": "mesh", "n": 327692, "accel": "bvh", "treelet": 7, "w": 1024,
         "h": 768, "spp": 16, "depth": 6},
        # the KD-tree mode at the reference's default window size
        {"name": "kd_frame", "kind": "frame", "scene": "mesh", "n": 20492, "accel": "kd_sah", "treelet": 0, "w": 640,
         "h": 480, "spp": 4, "depth": 6},
        # an animated scene: tree rebuilt and restructured for every (ragged) frame
        {"name": "animate", "kind": "animate", "scene": "soup", "n": 16001, "accel": "bvh", "treelet": 5, "w": 641,
         "h": 359, "spp": 2, "depth": 5},
        # a small scene's rebuild: launches and their gaps
        {"name": "build_small", "kind": "build", "scene": "soup", "n": 1003, "accel": "bvh"},
        # a large scene's rebuild: memory traffic
        {"name": "build_large", "kind": "build", "scene": "soup", "n": 4000003, "accel": "bvh"},
        # a set of scenes of uneven size, all rebuilt and rendered together
        {"name": "scene_batch", "kind": "batch", "scenes": 16, "n_lo": 1000, "n_hi": 200000, "spp": 4, "depth": 5},
        # a burst of served requests on resident scenes
        {"name": "serve_burst", "kind": "serve", "scenes": 5, "n_lo": 1000, "n_hi": 200000, "requests": 12, "depth": 5},
        # the reference's per-frame call with the reference's own tree arrays
        {"name": "drawframe_ref", "kind": "drawframe", "scene": "soup", "n": 65538, "accel": "bvh", "w": 640, "h": 480,
         "spp": 1, "depth": 6},
        # visibility and picking queries of a simulation over the soup
        {"name": "ray_queries", "kind": "queries", "scene": "soup", "n": 65538, "accel": "bvh", "rays": 1000003},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case.  Image sizes, sample counts, shape counts, ray counts and request counts are spread
    over the ranges above; pixels x samples are held so that no drawn image costs more than mesh_frame."""
    kind = rng.choice(["frame", "frame", "frame", "viewer", "animate", "build", "build", "batch", "serve", "drawframe",
                       "queries", "queries"])
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(3, 16), "n_lo": 1000, "n_hi": _log(rng, 4000, 200000),
                "spp": rng.choice([1, 2, 4]), "depth": 5}
    if kind == "serve":
        return {"kind": kind, "scenes": rng.randint(1, 5), "n_lo": 1000, "n_hi": _log(rng, 4000, 200000),
                "requests": rng.randint(1, 12), "depth": 5}
    if kind == "build":
        return {"kind": kind, "scene": "soup", "n": _log(rng, 300, 4000000), "accel": "bvh"}
    if kind == "queries":
        return {"kind": kind, "scene": "soup", "n": _log(rng, 1000, 65538), "accel": rng.choice(["bvh", "bvh", "kd_sah"]),
                "rays": _log(rng, 500, 1000000)}
    scene = rng.choice(["soup", "mesh"])
    if kind == "viewer":
        n = _log(rng, 300, 30000) if scene == "soup" else 12 + 20 * 4 ** rng.randint(1, 5)
        return {"kind": kind, "scene": scene, "n": n, "accel": "bvh", "treelet": 0, "w": _log(rng, 40, 320),
                "h": _log(rng, 30, 240), "spp": 1, "depth": rng.randint(3, 6)}
    if kind == "animate":
        n = _log(rng, 1000, 100000) if scene == "soup" else 12 + 20 * 4 ** rng.randint(3, 6)
        return {"kind": kind, "scene": scene, "n": n, "accel": "bvh", "treelet": rng.choice([0, 5, 7]),
                "w": _log(rng, 160, 800), "h": _log(rng, 120, 600), "spp": rng.randint(1, 4), "depth": 5}
    if kind == "drawframe":
        n = _log(rng, 300, 100000) if scene == "soup" else 12 + 20 * 4 ** rng.randint(2, 6)
        accel = rng.choice(["bvh", "bvh", "kd"])
        if accel == "kd":
            n = _log(rng, 300, 2000) if scene == "soup" else 332   # the int16 heap arrays hold small trees
        return {"kind": kind, "scene": scene, "n": n, "accel": accel, "w": _log(rng, 160, 800), "h": _log(rng, 120, 600),
                "spp": 1, "depth": 6}
    accel = rng.choice(["bvh", "bvh", "bvh", "none", "kd_sah", "kd"])
    if accel == "none":
        return {"kind": kind, "scene": "cornell", "n": 9, "accel": accel, "treelet": 0, "w": _log(rng, 64, 512),
                "h": _log(rng, 48, 512), "spp": rng.randint(1, 8), "depth": rng.randint(3, 6)}
    if accel == "kd":   # the mean-split tree: leaves of a dozen shapes
        n = _log(rng, 300, 10000) if scene == "soup" else 12 + 20 * 4 ** rng.randint(2, 4)
        return {"kind": kind, "scene": scene, "n": n, "accel": accel, "treelet": 0, "w": _log(rng, 64, 400),
                "h": _log(rng, 48, 300), "spp": rng.randint(1, 4), "depth": 5}
    big = 100000 if accel == "bvh" else 20000
    n = _log(rng, 1000, big) if scene == "soup" else 12 + 20 * 4 ** rng.randint(3, 7 if accel == "bvh" else 5)
    return {"kind": kind, "scene": scene, "n": n, "accel": accel,
            "treelet": rng.choice([0, 5, 7]) if accel == "bvh" else 0, "w": _log(rng, 64, 900), "h": _log(rng, 48, 700),
            "spp": rng.choice([1, 2, 4, 8]), "depth": rng.randint(4, 6)}


# ---- inputs -------------------------------------------------------------------------------------

def _mesh_level(n):
    level = 0
    while 20 * 4 ** level + 12 < n:
        level += 1
    return level


def _shapes(case, seed):
    """(shapes, light count, camera) of a single-scene case, on the host."""
    w, h = int(case.get("w", 64)), int(case.get("h", 64))
    if case["scene"] == "cornell":
        s, lc, cam = scenes.cornell(w, h)
        # another seed: the two glass and mirror balls elsewhere on the floor
        r = np.random.default_rng(seed)
        s["p"][6:8, 0] += r.uniform(-6.0, 6.0, 2).astype(np.float32)
        s["p"][6:8, 2] += r.uniform(-6.0, 6.0, 2).astype(np.float32)
    elif case["scene"] == "soup":
        s, lc, cam = scenes.soup(int(case["n"]) - 2, seed=seed, width=w, height=h)
    else:
        s, lc, cam = scenes.icosphere_in_box(_mesh_level(int(case["n"])), seed, w, h)
    pt.update_camera(cam)
    return s, lc, cam


def _big_soup(ctx, n, seed):
    """The soup of scenes.soup in shape and distribution, made on the GPU: the words of `n` Shapes."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    m = n - 2
    d = ctx.alloc(n * SHAPE_DTYPE.itemsize, np.uint8)
    rec = _tensor(d, "<f4", (n, 26))
    rec.zero_()
    iv = rec.view(torch.int32)
    iv[:, 0] = 1
    cen = torch.rand((m, 1, 3), generator=g, device="cuda")
    tri = cen + (torch.rand((m, 3, 3), generator=g, device="cuda") * 0.02 - 0.01)
    rec[:m, 1:10] = tri.reshape(m, 9)
    rec[:m, 13:16] = 0.75
    e1, e2 = tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    rec[:m, 25] = torch.linalg.cross(e1, e2).norm(dim=1) * 0.5
    quad = torch.tensor([[.25, 1.25, .25, .75, 1.25, .25, .75, 1.25, .75], [.25, 1.25, .25, .75, 1.25, .75, .25, 1.25, .75]])
    rec[m:, 1:10] = quad.cuda()
    rec[m:, 10:13] = 12.0
    rec[m:, 25] = 0.125
    torch.cuda.synchronize()
    return d


class _Span:
    """Device memory seen by torch without a copy; keeps the object that holds it."""

    def __init__(self, ptr, typestr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (int(ptr), False), "version": 2}


def _tensor(buf, typestr, shape, ptr=None):
    return torch.as_tensor(_Span(buf.ptr if ptr is None else ptr, typestr, shape, buf), device="cuda")


def _seeds(w, h, seed):
    # as the reference seeds a frame: two random words of at least 2 per pixel
    return np.random.default_rng(seed + 77).integers(2, 1 << 31, 2 * w * h, dtype=np.uint32)


def _frame_buffers(ctx, w, h, seed):
    col = ctx.alloc(w * h * 12, np.float32).zero()
    sd0 = ctx.to_device(_seeds(w, h, seed))
    sd = ctx.to_device(_seeds(w, h, seed))
    pix = ctx.alloc(w * h * 4, np.uint32).zero()
    return col, sd0, sd, pix


def _outputs(col, sd, pix, w, h):
    return {"colors": _tensor(col, "<f4", (w * h, 3)), "seeds": _tensor(sd, "<i4", (w * h, 2)),
            "pixels": _tensor(pix, "<i4", (w * h,))}


def _tree(ctx, case, shapes, d_shapes):
    """(bvh, kd) of a single-scene case."""
    accel = case["accel"]
    if accel == "none":
        return None, None
    if accel in ("kd", "kd_sah"):
        return None, pt.KDTree(ctx, shapes, sah=accel == "kd_sah", max_depth=24)
    bvh = pt.CLBVH(ctx, d_shapes)
    bvh.buildRadixTree()
    bvh.buildBVHTree()
    if case.get("treelet"):
        bvh.optimize(int(case["treelet"]))
    return bvh, None


def _rays(n, seed):
    """Half of the rays start inside the scene in any direction, half look at it from a point outside."""
    r = np.random.default_rng(seed + 5)
    out = np.empty((n, 6), np.float32)
    k = n // 2
    out[:k, :3] = r.random((k, 3), dtype=np.float32)
    out[k:, :3] = np.float32([0.5, 0.5, 2.5])
    d = r.standard_normal((n, 3)).astype(np.float32)
    d[k:] = np.float32([0.5, 0.5, 0.5]) + (r.random((n - k, 3), dtype=np.float32) - np.float32(0.5)) - out[k:, :3]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    out[:, 3:] = d
    maxt = r.uniform(0.1, 2.0, n).astype(np.float32)
    return out, maxt


def _scene_counts(case):
    """Triangle counts of a scene set, spread evenly over the range's logarithm, small and large in turn."""
    k, lo, hi = int(case["scenes"]), math.log(case["n_lo"]), math.log(case["n_hi"])
    at = [k - 1 - i // 2 if i % 2 else i // 2 for i in range(k)]
    return [int(math.exp(lo + (hi - lo) * (a + 0.5) / k)) for a in at]


def _scene_set(case, seed):
    """The scenes of a batch or a server: soup or truncated icosphere by seed."""
    return [scenes.mixed_scene(1000 * (seed % 100000) + k, n)[:2] for k, n in enumerate(_scene_counts(case))]


# frame sizes and sample counts of a batch's images and of served requests, in turn
_EDGES = (256, 512, 128, 256, 512)
_SPPS = (4, 1, 16)


def _orbit(r, edge):
    cam = scenes.orbit_camera(float(r.uniform(0, 2 * math.pi)), edge, edge)
    pt.update_camera(cam)
    return cam


def prepare(case, seed):
    ctx = _ctx()
    kind = case["kind"]
    st = {"ctx": ctx, "kind": kind, "case": case}
    if kind in ("frame", "viewer", "animate", "drawframe"):
        w, h = int(case["w"]), int(case["h"])
        shapes, lc, cam = _shapes(case, seed)
        d_shapes = ctx.to_device(shapes)
        bvh, kd = (None, None) if kind == "drawframe" else _tree(ctx, case, shapes, d_shapes)
        col, sd0, sd, pix = _frame_buffers(ctx, w, h, seed)
        st.update(bvh=bvh, kd=kd, sd0=sd0, sd=sd, k=0, out=_outputs(col, sd, pix, w, h),
                  args=dict(colors=col, seeds=sd, camera=ctx.to_device(cam), shapes=d_shapes, shapeCnt=len(shapes),
                            lightCnt=lc, width=w, height=h, pixels=pix))
        if kind == "drawframe":
            if case["accel"] == "kd":
                kng, kn = pt.KDTree(None, shapes).getTrees()
                st["tree"] = dict(kng=ctx.to_device(kng), kngCnt=len(kng), kn=ctx.to_device(kn), knCnt=len(kn))
            else:
                b = pt.CLBVH(ctx, d_shapes)
                b.buildRadixTree()
                b.buildBVHTree()
                btn, btl = b.getTrees()
                st["tree"] = dict(btn=ctx.to_device(btn), btl=ctx.to_device(btl))
        else:
            st["args"].update(spp=int(case["spp"]), max_depth=int(case["depth"]))
    elif kind == "build":
        n = int(case["n"])
        d_shapes = _big_soup(ctx, n, seed)
        st.update(d_shapes=d_shapes, n=n, bvh=pt.CLBVH(ctx, d_shapes))
    elif kind == "queries":
        n = int(case["rays"])
        shapes, _, _ = _shapes(case, seed)
        d_shapes = ctx.to_device(shapes)
        bvh, kd = _tree(ctx, case, shapes, d_shapes)
        rays, maxt = _rays(n, seed)
        t, ids, hit = (ctx.alloc(4 * n, d) for d in (np.float32, np.int32, np.int32))
        st.update(bvh=bvh, kd=kd, d_shapes=d_shapes, n_shapes=len(shapes), n=n, rays=ctx.to_device(rays),
                  maxt=ctx.to_device(maxt), t=t, ids=ids, hit=hit,
                  out={"t": _tensor(t, "<f4", (n,)), "id": _tensor(ids, "<i4", (n,)), "hit": _tensor(hit, "<i4", (n,))})
    elif kind == "batch":
        jobs, handles, outs, src = [], [], [], []
        r = np.random.default_rng([seed, 9])
        for k, (s, lc) in enumerate(_scene_set(case, seed)):
            w = h = _EDGES[k % len(_EDGES)]
            cam = _orbit(r, w)
            d_shapes = ctx.to_device(s)
            col, sd0, sd, pix = _frame_buffers(ctx, w, h, seed + k)
            handles.append(pt.CLBVH(ctx, d_shapes))
            jobs.append(dict(bvh=handles[-1], colors=col, seeds=sd, camera=ctx.to_device(cam), shapes=d_shapes,
                             shapeCnt=len(s), lightCnt=lc, width=w, height=h, spp=int(case["spp"]),
                             max_depth=int(case["depth"]), pixels=pix))
            src.append((sd, sd0))
            outs.append(_outputs(col, sd, pix, w, h))
        st.update(jobs=jobs, handles=handles, src=src, out=outs)
    elif kind == "serve":
        pool = _scene_set(case, seed)
        r = np.random.default_rng([seed, 9])
        reqs = []
        for k in range(int(case["requests"])):
            sc, w = k % len(pool), _EDGES[k % len(_EDGES)]
            reqs.append((sc, *pool[sc], _orbit(r, w), w, w, _SPPS[(k // 2) % len(_SPPS)]))
        st.update(reqs=reqs, srv=pt.Server(ctx, 8 << 30, spp_per_tick=16))
    else:
        raise ValueError(kind)
    return st


def run(st):
    ctx, kind = st["ctx"], st["kind"]
    if kind == "frame":
        st["sd"].copy_from(st["sd0"])
        pt.render(ctx, st["bvh"], st["kd"], **st["args"])
        return st["out"]
    if kind == "viewer":
        pt.render(ctx, st["bvh"], st["kd"], currentSample=st["k"], **st["args"])
        st["k"] += 1
        return st["out"]
    if kind == "animate":
        b = st["bvh"]
        b.reset()
        b.buildRadixTree()
        b.buildBVHTree()
        if st["case"]["treelet"]:
            b.optimize(int(st["case"]["treelet"]))
        st["sd"].copy_from(st["sd0"])
        pt.render(ctx, b, None, **st["args"])
        return st["out"]
    if kind == "build":
        b = st["bvh"]
        b.reset()
        b.buildRadixTree()
        b.buildBVHTree()
        n = st["n"]
        if "out" not in st:
            btn, btl = b.device_trees()
            st["out"] = {"btn": _tensor(b, "<i4", (n - 1, 15), btn), "btl": _tensor(b, "<i4", (n, 15), btl),
                         "shapes": _tensor(st["d_shapes"], "<i4", (n, 26))}
        return st["out"]
    if kind == "batch":
        pt.CLBVH.build_batch(ctx, st["handles"])
        for sd, sd0 in st["src"]:
            sd.copy_from(sd0)
        pt.render_batch(ctx, st["jobs"])
        return st["out"]
    if kind == "serve":
        srv, depth = st["srv"], int(st["case"]["depth"])
        ids = [srv.submit(sc, s, lc, cam, w, h, spp, depth) for sc, s, lc, cam, w, h, spp in st["reqs"]]
        out, left = {}, len(ids)
        while left:
            srv.tick()
            for rid in srv.finished():
                col, pix, _ = srv.result(rid)
                out[ids.index(rid)] = {"colors": col, "pixels": pix.view(np.int32)}
                left -= 1
        return [out[k] for k in range(len(ids))]
    if kind == "drawframe":
        a = st["args"]
        accel = lib.ACCEL_KD if st["case"]["accel"] == "kd" else lib.ACCEL_BVH
        pt.radiance_gpu(ctx, accel, a["colors"], a["seeds"], a["camera"], a["shapes"], a["shapeCnt"], a["lightCnt"],
                        width=a["width"], height=a["height"], currentSample=st["k"], pixels=a["pixels"], **st["tree"])
        st["k"] += 1
        return st["out"]
    pt.trace_closest(ctx, st["bvh"], st["kd"], st["d_shapes"], st["n_shapes"], st["rays"], st["n"], st["t"], st["ids"])
    pt.trace_any(ctx, st["bvh"], st["kd"], st["d_shapes"], st["n_shapes"], st["rays"], st["maxt"], st["n"], st["hit"])
    return st["out"]


def work(case):
    """What a pass cannot do without.  Bytes: each input read and each output written once (a Shape is 104
    bytes, an exported node 60, a pixel 24 bytes of colour, seeds and packed colour, its seeds read too).
    Operations: per ray, two box tests of 18 operations per tree level and one triangle test of 45; rays per
    sample: 2.7 in the open soup, about two per bounce in a closed box."""
    kind = case["kind"]

    def ray_flops(n):
        return 36.0 * math.log2(max(n, 2)) + 45.0

    if kind == "build":
        n = case["n"]
        return {"bytes": 104.0 * n + 32.0 * n + 60.0 * (2 * n - 1), "flops": 40.0 * n}
    if kind == "queries":
        return {"bytes": 104.0 * case["n"] + 40.0 * case["rays"], "flops": 2.0 * case["rays"] * ray_flops(case["n"])}
    if kind in ("batch", "serve"):
        counts = _scene_counts(case)
        b = sum(104.0 * n for n in counts)
        f = 0.0
        if kind == "batch":
            b += sum(152.0 * n for n in counts)
            f += sum(40.0 * n for n in counts)
        for k in range(case["scenes"] if kind == "batch" else case["requests"]):
            px = float(_EDGES[k % len(_EDGES)]) ** 2
            spp = case["spp"] if kind == "batch" else _SPPS[(k // 2) % len(_SPPS)]
            b += 32.0 * px
            f += px * spp * 2.7 * ray_flops(counts[k % len(counts)])
        return {"bytes": b, "flops": f}
    n, px = case["n"], case["w"] * case["h"]
    q = 2.7 if case["scene"] == "soup" else 2.0 * case["depth"]
    per_ray = 20.0 * n if case["accel"] == "none" else ray_flops(n)
    b = 104.0 * n + 32.0 * px + (120.0 * n if kind == "drawframe" else 32.0 * n if kind == "animate" else 0)
    return {"bytes": b, "flops": px * case["spp"] * q * per_ray + (40.0 * n if kind == "animate" else 0)}


# ---- 64-bit answers -----------------------------------------------------------------------------

def exact(case, seed):
    """Closest-hit distances in 64 bits, by testing every ray against every triangle (Pluecker form).  Images
    have no such value: a path is a chain of discrete choices (which shape is hit, whether a light is seen,
    which way a ray refracts), so 64 bits would follow other paths; builds return integers and copies."""
    if case["kind"] != "queries" or case["scene"] != "soup" or case["n"] * case["rays"] > 1e11:
        return None
    shapes, _, _ = _shapes(case, seed)
    rays, _ = _rays(int(case["rays"]), seed)
    f64 = dict(dtype=torch.float64, device="cuda")
    v0, v1, v2 = (torch.tensor(np.ascontiguousarray(shapes[k]), **f64) for k in ("p1", "p2", "p3"))
    e1, e2 = v1 - v0, v2 - v0
    nrm = torch.linalg.cross(e1, e2)
    den_w = -nrm.T.contiguous()                                    # det = -d.n
    t_w = torch.cat([nrm, -(v0 * nrm).sum(1, keepdim=True)], 1).T.contiguous()   # t det = (o - v0).n
    # u det = (o - v0).(d x e2) = (o x d).e2 - d.(e2 x v0);  v det = d.((o - v0) x e1)
    u_w = torch.cat([e2, -torch.linalg.cross(e2, v0)], 1).T.contiguous()
    v_w = torch.cat([-e1, torch.linalg.cross(e1, v0)], 1).T.contiguous()
    r = torch.tensor(rays, **f64)
    out = torch.zeros(len(r), **f64)
    for a in range(0, len(r), 4096):
        o, d = r[a:a + 4096, :3], r[a:a + 4096, 3:]
        od = torch.cat([torch.linalg.cross(o, d), d], 1)
        inv = 1.0 / (d @ den_w)
        t = (torch.cat([o, torch.ones_like(o[:, :1])], 1) @ t_w).mul_(inv)
        u = (od @ u_w).mul_(inv)
        v = (od @ v_w).mul_(inv)
        bad = (u < 0) | (v < 0) | (u.add_(v) > 1) | ~(t > 0.01)
        t.masked_fill_(bad, 1e20)
        best = t.min(1).values
        out[a:a + 4096] = torch.where(best < 1e20, best, torch.zeros_like(best))
    return {"t": out, "id": None, "hit": None}
