"""Measured work of the grid-acceleration path, one case per way the library
is used: rebuilds of static and moving meshes, camera frames, ray batches of
every size, any-hit segments, diffuse paths, batched scenes and served
requests, on both grid kinds.

A case is a dict of plain values; ``prepare`` makes its inputs from a seed,
``run`` makes one pass through the public entry points.  Cases that return a
grid's arrays take the geometry from their ``scene_seed`` (which fixes the
arrays' sizes) and the order of the triangles, camera and bounce seeds from
the seed; the others take everything from the seed.
"""
from __future__ import annotations

import ctypes as C
import math
import os

import numpy as np
import torch

import shinobi_amd as sa
from shinobi_amd import _lib as L
from shinobi_amd import workloads as W

GOLDEN = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(sa.__file__))), "tests", "golden")
FLT_MAX = 3.4028234663852886e38
RUINS_TRIS = 38_665


def listed():
    return [
        # the smallest rebuild: the 10,000-triangle soup of the uniform grid's
        # own configuration, where the launches of a build count
        dict(name="soup10k_rebuild", path="rebuild", kind="uniform", scene="soup", tris=10_000, lam=5.0, radix=8,
             scene_seed=1),
        # the same configuration's view: 256 x 256 camera rays
        dict(name="soup10k_camera", path="camera", kind="uniform", scene="soup", tris=10_000, lam=5.0,
             res_x=256, res_y=256, tile_w=2, tile_h=32),
        # the smallest served request: 1,000 incoherent rays, two-level grid
        dict(name="rays1k_twolevel", path="rays", kind="two_level", scene="soup", tris=225_615, lam=5.0, rays=1_000),
        # the largest served request: 1,000,000 incoherent rays
        dict(name="rays1m_uniform", path="rays", kind="uniform", scene="soup", tris=61_005, lam=5.0, rays=1_000_000),
        # direct illumination in an OBJ scene: any-hit segments to one light
        dict(name="ruins_shadow", path="shadow", kind="two_level", scene="ruins", tris=RUINS_TRIS, lam=5.0,
             rays=300_007),
        # a moving mesh: new vertices (in device memory) and its rebuild
        dict(name="sphere200k_dynamic", path="dynamic", kind="two_level", scene="sphere", tris=200_000, lam=5.0,
             scene_seed=5),
        # the headline scene's rebuild, 2,093,058 triangles
        dict(name="heightfield2m_rebuild", path="rebuild", kind="two_level", scene="heightfield", tris=2_093_058,
             lam=5.0, radix=8, scene_seed=2),
        # a dense cluster in a large scene: top cells of very many triangles,
        # and (in about half of such scenes) a large triangle across them
        dict(name="cluster502k_rebuild", path="rebuild", kind="two_level", scene="cluster", tris=502_000, lam=5.0,
             radix=8, scene_seed=4),
        # the headline frame: rebuild, camera rays, one bounce per hit (longest
        # rays first) and its trace
        dict(name="heightfield2m_frame", path="frame", kind="two_level", scene="heightfield", tris=2_093_058,
             lam=5.0, res_x=1920, res_y=1080, tile_w=2, tile_h=32, scene_seed=2),
        # diffuse paths of four segments in the dense cluster, direction-class
        # bounce order, counts kept on the device
        dict(name="cluster_paths", path="paths", kind="two_level", scene="cluster", tris=502_000, lam=5.0,
             res_x=1280, res_y=720, depth=4),
        # many scenes of very different sizes: one captured graph rebuilds
        # every grid and traces every batch
        dict(name="batch30", path="batch", kind="uniform", scene="soup", scenes=30, tris_lo=1_000, tris_hi=500_000,
             rays_lo=10_000, rays_hi=2_000_000, lam=5.0, scene_seed=4),
        # a burst of requests from host memory against resident grids
        dict(name="serve24", path="serve", kind="two_level", scene="soup", requests=24, rays_lo=1_000,
             rays_hi=1_000_000, lam=5.0),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    path = rng.choice(["rebuild", "rebuild", "camera", "rays", "rays", "shadow", "dynamic", "frame", "paths", "batch",
                       "serve"])
    kind = rng.choice(["uniform", "two_level"])
    scene_seed = rng.randint(1, 1 << 20)
    if path == "rebuild":
        if kind == "uniform":
            return dict(path=path, kind=kind, scene="soup", tris=log_int(1_000, 500_000),
                        lam=rng.choice([1.0, 2.0, 3.0, 5.0, 8.0]), radix=rng.choice([4, 6, 8]), scene_seed=scene_seed)
        scene = rng.choice(["soup", "heightfield", "cluster"])
        hi = 500_000 if scene == "cluster" else 2_000_000
        return dict(path=path, kind=kind, scene=scene, tris=log_int(5_000, hi), lam=rng.choice([3.0, 5.0, 8.0]),
                    radix=8, scene_seed=scene_seed)
    if path == "camera":
        scene = "soup" if kind == "uniform" else "heightfield"
        return dict(path=path, kind=kind, scene=scene, tris=log_int(5_000, 1_000_000), lam=5.0,
                    res_x=log_int(64, 1920), res_y=log_int(64, 1080), tile_w=rng.choice([1, 2, 8]),
                    tile_h=rng.choice([1, 8, 32]))
    if path == "rays":
        return dict(path=path, kind=kind, scene=rng.choice(["soup", "heightfield"]), tris=log_int(5_000, 1_000_000),
                    lam=rng.choice([3.0, 5.0]), rays=log_int(500, 1_000_000))
    if path == "shadow":
        return dict(path=path, kind=kind, scene="ruins", tris=RUINS_TRIS, lam=rng.choice([3.0, 5.0]),
                    rays=log_int(1_000, 1_000_000))
    if path == "dynamic":
        return dict(path=path, kind=kind, scene="sphere", tris=log_int(2_000, 500_000), lam=5.0,
                    scene_seed=scene_seed)
    if path == "frame":
        return dict(path=path, kind="two_level", scene="heightfield", tris=log_int(30_000, 2_000_000), lam=5.0,
                    res_x=log_int(320, 1920), res_y=log_int(240, 1080), tile_w=2, tile_h=32,
                    scene_seed=scene_seed)
    if path == "paths":
        return dict(path=path, kind="two_level", scene="cluster", tris=log_int(20_000, 500_000), lam=5.0,
                    res_x=log_int(160, 1280), res_y=log_int(120, 720), depth=rng.choice([2, 3, 4]))
    if path == "batch":
        return dict(path=path, kind="uniform", scene="soup", scenes=rng.randint(3, 24), tris_lo=1_000,
                    tris_hi=log_int(20_000, 500_000), rays_lo=10_000, rays_hi=log_int(50_000, 2_000_000), lam=5.0,
                    scene_seed=scene_seed)
    return dict(path=path, kind="two_level", scene="soup", requests=rng.randint(4, 24), rays_lo=1_000,
                rays_hi=log_int(20_000, 1_000_000), lam=5.0)


# ------------------------------------------------------------------ inputs
_CTX = None


def _ctx():
    global _CTX
    if _CTX is None:
        _CTX = sa.Context(0)
    return _CTX


def _triangles(case, seed):
    """(9, N) float32 vertices of the case's scene.  With a scene_seed the
    seed only turns the triangle list: it starts at another triangle."""
    if "scene_seed" in case:
        tri = _scene(case, case["scene_seed"])
        return np.roll(tri, _turn(tri.shape[1], seed), axis=1)
    return _scene(case, seed)


def _turn(n, seed):
    return int(np.random.default_rng(seed).integers(1, n))


def _scene(case, seed):
    n, scene = case["tris"], case["scene"]
    if scene == "soup":
        return sa.gen_soup(seed, n, 0.01 * (1e4 / n) ** (1.0 / 3.0))
    if scene == "heightfield":
        return sa.gen_heightfield(seed, _field_side(n), 0.2)
    if scene == "cluster":
        large = max(16, n // 251)
        return sa.gen_cluster(seed, n - large, large)
    if scene == "sphere":
        return W.sphere_mesh(n, frame=0, seed=seed)
    return _ruins().scene


def _field_side(n):
    return max(8, int(round(math.sqrt(n / 2.0))) + 1)


def _ruins():
    return W.scene_file(os.path.join(GOLDEN, "ruins.obj.gz"), os.path.join(GOLDEN, "ruins_camera.cfg"))


def _camera(case, seed):
    res = (case["res_x"], case["res_y"])
    if case["scene"] == "heightfield":
        eye, fwd, *rest = W.heightfield_pinhole(case.get("scene_seed", seed), *res)
        side = float(np.random.default_rng(seed).uniform(-0.1, 0.1))   # the viewer steps aside
        return ((eye[0] + side,) + eye[1:], (fwd[0] - side,) + fwd[1:], *rest)
    z = -0.6 if case["scene"] == "cluster" else -1.0
    return ((0.5, 0.5, z), (0.0, 0.0, 1.0), (0.0, 1.0, 0.0), 60.0) + res


def _shadow_rays(tri, n, seed):
    """Segments from random points of the surfaces (area-weighted) to one
    light above the scene: direction = light - origin, tmax 1."""
    rng = np.random.default_rng(seed)
    v = tri.reshape(3, 3, -1).astype(np.float64)
    nrm = np.cross(v[1] - v[0], v[2] - v[0], axis=0)
    area = np.linalg.norm(nrm, axis=0)
    k = rng.choice(area.size, n, p=area / area.sum())
    a, b = rng.random(n), rng.random(n)
    flip = a + b > 1.0
    a, b = np.where(flip, 1.0 - a, a), np.where(flip, 1.0 - b, b)
    p = v[0][:, k] + a * (v[1] - v[0])[:, k] + b * (v[2] - v[0])[:, k]
    lo, hi = v.min(axis=(0, 2)), v.max(axis=(0, 2))
    light = (lo + (hi - lo) * rng.uniform(0.3, 0.7, 3))[:, None]
    light[1] = hi[1] + 0.5 * (hi[1] - lo[1])
    u = nrm[:, k] / np.maximum(area[k], 1e-30)
    u = np.where((u * (light - p)).sum(axis=0) < 0.0, -u, u)
    p = p + 1e-3 * np.linalg.norm(hi - lo) * u
    return np.concatenate([p, light - p, np.ones((1, n))]).astype(np.float32)


def _rays(case, seed, tri):
    n = case["rays"]
    if case["path"] == "shadow":
        return _shadow_rays(tri, n, seed)
    return sa.gen_random_rays(seed + 77, n, 0.0, 1.0)


class _Out:
    """A torch tensor where the Python interface takes a DeviceBuffer."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = C.c_void_p(tensor.data_ptr())


def _words(n):
    return _Out(torch.zeros(max(int(n), 1), dtype=torch.int32, device="cuda"))


def _floats(n):
    return _Out(torch.zeros(max(int(n), 1), dtype=torch.float32, device="cuda"))


class _RayTensor:
    """7 x n rays in one torch tensor, where the interface takes a RayBatch."""

    def __init__(self, n):
        self.n = n
        self.tensor = torch.zeros((7, n), dtype=torch.float32, device="cuda")

    def struct(self):
        r = L.Rays()
        p = self.tensor.data_ptr()
        for i in range(3):
            r.o[i] = p + 4 * i * self.n
            r.d[i] = p + 4 * (3 + i) * self.n
        r.tmax = p + 24 * self.n
        return r


class _DeviceWords:
    """uint32 words of a grid's device arrays as a torch tensor (int32)."""

    def __init__(self, owner, addr, n):
        self.owner = owner   # the grid lives as long as the tensor
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": "<i4", "data": (int(addr), False),
                                         "version": 2}


def _grid_arrays(grid):
    v = grid.device_view()
    if v.status != 0:
        raise RuntimeError(f"grid status {v.status}")
    out = [torch.as_tensor(_DeviceWords(grid, v.cells, 2 * v.n_cells), device="cuda")]
    if v.leaves:
        out.append(torch.as_tensor(_DeviceWords(grid, v.leaves, 2 * v.n_leaves), device="cuda"))
    out.append(torch.as_tensor(_DeviceWords(grid, v.indices, v.n_refs), device="cuda"))
    return out


def _build(case, scene):
    if case["kind"] == "uniform":
        b = sa.FastSimpleGridBuilder(_ctx(), lam=case["lam"], radix_bits=case.get("radix", 8))
    else:
        leaf = 1.2 if case["scene"] == "ruins" else 2.0
        b = sa.FastTwoLevelGridBuilder(_ctx(), lam=case["lam"], top_divisor=6, lambda_leaf=leaf, leaf_min_refs=16,
                                       radix_bits=case.get("radix", 8))
    b.init(scene)
    return b.build()


def _log_sizes(rng, lo, hi, n):
    return [int(x) for x in np.exp(rng.uniform(math.log(lo), math.log(hi), n))]


def _prepare_batch(case, seed):
    ctx, k = _ctx(), case["scenes"]
    # the sizes are the case's; the seed decides what the scenes hold
    rng = np.random.default_rng(4)
    tris = _log_sizes(rng, case["tris_lo"], case["tris_hi"], k)
    rays = _log_sizes(rng, case["rays_lo"], case["rays_hi"], k)
    st = {"grids": [], "rays": []}
    prim, t = _words(sum(rays)), _floats(sum(rays))
    batch = sa.Batch(ctx, k)
    at = 0
    for i in range(k):
        soup = sa.gen_soup(case["scene_seed"] + 4000 + i, tris[i], 0.01 * tris[i] ** (-1.0 / 3.0))
        soup = sa.FaceSoup(ctx, np.roll(soup, _turn(tris[i], seed), axis=1))
        grid = _build(case, soup)
        rb = sa.RayBatch(ctx, sa.gen_random_rays(seed + 6000 + i, rays[i], 0.0, 1.0))
        batch.add(grid, rb, _Out(prim.tensor[at:]), _Out(t.tensor[at:]))
        st["grids"].append(grid)
        st["rays"].append(rb)
        at += rays[i]
    batch.commit()
    ctx.sync()
    with sa.Graph.capture(ctx) as graph:
        batch.rebuild(branches=16)
        batch.launch()
    st.update(batch=batch, graph=graph, out=[prim.tensor, t.tensor] + [a for g in st["grids"] for a in _grid_arrays(g)])
    return st


def _prepare_serve(case, seed):
    ctx = _ctx()
    rng = np.random.default_rng(5)
    st = {"grids": [], "reqs": []}
    st["server"] = sa.Server(ctx, mode="batched", hbm_budget=3 << 30, max_requests=512, max_waves=4,
                             max_wave_rays=1 << 22)
    ids = []
    for i, n in enumerate((61_005, 142_578, 334_620, 554_759)):
        scene = "soup" if i % 2 == 0 else "heightfield"
        sub = dict(case, scene=scene, tris=n)
        grid = _build(sub, sa.FaceSoup(ctx, _triangles(sub, seed + i)))
        st["grids"].append(grid)
        ids.append(st["server"].add_grid(grid))
    sizes = _log_sizes(rng, case["rays_lo"], case["rays_hi"], case["requests"])
    prim = sa.PinnedArray(ctx, (sum(sizes),), np.uint32)
    t = sa.PinnedArray(ctx, (sum(sizes),), np.float32)
    at = 0
    for i, n in enumerate(sizes):
        r = sa.PinnedArray(ctx, (7, n), np.float32)
        r.a[:] = sa.gen_random_rays(seed + 900 + i, n, 0.0, 1.0)
        st["reqs"].append((ids[int(rng.integers(0, len(ids)))], r, prim.a[at:at + n], t.a[at:at + n]))
        at += n
    st["out"] = [prim.a.view(np.int32), t.a]
    return st


def prepare(case, seed):
    torch.zeros(1, device="cuda")
    ctx, path = _ctx(), case["path"]
    if path == "batch":
        st = _prepare_batch(case, seed)
    elif path == "serve":
        st = _prepare_serve(case, seed)
    else:
        tri = _triangles(case, seed)
        scene = sa.FaceSoup(ctx, tri)
        grid = _build(case, scene)
        st = {"scene": scene, "grid": grid}
        if path == "dynamic":
            # the next frame's vertices, where a simulation leaves them
            nxt = W.sphere_mesh(case["tris"], frame=1, seed=case["scene_seed"])
            nxt = torch.from_numpy(np.roll(nxt, _turn(nxt.shape[1], seed), axis=1)).cuda()
            st["next"] = nxt
            st["ptrs"] = L.Float9(*[nxt[i].data_ptr() for i in range(9)])
            torch.cuda.synchronize()
            _next_frame(st)
        if path in ("rebuild", "dynamic", "frame"):
            st["out"] = _grid_arrays(grid)
        if path in ("camera", "frame"):
            n = case["res_x"] * case["res_y"]
            st["cam"] = sa.pinhole(*_camera(case, seed))
            st["prim"], st["t"] = _words(n), _floats(n)
        if path in ("rays", "shadow"):
            st["rays"] = sa.RayBatch(ctx, _rays(case, seed, tri))
            st["prim"], st["t"] = _words(case["rays"]), _floats(case["rays"])
        if path == "frame":
            st["primary"], st["bounced"] = _RayTensor(n), _RayTensor(n)
            st["count"] = _words(1)
            st["bprim"], st["bt"] = _words(n), _floats(n)
            st["order"] = sa.bounce_order("exit", grid=grid)
        if path == "paths":
            rays = sa.RayBatch(ctx, sa.gen_camera_rays(*_camera(case, seed)))
            n, depth = rays.n, case["depth"]
            st["segs"] = [rays] + [_RayTensor(n) for _ in range(depth - 1)]
            st["counts"] = [None] + [_words(1) for _ in range(depth - 1)]
            st["prims"], st["ts"] = [_words(n) for _ in range(depth)], [_floats(n) for _ in range(depth)]
    st["case"], st["seed"] = case, seed
    ctx.sync()
    torch.cuda.synchronize()
    return st


# -------------------------------------------------------------------- passes
def _next_frame(st):
    ctx = _ctx()
    L.check(sa.lib().sg_scene_update(st["scene"].h, st["ptrs"], 1, ctx.stream), "sg_scene_update")
    st["grid"].rebuild()


def run(st):
    case, ctx = st["case"], _ctx()
    path = case["path"]
    if path == "rebuild":
        st["grid"].rebuild()
        return st["out"]
    if path == "dynamic":
        _next_frame(st)
        return st["out"]
    if path == "camera":
        st["grid"].trace_camera(st["cam"], (case["tile_w"], case["tile_h"]), prim=st["prim"], t=st["t"])
        return {"prim": st["prim"].tensor, "t": st["t"].tensor}
    if path in ("rays", "shadow"):
        st["grid"].trace(st["rays"], prim=st["prim"], t=st["t"], shadow=path == "shadow")
        return {"prim": st["prim"].tensor, "t": st["t"].tensor}
    if path == "frame":
        g = st["grid"]
        g.rebuild()
        g.trace_camera(st["cam"], (case["tile_w"], case["tile_h"]), prim=st["prim"], t=st["t"],
                       rays_out=st["primary"])
        sa.bounce(ctx, st["scene"], st["primary"], st["prim"], st["t"], st["seed"] + 100, st["bounced"],
                  count=st["count"], order=st["order"])
        g.trace(st["bounced"], prim=st["bprim"], t=st["bt"], d_count=st["count"].ptr)
        return {"grid": st["out"], "prim": st["prim"].tensor, "t": st["t"].tensor, "count": st["count"].tensor,
                "bounced": st["bounced"].tensor, "bounce_prim": st["bprim"].tensor, "bounce_t": st["bt"].tensor}
    if path == "paths":
        g, segs, counts = st["grid"], st["segs"], st["counts"]
        n = segs[0].n
        for d in range(case["depth"]):
            d_n = counts[d].ptr if d else None
            g.trace(segs[d], prim=st["prims"][d], t=st["ts"][d], d_count=d_n, n=n)
            if d + 1 < case["depth"]:
                sa.bounce(ctx, st["scene"], segs[d], st["prims"][d], st["ts"][d], st["seed"] + 103 + d, segs[d + 1],
                          count=counts[d + 1], d_n=d_n)
        return {"prim": [p.tensor for p in st["prims"]], "t": [t.tensor for t in st["ts"]],
                "rays": [s.tensor for s in segs[1:]], "count": [c.tensor for c in counts[1:]]}
    if path == "batch":
        st["graph"].launch()
        return st["out"]
    srv = st["server"]
    for sid, rays, prim, t in st["reqs"]:
        srv.submit(sid, rays.a, prim, t)
    srv.drain()
    return st["out"]


# --------------------------------------------------------------------- floors
# cells and references per triangle (pairs of the finished grid), and the
# arithmetic of one ray: 40 + 56 per test + 20 per step + 48 per entered cell
_CELLS = {"soup": 5.0, "heightfield": 2.0, "cluster": 2.0, "sphere": 2.5, "ruins": 1.4}
_REFS = {"soup": 2.5, "heightfield": 3.4, "cluster": 1.1, "sphere": 3.4, "ruins": 6.4}
_RAY_FLOPS = 1000.0


def _build_bytes(case, tris):
    # vertices in, cell ranges and references out
    return tris * (36.0 + 8.0 * _CELLS[case["scene"]] + 4.0 * _REFS[case["scene"]])


def _grid_bytes(case, tris):
    # what a full traversal of the scene reads once
    return tris * (36.0 + 8.0 * _CELLS[case["scene"]] + 4.0 * _REFS[case["scene"]])


def work(case):
    path = case["path"]
    if path in ("rebuild", "dynamic"):
        n = case["tris"]
        return {"bytes": _build_bytes(case, n), "flops": 60.0 * n}
    if path == "batch":
        rng = np.random.default_rng(4)
        tris = sum(_log_sizes(rng, case["tris_lo"], case["tris_hi"], case["scenes"]))
        rays = sum(_log_sizes(rng, case["rays_lo"], case["rays_hi"], case["scenes"]))
        return {"bytes": _build_bytes(case, tris) + _grid_bytes(case, tris) + 36.0 * rays,
                "flops": 60.0 * tris + _RAY_FLOPS * rays}
    if path == "serve":
        rays = sum(_log_sizes(np.random.default_rng(5), case["rays_lo"], case["rays_hi"], case["requests"]))
        return {"bytes": 2 * 36.0 * rays, "flops": _RAY_FLOPS * rays}
    n = case["rays"] if "rays" in case else case["res_x"] * case["res_y"]
    # a small batch reads no more of the scene than its rays cross
    scene = min(_grid_bytes(case, case["tris"]), 2000.0 * n)
    if path == "camera":
        return {"bytes": scene + 8.0 * n, "flops": _RAY_FLOPS * n}
    if path in ("rays", "shadow"):
        return {"bytes": scene + 36.0 * n, "flops": _RAY_FLOPS * n}
    if path == "frame":   # about 0.4 bounce rays per pixel
        return {"bytes": _build_bytes(case, case["tris"]) + 2 * scene + n * (36.0 + 0.4 * (28 + 28 + 36)),
                "flops": 60.0 * case["tris"] + 1.4 * _RAY_FLOPS * n}
    # paths: a fifth of the camera rays' count goes on, all segments together
    return {"bytes": scene + n * (36.0 + 0.2 * (28 + 28 + 36)), "flops": 1.2 * _RAY_FLOPS * n}


# ---------------------------------------------------------------------- exact
def _closest_t(tri, rays):
    """Distance of the closest hit of every ray (7, n) with every triangle
    (9, N), by Moeller and Trumbore's test written with Pluecker coordinates,
    in 64 bits; the ray's tmax where nothing is hit."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    v = torch.from_numpy(tri).to(dev).double().reshape(3, 3, -1)
    v0, e1, e2 = v[0].T, (v[1] - v[0]).T, (v[2] - v[0]).T
    r = torch.from_numpy(rays).to(dev).double()
    o, d, tmax = r[0:3].T, r[3:6].T, r[6]
    nrm = torch.linalg.cross(e1, e2)
    zero = torch.zeros_like(v0)
    # det = d . (e2 x e1) etc. for the ray (d, m = o x d): one product each
    det_c = torch.cat([-nrm, zero], 1)
    al_c = torch.cat([torch.linalg.cross(v0, e2), e2], 1)
    be_c = -torch.cat([torch.linalg.cross(v0, e1), e1], 1)
    plane = (nrm * v0).sum(1)
    best = tmax.clone()
    nt = v0.shape[0]
    step = max(1, (1 << 25) // nt)
    for a in range(0, o.shape[0], step):
        oo, dd = o[a:a + step], d[a:a + step]
        dm = torch.cat([dd, torch.linalg.cross(oo, dd)], 1)
        inv = (dm @ det_c.T).reciprocal_()
        al = (dm @ al_c.T).mul_(inv)
        be = (dm @ be_c.T).mul_(inv)
        t = (oo @ nrm.T).sub_(plane).mul_(inv)
        ok = (al >= 0) & (be >= 0) & (al.add_(be) <= 1) & (t > 1e-5)
        t = torch.where(ok, t, torch.full_like(t, math.inf)).amin(1)
        best[a:a + step] = torch.minimum(best[a:a + step], t)
    return best


def exact(case, seed):
    """The closest distances of camera and ray batches in 64 bits; ids, grids
    and bounce chains (whose rays follow the ids) have no such value."""
    if case["path"] not in ("camera", "rays"):
        return None
    n = case["rays"] if case["path"] == "rays" else case["res_x"] * case["res_y"]
    if n * case["tris"] > 7e10:
        return None
    tri = _triangles(case, seed)
    rays = _rays(case, seed, tri) if case["path"] == "rays" else sa.gen_camera_rays(*_camera(case, seed))
    return {"prim": None, "t": _closest_t(tri, rays)}
