"""The work this framework is used for, as cases that can be timed: cone
queries from the host and on the device, whole views, animated frames,
batches, the sky, the view cache and the lightmap.

A case is a dict of plain values. `prepare` makes what a program holds
before the call (a resident world, its frame buffers, cameras, lights and
poses drawn from the seed); `run` is one pass through the public entry
points; `work` counts what a pass cannot do without; `exact` evaluates the
cases over the room and the lightmap's room again in 64 bits, by plain
tensor code over every triangle.

Worlds are what a program loads once and keeps (the scene in HBM and one
set of frame buffers); what changes from seed to seed is what changes from
call to call: cameras, shading points, lights and poses.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from continuum_amd import _lib
from continuum_amd.kernel import Batch, Device, Flat, LiveLightmap, Scene, ViewCache
from continuum_amd.lightmap import Lightmap
from continuum_amd.renderer import Renderer, RendererOptions
from continuum_amd.scenes import (Pcg32, boulder_field, boulder_field_surface, camera_uniform, courtyard, lit_room,
                                  meshes_to_arrays, rect_light, rock_field, room_scene, vcache_world)
from continuum_amd.workloads import random_pose, random_rect_light

# Per query (cone), by world, the walk's work as the library's own counters
# give it: object nodes tested, triangle-hierarchy nodes tested, triangles
# tested, triangles drawn, meshes entered, nodes splatted.
WORK = {
    "room": (6.8, 22.6, 7.0, 0.1, 7.0, 0.0),
    "rock": (21.8, 52.4, 22.8, 1.8, 3.4, 0.0),
    "rock sky": (44.3, 784.0, 387.0, 60.1, 21.3, 249.0),
    "courtyard": (26.6, 228.0, 213.0, 70.3, 7.8, 25.7),
    "boulders": (19.0, 47.6, 21.6, 3.1, 2.0, 0.0),
    "field": (37.0, 180.0, 88.0, 12.7, 4.9, 0.0),
    "field moves": (82.0, 572.0, 290.0, 45.6, 15.2, 0.0),
    "yard": (42.0, 27.0, 41.0, 3.3, 21.0, 0.0),
}
# The least arithmetic of one of each (multiplies and adds): a box against
# the cone's six planes, a triangle against them, a drawn triangle's three
# edges, a splatted box's hull of six.
FLOPS = (60.0, 60.0, 90.0, 250.0, 100.0, 500.0)
QUERY_FLOPS = 500.0  # the cone's set-up and its window's weights


def listed() -> list:
    return [
        # A few shading points of a program that asks from the host (the
        # reference's `irradiance` calls): latency is everything.
        dict(name="room_query", kind="query", world="room", n=300, lights=1),
        # The smallest whole view: camera pass and cones, one light.
        dict(name="room_view", kind="view", world="room", w=256, h=256, lights=1, tile=16),
        # Scattered points (probes, texels, picked samples), a ragged list.
        dict(name="rock_points", kind="points", world="rock", n=20011, lights=3),
        # An ordinary view from a new camera each time.
        dict(name="rock_view", kind="view", world="rock", w=1280, h=720, lights=3, tile=16),
        # The sky's six cube faces over a view's points.
        dict(name="rock_sky", kind="sky", world="rock", w=640, h=360, tile=8),
        # An animated frame: refit of the moved curtains, camera pass, four
        # lights' cones, from a camera on a dolly.
        dict(name="courtyard_frame", kind="frame", world="courtyard", w=1280, h=720, lights=4, tile=8),
        # Several users' views of uneven sizes in one launch, read back.
        dict(name="courtyard_batch", kind="batch", world="courtyard", views=5, most=640, lights=3, tile=8),
        # A served view of the million-instance world, odd in size.
        dict(name="boulders_view", kind="view", world="boulders", w=853, h=479, lights=5, tile=16),
        # The view cache: pages new to the cache baked whole.
        dict(name="cache_bake", kind="cache bake", world="field", objects=64, radius=10.0),
        # The view cache: sixteen objects moved, the pages they reach re-baked.
        dict(name="cache_moves", kind="cache moves", world="field", objects=96, radius=12.0, movers=16),
        # The renderer's frame from its cache, one object moving.
        dict(name="cached_view", kind="renderer", world="yard", w=640, h=360),
        # The lightmap kept current as boxes move.
        dict(name="lightmap_moves", kind="lightmap", world="lit room", texel=0.08, boxes=8, moved=2),
    ]


def _log(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["query", "points", "points", "view", "view", "view", "sky", "frame", "batch", "cache bake",
                       "cache moves", "lightmap"])
    tile = rng.choice([8, 8, 16, 16, 32, 4])
    if kind == "query":
        return dict(kind=kind, world=rng.choice(["room", "room", "rock"]), n=int(_log(rng, 40, 6000)),
                    lights=rng.randint(1, 3))
    if kind == "points":
        return dict(kind=kind, world=rng.choice(["room", "rock", "courtyard"]), n=int(_log(rng, 500, 60000)),
                    lights=rng.randint(1, 4))
    if kind in ("view", "frame"):
        world = "courtyard" if kind == "frame" else rng.choice(["room", "rock", "courtyard", "boulders"])
        w = int(_log(rng, 100, 1000 if world in ("room", "rock") else 700))
        return dict(kind=kind, world=world, w=w, h=int(w * rng.uniform(0.5, 1.0)), lights=rng.randint(1, 4), tile=tile)
    if kind == "sky":
        w = int(_log(rng, 60, 400))
        return dict(kind=kind, world=rng.choice(["room", "rock"]), w=w, h=int(w * rng.uniform(0.5, 1.0)), tile=tile)
    if kind == "batch":
        return dict(kind=kind, world="courtyard", views=rng.randint(2, 6), most=int(_log(rng, 150, 640)),
                    lights=rng.randint(1, 3), tile=tile)
    if kind == "cache bake":
        return dict(kind=kind, world="field", objects=int(_log(rng, 2, 64)), radius=rng.uniform(2.0, 10.0))
    if kind == "cache moves":
        return dict(kind=kind, world="field", objects=rng.randint(20, 96), radius=rng.uniform(4.0, 12.0),
                    movers=rng.randint(1, 16))
    return dict(kind=kind, world="lit room", texel=rng.choice([0.08, 0.11, 0.16]), boxes=rng.randint(2, 8), moved=2)


# ---- worlds


@functools.lru_cache(maxsize=None)
def _device() -> Device:
    return Device(0)


def _gpu(a) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


class World:
    """A scene resident in HBM, with one set of frame buffers a view size."""

    def __init__(self, flat: Flat, lights, prefilter: float, spec=None):
        self.flat = flat
        self.scene = Scene(_device(), flat)
        self.lights = np.asarray(lights, np.float32)
        self.spec = spec
        self.opts = _lib.default_options(hierarchy=2, prefilter=prefilter, object_cov=flat.object_cov)
        self.buffers = {}

    def frame(self, w: int, h: int, n_lights: int) -> dict:
        key = (w, h, n_lights)
        if key not in self.buffers:
            px, dev = w * h, "cuda:0"
            self.buffers[key] = dict(
                hits=torch.zeros((px, 4), dtype=torch.int32, device=dev),
                recv=torch.zeros((px, 8), dtype=torch.float32, device=dev),
                vis=torch.zeros(px * n_lights, dtype=torch.float32, device=dev),
                full=torch.zeros(px * n_lights, dtype=torch.int64, device=dev),
                touched=torch.zeros(px * n_lights, dtype=torch.int64, device=dev))
        return self.buffers[key]


@functools.lru_cache(maxsize=None)
def _field():
    """The boulder field's 20,000 nearest boulders, for the view cache."""
    tris9, counts, pl, lights, eye, _ = boulder_field(count=20000)
    centre = lights[1:, 0:3] + 0.5 * (lights[1:, 4:7] + lights[1:, 8:11])
    near = 1 + np.argsort(np.linalg.norm(centre[:, :2] - eye[:2], axis=1))[:3]
    return dict(tris9=tris9, counts=counts, pl=pl, lights=np.ascontiguousarray(lights[[0, *near]]), eye=eye,
                surf=boulder_field_surface())


@functools.lru_cache(maxsize=None)
def _field_flat(movers: int) -> Flat:
    f = _field()
    return Flat.build_instanced(f["tris9"], f["counts"], f["pl"], object_prefilter=True,
                                movable=list(range(1, movers + 1)))


@functools.lru_cache(maxsize=None)
def _lightmap(texel: float, boxes: int):
    sc = lit_room(boxes=boxes, size=2.0)
    dyn = sc.notes["dynamic"]
    tris9, counts = meshes_to_arrays(sc.meshes)
    return sc, dyn, tris9, counts, Lightmap.from_meshes(sc.meshes, texel, lambda m: not dyn[m])


@functools.lru_cache(maxsize=None)
def _flat(name: str):
    sc = {"room": room_scene, "rock": rock_field, "courtyard": courtyard}[name]()
    return sc, Flat.build_arrays(*meshes_to_arrays(sc.meshes))


@functools.lru_cache(maxsize=None)
def _world(name: str) -> World:
    if name == "boulders":
        tris9, counts, pl, lights, _, _ = boulder_field()
        return World(Flat.build_instanced(tris9, counts, pl, object_prefilter=True), lights, 1.0)
    sc, flat = _flat(name.split()[0])
    w = World(flat, sc.lights, sc.prefilter, sc)
    if name == "courtyard moving":  # the rest pose, and which of its triangles hang in a curtain
        w.rest = _gpu(w.flat.tris)
        w.curtain = torch.cat([torch.arange(int(f), int(f) + int(c), device="cuda:0")
                               for f, c in (w.flat.ranges[m][:2] for m in sc.notes["curtains"])])
    return w


# ---- inputs


def _camera(world: str, rng, w: int, h: int, dolly: bool = False) -> np.ndarray:
    if world == "room":
        eye, tgt = (rng.uniform(0.3, 0.8), rng.uniform(0.3, 0.8), rng.uniform(1.2, 2.0)), (
            rng.uniform(3.0, 3.7), rng.uniform(3.0, 3.7), rng.uniform(0.4, 1.2))
    elif world == "rock":  # above the field, looking down into it
        ang, dist = rng.uniform(0, 2 * math.pi), rng.uniform(2.0, 8.0)
        tgt = np.array([rng.uniform(-8, 8), rng.uniform(-8, 8), 0.0])
        eye = tgt + [dist * math.cos(ang), dist * math.sin(ang), rng.uniform(12.0, 20.0)]
    elif world == "courtyard" and dolly:
        eye = (2.5 + rng.uniform(0.0, 0.1), 7.5 + rng.uniform(0.0, 0.1), 3.0)
        tgt = (22.0, 6.0 + rng.uniform(0.0, 0.2), 7.0)
    elif world == "courtyard":
        eye, tgt = random_pose(Pcg32(int(rng.integers(1 << 31)), 17))
    else:  # anywhere in the boulder field, as the served requests look
        eye = np.array([rng.uniform(-900, 900), rng.uniform(-900, 900), rng.uniform(1.5, 20.0)])
        ang, dist = rng.uniform(0, 2 * np.pi), rng.uniform(20.0, 200.0)
        tgt = eye + [np.cos(ang) * dist, np.sin(ang) * dist, -eye[2] + rng.uniform(0.0, 2.0)]
    return camera_uniform(eye, tgt, 60.0, w, h)


def _lights(world: World, name: str, n: int, rng) -> np.ndarray:
    """`n` lights: the world's own, and where it has fewer, rectangles more."""
    if name == "boulders":  # the sun and the nearest of a random place
        return np.ascontiguousarray(world.lights[[0, *(1 + rng.permutation(len(world.lights) - 1)[:n - 1])]])
    rows = [r.copy() for r in world.lights[:n]]
    while len(rows) < n:
        if name == "room":
            x, y, s = rng.uniform(0.5, 3.0), rng.uniform(1.0, 3.5), rng.uniform(0.2, 0.6)
            rows.append(rect_light([x, y, 2.9], [s, 0, 0], [0, -s, 0], one_sided=True))
        else:
            rows.append(random_rect_light(Pcg32(int(rng.integers(1 << 31)), 17)))
    return np.stack(rows)


def _points(world: World, n: int, rng) -> np.ndarray:
    """Shading points scattered over the world's triangles, a hair in front."""
    t = world.flat.tris[rng.integers(len(world.flat.tris), size=n)].reshape(n, 3, 4)[..., :3].astype(np.float64)
    a, b = rng.uniform(size=(2, n, 1))
    a, b = np.where(a + b > 1, 1 - a, a), np.where(a + b > 1, 1 - b, b)
    nrm = np.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
    nrm /= np.maximum(np.linalg.norm(nrm, axis=1, keepdims=True), 1e-30)
    out = np.zeros((n, 8), np.float32)
    out[:, 0:3] = t[:, 0] + a * (t[:, 1] - t[:, 0]) + b * (t[:, 2] - t[:, 0]) + 1e-4 * nrm
    out[:, 4:7] = nrm
    return out


def _box_moves(case: dict, seed: int) -> list:
    """Two poses of the lit room's first `moved` boxes: [(mesh, triangles)]."""
    sc, dyn, _, _, _ = _lightmap(case["texel"], case["boxes"])
    rng = np.random.default_rng(seed)
    movers = [i for i, d in enumerate(dyn) if d][:case["moved"]]
    poses = []
    for _ in range(2):
        moved = []
        for m in movers:
            shift = np.array([rng.uniform(-0.3, 0.3), rng.uniform(-0.3, 0.3), 0.0], np.float32)
            moved.append((m, (np.asarray(sc.meshes[m], np.float32).reshape(-1, 3, 3) + shift).reshape(-1, 9)))
        poses.append(moved)
    return poses


def _cache_keys(vc: ViewCache, objects: int, radius: float) -> np.ndarray:
    f = _field()
    keys = []
    for m in range(1, objects + 1):
        keys += vc.pages_of(m, int(f["pl"][m]["geometry"]), 0)
    gx, gy = vc.grid(0, 0, 1)
    texel, eye = 2100.0 / gx, f["eye"]
    at = lambda p: -1050.0 + (p * 8 + 4) * texel  # noqa: E731
    lo = [int((e - radius + 1050.0) / (8 * texel)) for e in eye[:2]]
    hi = [int((e + radius + 1050.0) / (8 * texel)) + 1 for e in eye[:2]]
    for py in range(max(lo[1], 0), min(hi[1], gy // 8) + 1):
        for px in range(max(lo[0], 0), min(hi[0], gx // 8) + 1):
            if math.hypot(at(px) - eye[0], at(py) - eye[1]) <= radius:
                keys.append(vc.key(0, 0, 1, px, py))
    return np.ascontiguousarray(keys, np.uint32)


def prepare(case: dict, seed: int) -> dict:
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("query", "points"):
        w = st["world"] = _world(case["world"])
        recv, lights = _points(w, case["n"], rng), _lights(w, case["world"], case["lights"], rng)
        if kind == "query":
            st.update(recv=recv, lights=lights)
        else:
            q = case["n"] * case["lights"]
            st.update(recv=_gpu(recv), lights=_gpu(lights), vis=torch.zeros(q, device="cuda:0"),
                      full=torch.zeros(q, dtype=torch.int64, device="cuda:0"),
                      touched=torch.zeros(q, dtype=torch.int64, device="cuda:0"))
    elif kind in ("view", "frame"):
        # (a frame moves its scene's curtains, so it has a courtyard of its own)
        w = st["world"] = _world(case["world"] + (" moving" if kind == "frame" else ""))
        st["camera"] = _gpu(_camera(case["world"], rng, case["w"], case["h"], kind == "frame"))
        st["lights"] = _gpu(_lights(w, case["world"], case["lights"], rng))
        st["frame"] = w.frame(case["w"], case["h"], case["lights"])
        if kind == "frame":  # the curtains swung across, by a sine of time and place
            v = w.rest[w.curtain].reshape(-1, 3, 4)
            amp = 0.15 * ((15.8 - v[..., 2]) / 5.2).clamp(0.0, 1.0)
            v[..., 1] += amp * torch.sin(1.3 * v[..., 0] + 0.9 * v[..., 2] + float(rng.uniform(0.0, 6.0)))
            pose = w.rest.clone()
            pose[w.curtain] = v.reshape(-1, 12)
            st["pose"] = pose
    elif kind == "sky":
        w = st["world"] = _world(case["world"])
        n = case["w"] * case["h"]
        cam = _gpu(_camera(case["world"], rng, case["w"], case["h"]))
        st["recv"] = torch.zeros((n, 8), device="cuda:0")
        hits = torch.zeros((n, 4), dtype=torch.int32, device="cuda:0")
        w.scene.primary_device(cam, case["w"], case["h"], _gpu(w.lights), w.opts, hits, st["recv"])
        st["out"] = torch.zeros(n, device="cuda:0")
        st["faces"] = torch.zeros(6 * n, device="cuda:0")
    elif kind == "batch":
        w = st["world"] = _world(case["world"])
        views, lights = [], []
        for k in range(case["views"]):  # each half the size of the one before, from the largest again after four
            vw = case["most"] >> (k % 4)
            vh, nl = vw * 9 // 16, 1 + (k + case["lights"] - 1) % case["lights"]
            views.append((_camera("courtyard", rng, vw, vh), vw, vh, len(lights), nl))
            lights += [random_rect_light(Pcg32(int(rng.integers(1 << 31)), 17)) for _ in range(nl)]
        st["batch"] = Batch(w.scene, views, np.stack(lights))
        st["tuning"] = Batch.tuning(tile_w=case["tile"])
    elif kind.startswith("cache"):
        f, movers = _field(), case.get("movers", 1)
        flat = _field_flat(movers)
        scene = st["scene"] = Scene(_device(), flat)
        lights = f["lights"].copy()
        lights[1:, 0:2] += rng.uniform(-2.0, 2.0, (len(lights) - 1, 2)).astype(np.float32)
        opts = _lib.default_options(hierarchy=2, prefilter=1.0, object_cov=flat.object_cov)
        vc = st["cache"] = ViewCache(scene, f["surf"], lights, opts, pages=16384, append_pages=8192,
                                     candidates=32768, base_texel=0.05)
        st["keys"] = _cache_keys(vc, case["objects"], case["radius"])
        if kind == "cache moves":
            vc.request(st["keys"])
            vc.frame()
            st["poses"] = [[(m, f["pl"][m]["rotation"], f["pl"][m]["translation"] + np.array(
                [rng.uniform(-0.25, 0.25), rng.uniform(-0.25, 0.25), 0.0], np.float32))
                for m in range(1, movers + 1)] for _ in range(2)]
            st["at"] = 0
    elif kind == "renderer":
        tris9, counts, pl, surf, lights, movable = vcache_world()
        lights = np.array(lights, np.float32, copy=True)
        lights[0, 0:2] += rng.uniform(-1.0, 1.0, 2).astype(np.float32)
        lights[0, 12:15] = [3.0, 2.5, 2.0]
        r = st["renderer"] = Renderer(_device(), (case["w"], case["h"]), tris9, counts, pl, surf, lights,
                                      RendererOptions(cache=True, movable=movable, pages=16384))
        st["camera"] = camera_uniform([rng.uniform(-7.5, -6.5), rng.uniform(-7.5, -6.5), 3.0], [2.0, 2.0, 0.0], 60.0,
                                      case["w"], case["h"])
        st["moves"] = [pl[movable[0]]["translation"] + np.array([dx, dy, 0.0], np.float32)
                       for dx, dy in rng.uniform(-0.2, 0.2, (2, 2))]
        st["object"], st["rotation"], st["at"] = movable[0], pl[movable[0]]["rotation"], 0
        for _ in range(40):
            r.render(st["camera"])
            if r.is_settled(2):
                break
    else:
        sc, dyn, tris9, counts, lm = _lightmap(case["texel"], case["boxes"])
        scene = Scene(_device(), Flat.build_arrays(tris9, counts))
        st["cache"] = LiveLightmap(scene, lm.texels, lm.blocks, sc.lights[0], dyn)
        st["poses"], st["at"] = _box_moves(case, seed), 0
    return st


# ---- one pass


def run(st: dict):
    case, kind = st["case"], st["case"]["kind"]
    if kind == "query":
        vis, full, touched, _ = st["world"].scene.query(st["recv"], st["lights"], st["world"].opts)
        return dict(vis=vis, full=full.view(np.int64), touched=touched.view(np.int64))
    if kind == "points":
        st["world"].scene.query_device(st["recv"], st["lights"], st["world"].opts, st["vis"], st["full"],
                                       st["touched"])
        return dict(vis=st["vis"], full=st["full"], touched=st["touched"])
    if kind in ("view", "frame"):
        w, f = st["world"], st["frame"]
        if kind == "frame":
            w.scene.refit_device(st["pose"])
        w.scene.primary_device(st["camera"], case["w"], case["h"], st["lights"], w.opts, f["hits"], f["recv"])
        w.scene.view_query_device(f["recv"], case["w"], case["h"], st["lights"], w.opts, f["vis"], f["full"],
                                  f["touched"], tile_w=case["tile"])
        return f
    if kind == "sky":
        st["world"].scene.sky_view_device(st["recv"], case["w"], case["h"], st["world"].opts, st["out"], st["faces"],
                                          tile_w=case["tile"])
        return dict(out=st["out"], faces=st["faces"])
    if kind == "batch":
        b = st["batch"]
        b.run(st["world"].opts, st["tuning"])
        return [[x.view(np.int64) if x.dtype == np.uint64 else x.view(np.int32) if x.dtype == np.uint32 else x
                 for x in b.read(k)] for k in range(len(b.shapes))]
    if kind == "cache bake":
        vc = st["cache"]
        vc.evict(st["keys"])
        vc.request(st["keys"])
        vc.frame()
        return vc.read(st["keys"])[0]
    if kind == "cache moves":
        vc, scene = st["cache"], st["scene"]
        st["at"] ^= 1
        for m, rot, pos in st["poses"][st["at"]]:
            scene.set_transform(m, rot, pos)
        scene.apply_moves()
        vc.set_moved(scene.last_moves())
        vc.request(st["keys"])
        vc.frame()
        return vc.read(st["keys"])[0]
    if kind == "renderer":
        st["at"] ^= 1
        st["renderer"].set_transform(st["object"], st["rotation"], st["moves"][st["at"]])
        st["renderer"].render(st["camera"])
        return st["renderer"].read_colors()
    st["at"] ^= 1
    st["cache"].update_meshes(st["poses"][st["at"]])
    return st["cache"].read_texels()


# ---- what a pass cannot do without, and how far two may be apart


def _cones(case: dict) -> tuple:
    """(cones, the world whose walk they take, bytes of results)."""
    kind = case["kind"]
    if kind in ("query", "points"):
        return case["n"] * case["lights"], case["world"], 20
    if kind in ("view", "frame"):
        return case["w"] * case["h"] * case["lights"], case["world"], 20
    if kind == "sky":
        return 6 * case["w"] * case["h"], "rock sky" if case["world"] == "rock" else "room", 4
    if kind == "batch":
        px = [(case["most"] >> (k % 4)) * ((case["most"] >> (k % 4)) * 9 // 16) for k in range(case["views"])]
        return sum(p * (1 + (k + case["lights"] - 1) % case["lights"]) for k, p in enumerate(px)), "courtyard", 20
    if kind.startswith("cache"):  # 8 x 8 texels a page, four lights; a move reaches about a tenth
        pages = 37 * case["objects"] + math.pi * case["radius"] ** 2 / 0.64
        return 256 * pages * (1.0 if kind == "cache bake" else 0.1), "field" + kind[5:].replace(" bake", ""), 4
    if kind == "renderer":  # about what one move re-bakes
        return 2000, "yard", 4
    return 60.0 / case["texel"] ** 2 * 0.1, "room", 4


def work(case: dict) -> dict:
    cones, world, out = _cones(case)
    n = WORK[world]
    points = cones / case.get("lights", 1) if case["kind"] != "sky" else cones / 6
    walked = 32 * n[0] + 32 * n[1] + 36 * n[2] + 20 * n[4] + 108 * n[5]
    scene = {"room": 2.2e6, "rock": 1.0e8, "courtyard": 3.0e8, "boulders": 5.0e7, "field": 5.0e7,
             "yard": 1.0e5}[world.split()[0]]
    total = cones * out + points * 32 + min(scene, cones * walked)
    if case["kind"] == "frame":  # the pose read, leaves, boxes and coverage written
        total += 3048756 * (48 + 36) + 1.03e6 * 140
    return {"bytes": float(total), "flops": float(cones * (QUERY_FLOPS + sum(a * b for a, b in zip(FLOPS, n))))}


def tolerance(case: dict):
    """Every walk's arithmetic is fixed, so results are the same bit for bit,
    except where a walk stops at its cap of nodes: what it has met by then
    depends on which queries share its packet. In the courtyard 4% of the
    walks do (and some from odd corners of the boulder field); 16 x 4 against
    8 x 8 tiles change its view by 2.7e-3 relative and 2e-4 of its masks."""
    if case["world"] in ("courtyard", "boulders"):
        return {"rel": 1e-2, "max": 0.99, "differ": 1e-3}
    return "exact"


# ---- the room's cases again in 64 bits, over every triangle

F64 = torch.float64


def _clip(poly, count, keep):
    """Convex polygons (k, v, 3) of `count` vertices, cut to keep(x) >= 0 (a
    linear function); one vertex more at most."""
    k, v, _ = poly.shape
    i = torch.arange(v, device=poly.device)[None].expand(k, v)
    nxt = torch.where(i + 1 < count[:, None], i + 1, torch.zeros_like(i))
    d = keep(poly)
    e = torch.gather(d, 1, nxt)
    b = torch.gather(poly, 1, nxt[..., None].expand(k, v, 3))
    live = i < count[:, None]
    cross = live & ((d >= 0) != (e >= 0))
    cut = poly + (b - poly) * (d / torch.where(cross, d - e, torch.ones_like(d)))[..., None]
    pts = torch.stack([poly, cut], 2).reshape(k, 2 * v, 3)
    flag = torch.stack([live & (d >= 0), cross], 2).reshape(k, 2 * v)
    at = torch.argsort((~flag).to(torch.int8), dim=1, stable=True)[:, :v + 1]
    return torch.gather(pts, 1, at[..., None].expand(k, v + 1, 3)), flag.sum(1)


def _lambert(normal, poly, count):
    """Lambert's edge integrals of polygons of directions: |1/2 sum|."""
    k, v, _ = poly.shape
    i = torch.arange(v, device=poly.device)[None].expand(k, v)
    nxt = torch.where(i + 1 < count[:, None], i + 1, torch.zeros_like(i))
    b = torch.gather(poly, 1, nxt[..., None].expand(k, v, 3))
    a = poly / poly.norm(dim=-1, keepdim=True).clamp_min(1e-300)
    b = b / b.norm(dim=-1, keepdim=True).clamp_min(1e-300)
    g = torch.linalg.cross(a, b)
    s = g.norm(dim=-1)
    term = torch.atan2(s, (a * b).sum(-1)) * (normal[:, None] * g).sum(-1) / s.clamp_min(1e-300)
    return 0.5 * torch.where((i < count[:, None]) & (s > 1e-14), term, torch.zeros_like(term)).sum(1).abs()


def _above(normal, quad):
    """A quad of directions' weight, cut to the horizon of `normal`."""
    n = torch.full((len(quad),), 4, device=quad.device)
    poly, n = _clip(quad, n, lambda x: (x * normal[:, None]).sum(-1))
    w = _lambert(normal, poly, n)
    return torch.where(n >= 3, w, torch.zeros_like(w))


def _dirs(c, s, t):
    """Directions of the window's (s, t) in [0, 1], (n, len(s), 3)."""
    u = c["w"][:, 0:1] + s[None] * (c["w"][:, 2:3] - c["w"][:, 0:1])
    v = c["w"][:, 1:2] + t[None] * (c["w"][:, 3:4] - c["w"][:, 1:2])
    return c["fwd"][:, None] + c["right"][:, None] * u[..., None] + c["up"][:, None] * v[..., None]


def _corners(c, lo_s, hi_s, lo_t, hi_t):
    f = lambda *a: torch.tensor(a, dtype=F64, device=c["apex"].device)  # noqa: E731
    return _dirs(c, f(lo_s, hi_s, hi_s, lo_s), f(lo_t, lo_t, hi_t, hi_t))


def _coverage(c, tris, mesh, n_mesh: int, sky: bool):
    """The 64 bins' coverage of cones `c` by triangles (t, 3, 3) of `mesh`:
    each mesh's projected area a bin, meshes by the maximum (a sky's as
    independent occluders)."""
    dev, n = tris.device, len(c["apex"])
    cov = torch.zeros((n, n_mesh, 64), dtype=F64, device=dev)
    nrm = torch.linalg.cross(tris[:, 1] - tris[:, 0], tris[:, 2] - tris[:, 0])
    side = torch.stack([c["right"] - c["w"][:, 0:1] * c["fwd"], c["w"][:, 2:3] * c["fwd"] - c["right"],
                        c["up"] - c["w"][:, 1:2] * c["fwd"], c["w"][:, 3:4] * c["fwd"] - c["up"], c["fwd"]], 1)
    corner = _corners(c, 0.0, 1.0, 0.0, 1.0)
    for i0 in range(0, n, 96):
        s = slice(i0, min(i0 + 96, n))
        apex = c["apex"][s]
        keep = (apex @ nrm.T - (nrm * tris[:, 0]).sum(-1)[None] > 0) & c["on"][s, None]
        keep &= ~((corner[s].reshape(-1, 3) @ nrm.T).reshape(-1, 4, len(tris)) >= 0).all(1)
        planes = side[s].reshape(-1, 3)
        value = (planes @ tris.reshape(-1, 3).T).reshape(len(apex), 5, len(tris), 3)
        value -= (side[s] * apex[:, None]).sum(-1)[:, :, None, None]
        value[:, 4] -= 1e-4
        keep &= ~(value < 0).all(-1).any(1)
        if sky:
            up = (c["horizon"][s] @ tris.reshape(-1, 3).T).reshape(len(apex), len(tris), 3)
            keep &= (up - (c["horizon"][s] * apex).sum(-1)[:, None, None] >= 0).any(-1)
        else:
            deep = (c["fwd"][s] @ tris.reshape(-1, 3).T).reshape(len(apex), len(tris), 3)
            keep &= (deep <= c["far"][s][:, None, None]).any(-1)
        del value
        for pair in torch.split(keep.nonzero(), 40000):
            q, t = pair[:, 0] + i0, pair[:, 1]
            poly, cnt = tris[t], torch.full((len(t),), 3, device=dev)
            poly = poly - c["apex"][q][:, None]
            poly = torch.stack([(poly * c[k][q][:, None]).sum(-1) for k in ("right", "up", "fwd")], -1)
            if not sky:
                depth = c["far"][q] - (c["fwd"][q] * c["apex"][q]).sum(-1)
                poly, cnt = _clip(poly, cnt, lambda x: depth[:, None] - x[..., 2])
            poly, cnt = _clip(poly, cnt, lambda x: x[..., 2] - 1e-4)
            w = c["w"][q]
            z = poly[..., 2].clamp_min(1e-4)
            x = (poly[..., 0] / z - w[:, 0:1]) * 8 / (w[:, 2:3] - w[:, 0:1])
            y = (poly[..., 1] / z - w[:, 1:2]) * 8 / (w[:, 3:4] - w[:, 1:2])
            v = torch.arange(poly.shape[1], device=dev)[None].expand(x.shape)
            nxt = torch.where(v + 1 < cnt[:, None], v + 1, torch.zeros_like(v))
            x1, y1 = torch.gather(x, 1, nxt), torch.gather(y, 1, nxt)
            # an edge's part in each row, and the length of each bin to its right there
            g = torch.arange(8, dtype=F64, device=dev)
            lo, hi = torch.minimum(y, y1)[..., None], torch.maximum(y, y1)[..., None]
            ya, yb = torch.maximum(lo, g), torch.minimum(hi, g + 1)
            slope = ((x1 - x) / torch.where(y1 == y, torch.ones_like(y), y1 - y))[..., None]
            xa, xb = x[..., None] + (ya - y[..., None]) * slope, x[..., None] + (yb - y[..., None]) * slope
            ra, rb = g + 1 - xa[..., None], g + 1 - xb[..., None]
            area = lambda r: torch.where(r > 1, r - 0.5, 0.5 * r.clamp(0.0, 1.0) ** 2)  # noqa: E731
            flat = (rb - ra).abs() < 1e-9
            mean = torch.where(flat, (0.5 * (ra + rb)).clamp(0.0, 1.0),
                               (area(rb) - area(ra)) / torch.where(flat, torch.ones_like(ra), rb - ra))
            part = mean * (yb - ya).clamp_min(0.0)[..., None] * torch.where(y1 > y, 1.0, -1.0)[..., None, None]
            part = torch.where(((v < cnt[:, None]) & (cnt[:, None] >= 3))[..., None, None], part,
                               torch.zeros_like(part)).sum(1)
            cov.view(-1, 64).index_add_(0, q * n_mesh + mesh[t], part.reshape(-1, 64))
    cov = cov.abs()
    cov = torch.where(cov >= 1.0 - 1e-5, torch.ones_like(cov), cov)
    cov = torch.where(cov > 1e-6, cov, torch.zeros_like(cov))
    return 1.0 - (1.0 - cov).prod(1) if sky else cov.max(1).values


def _bins(c, normal, cov):
    """The covered weight: each bin's Lambert weight above the horizon times its coverage."""
    blocked = torch.zeros(len(normal), dtype=F64, device=normal.device)
    for b in range(64):
        quad = _corners(c, (b % 8) / 8, (b % 8 + 1) / 8, (b // 8) / 8, (b // 8 + 1) / 8)
        blocked += cov[:, b] * _above(normal, quad)
    return blocked


def _rect64(recv, row, tris, mesh, n_mesh: int):
    """The irradiance per unit radiance of receivers (n, 8) from a rect light
    row past the triangles."""
    p, nrm = recv[:, 0:3], recv[:, 4:7]
    corner, eu, ev = row[0:3], row[4:7], row[8:11]
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)  # noqa: E731
    fwd = unit(torch.linalg.cross(eu, ev))[None].expand(len(p), 3)
    on = (recv[:, 7] >= 0) & (((corner + 0.5 * (eu + ev) - p) * nrm).sum(-1) > 0)
    if float(row[3]) > 0.5:
        on &= ((p - corner) * fwd).sum(-1) > 0
    fwd = torch.where((((corner - p) * fwd).sum(-1) < 0)[:, None], -fwd, fwd)
    dist = ((corner - p) * fwd).sum(-1)
    on &= dist > 1e-6
    dist = torch.where(on, dist, torch.ones_like(dist))
    right = unit(eu)[None].expand(len(p), 3)
    up = torch.linalg.cross(fwd, right)
    rel = corner - p
    quad = torch.stack([rel, rel + eu, rel + eu + ev, rel + ev], 1)
    uv = torch.stack([(quad * right[:, None]).sum(-1), (quad * up[:, None]).sum(-1)], -1) / dist[:, None, None]
    lo, hi = uv.min(1).values, uv.max(1).values
    mid = unit(torch.cat([0.5 * (lo + hi), torch.ones_like(lo[:, :1])], 1))
    ends = torch.stack([torch.stack([a[:, 0], b[:, 1], torch.ones_like(a[:, 0])], -1) for a in (lo, hi) for b in (lo, hi)], 1)
    wide = ((hi - lo) > 8.0).any(1) & ((unit(ends) * mid[:, None]).sum(-1).min(1).values < 0.8660254)
    foot = torch.minimum(torch.maximum(torch.zeros_like(lo), lo), hi)
    cut = wide[:, None] & ((hi - lo) > 8.0)
    kept = torch.minimum(torch.maximum(foot - 4.0, lo), hi - 8.0)
    lo, hi = torch.where(cut, kept, lo), torch.where(cut, kept + 8.0, hi)
    c = dict(apex=p, right=right, up=up, fwd=fwd, w=torch.cat([lo, hi], 1), on=on,
             far=(fwd * p).sum(-1) + dist * (1.0 - 1e-5))
    cov = _coverage(c, tris, mesh, n_mesh, False)
    window = _above(nrm, _corners(c, 0.0, 1.0, 0.0, 1.0))
    value = (window - _bins(c, nrm, cov)).clamp_min(0.0)
    open_ = _above(nrm, quad)
    value = torch.where(wide, torch.where(window > 1e-9, value / window.clamp_min(1e-9), torch.ones_like(value)) * open_,
                        value)
    return torch.where(on, value, torch.zeros_like(value))


def _sky64(recv, tris, mesh, n_mesh: int):
    p, nrm = recv[:, 0:3], recv[:, 4:7]
    out = []
    for f in range(6):
        axis, sign = f // 2, -1.0 if f % 2 else 1.0
        e = torch.eye(3, dtype=F64, device=p.device)
        fwd = (sign * e[axis])[None].expand(len(p), 3)
        right = e[(axis + 1) % 3][None].expand(len(p), 3)
        w = torch.tensor([-1.0, -1.0, 1.0, 1.0], dtype=F64, device=p.device)[None].expand(len(p), 4)
        c = dict(apex=p, right=right, up=torch.linalg.cross(fwd, right), fwd=fwd, w=w, horizon=nrm)
        window = _corners(c, 0.0, 1.0, 0.0, 1.0)
        c["on"] = (recv[:, 7] >= 0) & ((window * nrm[:, None]).sum(-1) > 0).any(1)
        v = (_above(nrm, window) - _bins(c, nrm, _coverage(c, tris, mesh, n_mesh, True))).clamp_min(0.0)
        out.append(torch.where(c["on"], v, torch.zeros_like(v)))
    return torch.stack(out)


def _rays64(camera, w: int, h: int, lights, tris):
    """Receivers (w * h, 8) of a camera's nearest front-facing hits."""
    cam = _gpu(camera.cpu().numpy()).to(F64)
    y, x = torch.meshgrid(torch.arange(h, device=cam.device), torch.arange(w, device=cam.device), indexing="ij")
    sx = ((x.reshape(-1) + 0.5) / w * 2 - 1) * cam[18] * (w / h)
    sy = (1 - (y.reshape(-1) + 0.5) / h * 2) * cam[18]
    d = cam[4:7] + cam[8:11] * sx[:, None] + cam[12:15] * sy[:, None]
    d = d / d.norm(dim=-1, keepdim=True)
    eye = cam[0:3]
    e1, e2 = tris[:, 1] - tris[:, 0], tris[:, 2] - tris[:, 0]
    nrm = torch.linalg.cross(e1, e2)
    s = eye - tris[:, 0]
    q = torch.linalg.cross(s, e1)
    recv = torch.zeros((w * h, 8), dtype=F64, device=cam.device)
    for i0 in range(0, w * h, 2048):
        r = d[i0:i0 + 2048]
        det = -(r @ nrm.T)
        u = -(r @ torch.linalg.cross(s, e2).T) / det
        v = (r @ q.T) / det
        t = ((e2 * q).sum(-1)[None] / det)
        ok = (det > 1e-12) & (u >= -1e-5) & (v >= -1e-5) & (u <= 1 + 1e-5) & (u + v <= 1 + 1e-5) & (t > 0)
        t, at = torch.where(ok, t, torch.full_like(t, 3.4e38)).min(1)
        n = nrm[at] / nrm[at].norm(dim=-1, keepdim=True)
        lit = t < 1e38
        for row in lights:  # one-sided rects hide what is behind them
            facing = (r * torch.linalg.cross(row[4:7], row[8:11])).sum(-1)
            tl = ((row[0:3] - eye) * torch.linalg.cross(row[4:7], row[8:11])).sum() / facing
            on = eye + r * tl[:, None] - row[0:3]
            a, b = (on @ row[4:7]) / (row[4:7] @ row[4:7]), (on @ row[8:11]) / (row[8:11] @ row[8:11])
            lit &= ~((facing < 0) & (tl > 0) & (tl < t) & (a >= 0) & (a <= 1) & (b >= 0) & (b <= 1))
        point = eye + r * t[:, None] + n * (2e-6 * t).clamp_min(1e-4)[:, None]
        zero = torch.zeros_like(point)
        part = recv[i0:i0 + 2048]
        part[:, 0:3], part[:, 4:7] = torch.where(lit[:, None], point, zero), torch.where(lit[:, None], n, zero)
        part[:, 7] = torch.where(lit, 0.0, -1.0)
    return recv


def exact(case: dict, seed: int):
    if case["world"] not in ("room", "lit room"):
        return None
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "lightmap":
        sc, _, _, _, lm = _lightmap(case["texel"], case["boxes"])
        meshes = [np.asarray(m, np.float64).reshape(-1, 3, 3) for m in sc.meshes]
        for m, t in st["poses"][1]:
            meshes[m] = np.asarray(t, np.float64).reshape(-1, 3, 3)
        tris = _gpu(np.concatenate(meshes))
        mesh = _gpu(np.repeat(np.arange(len(meshes)), [len(m) for m in meshes]))
        texels = _gpu(lm.texels).to(F64)
        real = (texels[:, 4:7] != 0).any(1)
        v = torch.zeros(len(texels), dtype=F64, device=texels.device)
        v[real] = _rect64(texels[real], _gpu(sc.lights[0]).to(F64), tris, mesh, len(meshes))
        return v
    flat = st["world"].flat
    tris = _gpu(flat.tris.reshape(-1, 3, 4)[..., :3]).to(F64)
    mesh = _gpu(np.repeat(np.arange(len(flat.ranges)), flat.ranges[:, 1].astype(np.int64)))
    if kind == "sky":
        faces = _sky64(st["recv"].to(F64), tris, mesh, len(flat.ranges))
        return dict(out=faces.sum(0), faces=faces.reshape(-1))
    lights = (_gpu(st["lights"]) if kind == "query" else st["lights"]).to(F64)
    if kind == "view":
        recv = _rays64(st["camera"], case["w"], case["h"], lights, tris)
    else:
        recv = (_gpu(st["recv"]) if kind == "query" else st["recv"]).to(F64)
    vis = torch.cat([_rect64(recv, row, tris, mesh, len(flat.ranges)) for row in lights])
    out = dict(vis=vis, full=None, touched=None)
    if kind == "view":
        out.update(recv=recv, hits=None)
    return out
