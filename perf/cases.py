"""What this renderer is timed on: the work a program has it do, through rtxamd.

A case is a dict of plain values.  `kind` names the path:

  rays     a batch of closest-hit or occlusion queries on host arrays
  render   an image with the plain method
  cache    an image with the irradiance cache, built by its prepare frames
  adrrs    a frame with the cache, the pixel estimate, then roulette and splitting
  guided   recording frames with a guiding update each, then guided frames
  learned  frames that end into the learned radiance cache and train it
  network  the learned cache's network alone: gradients of a batch, then queries
  serve    jobs of several scenes and methods through the serving pool

Every size comes from the benchmark, the tests or the scene generators.
"""
import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "rtx-pathtracer_amd"))

import rtxamd  # noqa: E402
from rtxamd import abi  # noqa: E402

RESET = abi.RTX_FRAME_RESET_ACCUM
SCENES = {"cornell": abi.SCENE_CORNELL, "room": abi.SCENE_ROOM, "plates": abi.SCENE_PLATES, "spot": abi.SCENE_SPOT}
# triangles of the scenes with a fixed geometry, for work()
FIXED_TRIANGLES = {"cornell": 36, "plates": 12, "spot": 26, "gallery": 5000}


def listed():
    return [
        # a picking or probe query: a few thousand rays, the call's own latency
        {"name": "rays_probe", "kind": "rays", "query": "noalloc", "triangles": 12512, "rays": 2047},
        # a baker's or a sensor simulation's batch of incoherent closest hits
        {"name": "rays_closest", "kind": "rays", "query": "closest", "triangles": 262144, "rays": 1000003},
        # visibility of lamps from points all over the scene
        {"name": "rays_occluded", "kind": "rays", "query": "occluded", "triangles": 40000, "rays": 200001},
        # a preview of a small scene: launches and short queues
        {"name": "cornell_preview", "kind": "render", "scene": "cornell", "triangles": 0, "width": 256, "height": 256,
         "spp": 4, "depth": 8, "rr": False, "num_nee": 1, "mis": True, "nee": True, "samples_per_frame": 1},
        # the benchmark's image with the plain method, four of its 64 samples
        {"name": "room_plain", "kind": "render", "scene": "room", "triangles": 262144, "width": 1920, "height": 1080,
         "spp": 4, "depth": 12, "rr": False, "num_nee": 1, "mis": True, "nee": True, "samples_per_frame": 1},
        # the benchmark's image with its own method, at the same ratio of prepare frames to samples
        {"name": "room_cache", "kind": "cache", "triangles": 262144, "width": 1920, "height": 1080, "records": 10000,
         "prepare_frames": 20, "spp": 24, "depth": 12, "gradients": False},
        # textures, the alpha test and an environment map, odd size, roulette and several light samples
        {"name": "gallery_odd", "kind": "render", "scene": "gallery", "triangles": 0, "width": 641, "height": 363,
         "spp": 8, "depth": 6, "rr": True, "num_nee": 2, "mis": True, "nee": True, "samples_per_frame": 1},
        # adjoint-driven roulette and splitting on a small image
        {"name": "cornell_adrrs", "kind": "adrrs", "scene": "cornell", "triangles": 0, "width": 256, "height": 192,
         "records": 3000, "prepare_frames": 4, "spp": 4, "depth": 8},
        # online guiding of the benchmark's spot room: training frames, then the image
        {"name": "spot_guided", "kind": "guided", "scene": "spot", "triangles": 0, "width": 640, "height": 360,
         "region_splits": 8, "train_frames": 6, "spp": 10, "depth": 12},
        # the learned cache on the benchmark's image
        {"name": "room_learned", "kind": "learned", "triangles": 262144, "width": 1920, "height": 1080,
         "train_frames": 8, "spp": 8, "depth": 12},
        # its network alone at the default size: one training batch's gradients and a batch of queries
        {"name": "network", "kind": "network", "log2_table": 19, "train_rows": 16384, "rows": 300007},
        # a burst of requests over resident scenes, cache and guiding lookups among them
        {"name": "serve_burst", "kind": "serve", "scenes": 3, "jobs": 8, "largest": 512, "spp": 16, "triangles": 60000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _room(t):
    """The room generator's nearest valid triangle count: 20 + a multiple of 4, at least 124."""
    return 20 + 4 * ((max(124, int(t)) - 20) // 4)


def draw(rng):
    kind = rng.choice(["rays", "rays", "render", "render", "render", "cache", "cache", "adrrs", "guided", "learned",
                       "network", "serve"])
    if kind == "rays":
        query = rng.choice(["noalloc", "closest", "occluded"])
        return {"kind": kind, "query": query, "triangles": _room(_log(rng, 1000, 262144)),
                "rays": _log(rng, 1000, 65536 if query == "noalloc" else 1000000) | 1}
    width = _log(rng, 130, 1920)
    height = max(64, int(width * rng.choice([0.5625, 0.75, 1.0]))) + rng.randrange(7)
    height = min(height, 1080)
    if kind == "render":
        scene = rng.choice(["cornell", "room", "room", "plates", "gallery"])
        spp = max(1, min(16, int(8e6 / (width * height))))
        return {"kind": kind, "scene": scene, "triangles": _room(_log(rng, 10000, 262144)) if scene == "room" else 0,
                "width": width, "height": height, "spp": rng.randint(1, spp), "depth": rng.randint(4, 12),
                "rr": rng.random() < 0.3, "num_nee": rng.choice([1, 1, 2, 4]), "mis": rng.random() < 0.8,
                "nee": rng.random() < 0.9, "samples_per_frame": rng.choice([1, 1, 1, 2])}
    if kind == "cache":
        return {"kind": kind, "triangles": _room(_log(rng, 10000, 262144)), "width": width, "height": height,
                "records": _log(rng, 1000, 20000), "prepare_frames": rng.randint(4, 20), "spp": rng.randint(2, 20),
                "depth": rng.randint(6, 12), "gradients": rng.random() < 0.5}
    if kind == "adrrs":
        return {"kind": kind, "scene": rng.choice(["cornell", "spot"]), "triangles": 0, "width": min(width, 640),
                "height": min(height, 480), "records": _log(rng, 1000, 6000), "prepare_frames": rng.randint(2, 6),
                "spp": rng.randint(1, 6), "depth": rng.randint(4, 10)}
    if kind == "guided":
        return {"kind": kind, "scene": rng.choice(["spot", "plates"]), "triangles": 0, "width": min(width, 900),
                "height": min(height, 600), "region_splits": rng.randint(3, 8), "train_frames": rng.randint(1, 6),
                "spp": rng.randint(1, 16), "depth": rng.randint(6, 12)}
    if kind == "learned":
        return {"kind": kind, "triangles": _room(_log(rng, 10000, 262144)), "width": width, "height": height,
                "train_frames": rng.randint(4, 8), "spp": rng.randint(1, 8), "depth": rng.randint(6, 12)}
    if kind == "network":
        return {"kind": kind, "log2_table": rng.randint(14, 19), "train_rows": _log(rng, 256, 16384) | 1,
                "rows": _log(rng, 1000, 600000) | 1}
    return {"kind": kind, "scenes": rng.randint(1, 3), "jobs": rng.randint(2, 8), "largest": _log(rng, 192, 512),
            "spp": rng.randint(2, 16), "triangles": _room(_log(rng, 10000, 60000))}


# ------------------------------------------------------------------ scenes
def _quad(s, p, material, texcoords=None):
    s.add_mesh(np.array(p, np.float32), np.array([[0, 1, 2], [0, 2, 3]], np.uint32), material, texcoords=texcoords)


def _gallery(seed):
    """An environment-lit yard: textured boxes on a floor, leaves whose texture's alpha cuts them out, and a lamp."""
    rng = np.random.default_rng([seed, 1])
    s = rtxamd.HostScene.new()
    lamp = s.add_material(rtxamd.light((6.0, 6.0, 6.0)))
    floor = s.add_material(rtxamd.diffuse((0.5, 0.5, 0.5)))
    bricks = s.add_texture(np.concatenate([rng.integers(60, 255, (64, 64, 3)), np.full((64, 64, 1), 255)], 2)
                           .astype(np.uint8))
    y, x = np.mgrid[0:64, 0:64]
    leaf_rgba = np.stack([np.full_like(x, 40), 120 + x, np.full_like(x, 50),
                          np.where((x - 32) ** 2 + (y - 32) ** 2 < 900, 255, 0)], 2).astype(np.uint8)
    leaves = s.add_texture(leaf_rgba)
    coat = rtxamd.phong((0.6, 0.6, 0.6), (0.3, 0.3, 0.3), 20.0)
    coat.textureIdDiffuse = bricks
    coat = s.add_material(coat)
    leaf = rtxamd.diffuse((0.9, 0.9, 0.9))
    leaf.textureIdDiffuse = leaves
    leaf = s.add_material(leaf)
    glass = s.add_material(rtxamd.dielectric(1.5))
    _quad(s, [(-0.5, -0.5, 4.0), (-0.5, 0.5, 4.0), (0.5, 0.5, 4.0), (0.5, -0.5, 4.0)], lamp)
    _quad(s, [(-9, -9, 0), (9, -9, 0), (9, 9, 0), (-9, 9, 0)], floor)
    faces = np.array([[0, 2, 6, 4], [1, 5, 7, 3], [0, 4, 5, 1], [2, 3, 7, 6], [0, 1, 3, 2], [4, 6, 7, 5]])
    corner = np.array([[i & 1, (i >> 1) & 1, (i >> 2) & 1] for i in range(8)], np.float32)
    uv4 = np.array([(0, 0), (1, 0), (1, 1), (0, 1)], np.float32)
    pos, uvs = [], []
    for _ in range(200):
        lo = np.array([*rng.uniform(-8, 8, 2), 0.0])
        size = rng.uniform(0.1, 0.6, 3)
        pos.append((lo + corner[faces.reshape(-1)] * size).reshape(-1, 3))
        uvs.append(np.tile(uv4, (6, 1)))
    pos, uvs = np.concatenate(pos), np.concatenate(uvs)
    quads = np.arange(len(pos)).reshape(-1, 4)
    s.add_mesh(pos, np.concatenate([quads[:, [0, 1, 2]], quads[:, [0, 2, 3]]], 1).reshape(-1, 3), coat, texcoords=uvs)
    n = 1300
    centre = np.stack([rng.uniform(-8, 8, n), rng.uniform(-8, 8, n), rng.uniform(0.3, 3.0, n)], 1)
    a = rng.normal(size=(n, 3))
    a /= np.linalg.norm(a, axis=1, keepdims=True)
    b = np.cross(a, rng.normal(size=(n, 3)))
    b /= np.linalg.norm(b, axis=1, keepdims=True)
    r = rng.uniform(0.1, 0.3, (n, 1))
    pos = np.stack([centre - r * a - r * b, centre + r * a - r * b, centre + r * a + r * b, centre - r * a + r * b], 1)
    quads = np.arange(4 * n).reshape(-1, 4)
    s.add_mesh(pos.reshape(-1, 3), np.concatenate([quads[:, [0, 1, 2]], quads[:, [0, 2, 3]]], 1).reshape(-1, 3), leaf,
               texcoords=np.tile(uv4, (n, 1)))
    s.add_sphere((0.5, -3.0, 0.8), 0.6, glass)
    ey, ex = np.mgrid[0:64, 0:128]
    sky = np.stack([0.2 + 0.01 * ex, 0.3 + 0.02 * ey, 0.5 + 0.05 * (ex % 3), np.ones_like(ex)], -1).astype(np.float32)
    s.set_environment(sky, add_light=True)
    s.set_view((0.0, -9.0, 3.0), (0.0, 0.0, 0.8), (0.0, 0.0, 1.0), 50.0)
    return s.finalize()


def _scene(case, seed):
    if case.get("scene", "room") == "gallery":
        return _gallery(seed)
    name = case.get("scene", "room")
    return rtxamd.HostScene.generate(SCENES[name], seed, case["triangles"] if name == "room" else 0)


class State:
    """A renderer, its scene and what a pass needs; gives the device memory back with itself."""

    def __init__(self, case, seed):
        self.case, self.seed, self.others = case, seed, []
        self.renderer = rtxamd.Renderer(0)

    def upload(self, host):
        self.host, self.scene = host, self.renderer.upload(host)

    def params(self, spp, **kw):
        c = self.case
        kw = dict(dict(maxDepth=c["depth"], enableMIS=1, usePowerHeuristic=1, flags=RESET), **kw)
        return rtxamd.frame_params(self.host.camera(c["width"], c["height"]), c["width"], c["height"], spp,
                                   seed=self.seed + 1, **kw)

    def __del__(self):
        try:
            for other in self.others:
                other.close()
            if getattr(self, "scene", None):
                self.scene.close()
            self.renderer.close()
        except Exception:
            pass


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _rays(case, seed):
    """Rays that start all over the room: any direction, or towards a point of one of its four lamps."""
    rng = np.random.default_rng([seed, 2])
    n = case["rays"]
    org = rng.uniform((-9.9, 0.1, -9.9), (9.9, 9.9, 9.9), (n, 3))
    if case["query"] == "occluded":
        lamp = np.array([(x, 9.98, z) for x in (-5, 5) for z in (-5, 5)])[rng.integers(0, 4, n)]
        to = lamp + np.stack([rng.uniform(-1, 1, n), np.zeros(n), rng.uniform(-1, 1, n)], 1) - org
        length = np.linalg.norm(to, axis=1, keepdims=True)
        return rtxamd.rays_array(org, to / length, tmax=(length[:, 0] * 0.9999).astype(np.float32))
    d = rng.normal(size=(n, 3))
    return rtxamd.rays_array(org, d / np.linalg.norm(d, axis=1, keepdims=True))


def _prepare_rays(case, seed):
    s = State(case, seed)
    s.upload(rtxamd.HostScene.generate(abi.SCENE_ROOM, seed, case["triangles"]))
    s.rays = _rays(case, seed)
    return s


def _prepare_render(case, seed):
    s = State(case, seed)
    s.upload(_scene(case, seed))
    return s


def _prepare_cache(case, seed):
    s = State(case, seed)
    s.upload(_scene(case, seed))
    s.renderer.ic_create(case["records"])
    return s


def _prepare_adrrs(case, seed):
    return _prepare_cache(case, seed)


def _prepare_guided(case, seed):
    s = _prepare_render(case, seed)
    s.bounds = s.scene.bounds()
    return s


def _prepare_learned(case, seed):
    s = _prepare_render(case, seed)
    info = s.scene.info()
    s.renderer.nrc_create(list(info.boundsMin), list(info.boundsMax), seed=seed + 5)
    # an image under way: the cache has trained on its first frames
    s.renderer.render(s.scene, s.params(case["train_frames"], flags=RESET | abi.RTX_FRAME_NRC))
    return s


def _network(case, seed):
    """Parameters a cache may hold (values its BF16 copies keep whole), a training batch and queries in the room's box."""
    rng = np.random.default_rng([seed, 3])
    entries = 1 << case["log2_table"]
    grid = rng.random((16, entries, 2), np.float32)
    grid -= 0.5
    mlp = np.zeros(5 * 64 * 64 + 16 * 64, np.float32)
    b = math.sqrt(6.0 / 128)
    mlp[:5 * 4096] = rng.uniform(-b, b, 5 * 4096)
    mlp[5 * 4096:5 * 4096 + 192] = rng.uniform(-0.3, 0.3, 192)
    grid, mlp = (torch.from_numpy(v).bfloat16().float().numpy() for v in (grid, mlp))
    n = case["rows"] + case["train_rows"]
    x = np.zeros((n, 16), np.float32)
    x[:, 0:3] = rng.uniform((-10, 0, -10), (10, 10, 10), (n, 3))
    for c in (4, 8):
        v = rng.normal(size=(n, 3))
        x[:, c:c + 3] = v / np.linalg.norm(v, axis=1, keepdims=True)
    x[:, 3] = rng.uniform(0.05, 1, n)
    x[:, 12:15] = rng.uniform(0.1, 0.8, (n, 3))
    target = rng.uniform(0, 2, (case["train_rows"], 3)).astype(np.float32)
    return grid, mlp, x[:case["train_rows"]], target, x[case["train_rows"]:]


def _prepare_network(case, seed):
    s = State(case, seed)
    s.renderer.nrc_create((-10, 0, -10), (10, 10, 10), log2TableSize=case["log2_table"], seed=1)
    grid, mlp, s.train, s.target, s.queries = _network(case, seed)
    s.renderer.nrc_set_params(grid, mlp)
    return s


def _prepare_serve(case, seed):
    s = State(case, seed)
    rng = np.random.default_rng([seed, 4])
    s.jobs, scenes = [], []
    for k in range(case["scenes"]):
        host = rtxamd.HostScene.generate(abi.SCENE_ROOM, seed + k, _room(case["triangles"] // (1 << k)))
        scene, state = s.renderer.upload(host), rtxamd.Renderer(0)
        own = state.upload(host)
        camera = host.camera(128, 128)
        base = dict(seed=7, flags=RESET, maxDepth=8, enableMIS=1)
        state.ic_create(4000)
        state.render(own, rtxamd.frame_params(camera, 128, 128, 4, useIrradianceCache=1, isIrradiancePrepareFrame=1,
                                              irradianceCreateProb=0.01, **base))
        state.guiding_init(own.bounds(), 4)
        state.render(own, rtxamd.frame_params(camera, 128, 128, 2, updateGuiding=1, useGuiding=1, **base))
        s.others += [own, state, scene]
        scenes.append((host, scene, state))
    for k in range(case["jobs"]):
        host, scene, state = scenes[k % len(scenes)]
        side = max(64, case["largest"] >> (k % 3))
        width, height = side, side * 9 // 16 if k % 2 else side
        cached, guided = bool(k & 1), bool(k & 2)
        fp = rtxamd.frame_params(host.camera(width, height), width, height, max(1, case["spp"] >> (k % 2)),
                                 seed=int(rng.integers(1 << 30)), maxDepth=8 + k % 5, enableMIS=1,
                                 useIrradianceCache=int(cached), useGuiding=int(guided), guidingProb=0.5)
        s.jobs.append((scene, fp, state if cached or guided else None))
    s.server = rtxamd.Server(s.renderer, slotPaths=1 << 16, slots=16, framebufferBytes=1 << 28)
    s.others.insert(0, s.server)
    return s


# --------------------------------------------------------------------- run
def run(s):
    return globals()["_run_" + s.case["kind"]](s)


def _run_rays(s):
    r, query = s.renderer, s.case["query"]
    if query == "occluded":
        return r.trace_occluded(s.scene, s.rays)
    return (r.trace_closest_noalloc if query == "noalloc" else r.trace_closest)(s.scene, s.rays)


def _run_render(s):
    c = s.case
    s.renderer.render(s.scene, s.params(
        c["spp"], enableRR=int(c["rr"]), numNEE=c["num_nee"], enableNEE=int(c["nee"]), enableMIS=int(c["mis"]),
        samplesPerPixel=c["samples_per_frame"]))
    return s.renderer.read_image(c["width"], c["height"])


def _run_cache(s):
    c, r = s.case, s.renderer
    kw = dict(useIrradianceCache=1, useIrradianceGradients=int(c["gradients"]))
    r.ic_reset()
    r.render(s.scene, s.params(c["prepare_frames"], isIrradiancePrepareFrame=1, **kw))
    r.render(s.scene, s.params(c["spp"], sample_offset=c["prepare_frames"], **kw))
    return r.read_image(c["width"], c["height"])


def _run_adrrs(s):
    c, r = s.case, s.renderer
    n = c["prepare_frames"]
    cache = dict(useIrradianceCache=1, useIrradianceCacheOnGlossy=1)
    r.ic_reset()
    r.render(s.scene, s.params(n, isIrradiancePrepareFrame=1, irradianceCreateProb=0.02, irradianceUpdateProb=0.005,
                               **cache))
    r.render(s.scene, s.params(1, sample_offset=n, samplesPerPixel=16, numNEE=5, storeEstimate=1,
                               **dict(cache, maxDepth=1, maxFollowDiscrete=10)))
    r.render(s.scene, s.params(c["spp"], sample_offset=n + 1, useADRRS=1, adrrsS=5.0, adrrsSplit=1,
                               useIrradianceCacheOnGlossy=1))
    return r.read_image(c["width"], c["height"]), r.estimate_read(c["width"], c["height"])


def _run_guided(s):
    c, r = s.case, s.renderer
    r.guiding_init(s.bounds, c["region_splits"])
    r.render(s.scene, s.params(c["train_frames"], updateGuiding=1, useGuiding=1))
    r.render(s.scene, s.params(c["spp"], sample_offset=c["train_frames"], useGuiding=1))
    image = r.read_image(c["width"], c["height"])
    boxes, mixtures = r.guiding_get_wide()
    raw = np.frombuffer(b"".join(bytes(m) for m in mixtures), np.float32).reshape(len(mixtures), -1)
    first, lobes = abi.VmmThetaWide.pi.offset // 4, abi.RTX_MAX_LOBES
    used = raw[:, abi.VmmThetaWide.usedDistributions.offset // 4].view(np.int32)
    weights = np.where(np.arange(lobes) < used[:, None], raw[:, first:first + lobes], 0.0).astype(np.float32)
    return image, boxes, weights, used


def _run_learned(s):
    c, r = s.case, s.renderer
    r.render(s.scene, s.params(c["spp"], sample_offset=c["train_frames"], flags=RESET | abi.RTX_FRAME_NRC))
    return r.read_image(c["width"], c["height"])


def _run_network(s):
    loss, grid, mlp = s.renderer.nrc_gradients(s.train, s.target)
    return loss, grid, mlp, s.renderer.nrc_infer(s.queries)


def _run_serve(s):
    ids = [s.server.submit(scene, fp, state) for scene, fp, state in s.jobs]
    for i in ids:
        s.server.wait(i)
    return [s.server.read_image(i) for i in ids]


# -------------------------------------------------------------------- work
# Rays of a path on average (bounces, light samples), counted by the renderer
# on the listed scenes: the room's cached paths end after three bounces.
RAYS = {"render": 12.0, "cache": 4.5, "adrrs": 12.0, "guided": 14.0, "learned": 5.0, "serve": 9.0}
TRIANGLE_BYTES, RAY_BYTES, HIT_BYTES, PIXEL_BYTES = 36, 32, 16, 16


def _ray_flops(triangles):
    """Two boxes (3 slabs, 4 operations each) a level of a balanced tree, then one triangle's test."""
    return 24.0 * math.log2(max(2, triangles)) + 60.0


def work(case):
    kind = case["kind"]
    if kind == "rays":
        out = 1 if case["query"] == "occluded" else HIT_BYTES
        return {"bytes": case["rays"] * (RAY_BYTES + out) + case["triangles"] * TRIANGLE_BYTES,
                "flops": case["rays"] * _ray_flops(case["triangles"])}
    if kind == "network":
        layer, table = 2 * (5 * 64 * 64 + 64 * 3), (16 << case["log2_table"]) * 2
        rows, train = case["rows"], case["train_rows"]
        return {"bytes": rows * (64 + 12) + train * (64 + 12) + table * 2 + table * 4,
                "flops": layer * (rows + 3 * train)}
    if kind == "serve":
        paths = 0
        for k in range(case["jobs"]):
            side = max(64, case["largest"] >> (k % 3))
            paths += side * (side * 9 // 16 if k % 2 else side) * max(1, case["spp"] >> (k % 2))
        return {"bytes": paths / max(1, case["spp"]) * PIXEL_BYTES + case["triangles"] * 2 * TRIANGLE_BYTES,
                "flops": paths * RAYS[kind] * _ray_flops(case["triangles"])}
    pixels = case["width"] * case["height"]
    triangles = case["triangles"] or FIXED_TRIANGLES[case["scene"]]
    frames = case["spp"] * case.get("samples_per_frame", 1)
    frames += {"cache": case.get("prepare_frames", 0), "adrrs": case.get("prepare_frames", 0) + 16,
               "guided": case.get("train_frames", 0)}.get(kind, 0)
    return {"bytes": pixels * PIXEL_BYTES + triangles * TRIANGLE_BYTES,
            "flops": pixels * frames * RAYS[kind] * _ray_flops(triangles)}


def tolerance(case):
    kind = case["kind"]
    if kind == "rays":
        # against 64 bits: t 8e-8 off, u and v up to 6e-6; a ray within a rounding of an edge may find the neighbour
        return {"rel": 2e-5, "max": 0.05, "differ": 1e-4}
    if kind == "network":
        # with the encoding's sums rounded otherwise: 6e-5, and 0.013 at the worst entry, where a BF16 rounding flips
        return {"rel": 2e-3, "max": 0.1}
    # Images with every product rounded otherwise (no contraction into FMAs):
    # Cornell box 1e-6 and 3e-4 at the worst pixel, with splitting 9e-5 and
    # 0.03; the gallery 0.008 and the rooms 0.006 to 0.06, since a path whose
    # shading normal moves by a last bit goes elsewhere.
    if case.get("scene") == "cornell":
        return {"rel": 1e-3, "max": 0.5}
    return {"rel": 0.03, "max": 0.99, "differ": 1e-2}


# ------------------------------------------------------------------- exact
def _world_triangles(host):
    """(n, 3, 3) of the scene's input in the order of its primitive ids (the rooms' instances are untransformed)."""
    d, out = host.desc(), []
    for i in range(d.instanceCount):
        m = d.models[d.instances[i].modelIndex]
        v = np.ctypeslib.as_array(ctypes.cast(m.vertices, ctypes.POINTER(ctypes.c_float)), (m.vertexCount, 12))
        out.append(v[np.ctypeslib.as_array(m.indices, (m.indexCount,)), :3].reshape(-1, 3, 3))
    return np.concatenate(out).astype(np.float64)


def _exact_rays(case, seed):
    if case["query"] == "occluded":
        return None
    if case["rays"] * case["triangles"] > 2e10:
        return None
    tri = torch.from_numpy(_world_triangles(rtxamd.HostScene.generate(abi.SCENE_ROOM, seed, case["triangles"]))).cuda()
    rays = torch.from_numpy(_rays(case, seed).astype(np.float64)).cuda()
    a, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    normal = torch.linalg.cross(e1, e2)
    columns = []
    for part in rays.split(max(1, int(2e7 / len(tri)))):
        o, d = part[:, None, 0:3], part[:, None, 4:7]
        det = -(part[:, 4:7] @ normal.T)
        s = o - a
        q = torch.linalg.cross(s, d.expand_as(s))
        u, v = (q * e2).sum(-1) / det, -(q * e1).sum(-1) / det
        t = (s * normal).sum(-1) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= part[:, 3:4]) & (t <= part[:, 7:8])
        t = torch.where(ok, t, torch.inf)
        best, at = t.min(1)
        hit = torch.isfinite(best)
        pick = lambda x: torch.where(hit, x.gather(1, at[:, None])[:, 0], 0.0)  # noqa: E731
        columns.append(torch.stack([torch.where(hit, best, part[:, 7]), pick(u), pick(v)], 1))
    t, u, v = torch.cat(columns).T
    return t, None, u, v


def _exact_network(case, seed):
    """The encoding, the layers, the relative L2 loss and its gradients, nothing rounded on the way."""
    grid, mlp, train, target, queries = (torch.from_numpy(v).cuda().double() for v in _network(case, seed))
    grid.requires_grad_(True)
    mlp.requires_grad_(True)
    entries = 1 << case["log2_table"]
    # the configuration's resolutions: 16 to 2048 in 16 levels
    growth = math.exp((math.log(2048.0) - math.log(16.0)) / 15)

    def forward(x):
        p = ((x[:, 0:3] - torch.tensor([-10.0, 0, -10]).cuda()) / torch.tensor([20.0, 10, 20]).cuda()).clamp(0, 1)
        features = []
        for level in range(16):
            res = math.floor(16.0 * growth ** level)
            cell = torch.floor(p * res).clamp(0, res - 1)
            t, cell = p * res - cell, cell.long()
            sums = 0.0
            for corner in range(8):
                bit = torch.tensor([corner & 1, corner >> 1 & 1, corner >> 2], device="cuda")
                c = cell + bit
                if (res + 1) ** 3 <= entries:
                    at = c[:, 0] + (res + 1) * (c[:, 1] + (res + 1) * c[:, 2])
                else:
                    at = (c[:, 0] ^ (c[:, 1] * 2654435761 & 0xFFFFFFFF) ^ (c[:, 2] * 805459861 & 0xFFFFFFFF)) & (entries - 1)
                sums = sums + torch.where(bit == 1, t, 1 - t).prod(1, keepdim=True) * grid[level][at]
            features.append(sums)
        n = len(x)
        h = torch.cat(features + [x[:, 4:7], x[:, 8:11], x[:, 3:4], x[:, 12:15], torch.ones(n, 1, device="cuda"),
                                  torch.zeros(n, 21, device="cuda")], 1)
        for layer in range(5):
            h = torch.relu(h @ mlp[layer * 4096:(layer + 1) * 4096].reshape(64, 64).T)
        return h @ mlp[5 * 4096:5 * 4096 + 192].reshape(3, 64).T

    pred = forward(train)
    loss = ((pred - target) ** 2 / (pred.detach() ** 2 + 0.01)).mean()
    loss.backward()
    with torch.no_grad():
        rgb = torch.cat([forward(part) for part in queries.split(1 << 16)])
    return float(loss), grid.grad, mlp.grad, rgb


def exact(case, seed):
    # The images have no value of their own in 64 bits: a path's hits and its
    # 24-bit draws decide where it goes next, so a last bit anywhere sends it
    # elsewhere, and only a restatement of the whole renderer says where.
    f = {"rays": _exact_rays, "network": _exact_network}.get(case["kind"])
    return f(case, seed) if f else None
