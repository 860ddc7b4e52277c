"""The work a user of this framework has it do, as cases to be measured: frames of one or
several cameras, foveated frames, animated scenes, batches and served requests, through the
package's own entry points and its C interface (include/hvvr_gpu.h).

A frame ends with its image in page-locked host memory (hvvr_gpu_host_alloc), read as
Raycaster::render's caller reads its render target. Scenes are the package's seeded room
(meshes of 256 triangles) and a heightfield with boxes; the scene is the asset a program has
on disk, the seed decides the cameras, lens, gaze, transforms and displacements."""

import ctypes
import functools
import math
import weakref

import numpy as np
import torch

import hvvr_amd as H

SERVED_SIZES = [(256, 256), (360, 400), (540, 600)]
ROOM_CENTRE = (15.0, 7.5, 29.0)


def listed():
    return [
        # a picking or calibration call: the smallest frame, depth and barycentrics read back
        dict(name="depth_96x72", kind="depth", width=96, height=72, msaa=1, cells=16),
        # one pinhole camera over a small scene, colour and per-sample depth
        dict(name="depth_640x480", kind="depth", width=640, height=480, msaa=1, cells=64),
        # a preview of a textured scene at an odd size
        dict(name="textured_257x303", kind="views", width=257, height=303, msaa=8, meshes=391, count=1, bits=32,
             lens=False, textured=True),
        # the headset frame: both eyes in one submission, as Raycaster::render makes it
        dict(name="stereo_1080x1200", kind="views", width=1080, height=1200, msaa=4, meshes=1024, count=2, bits=32,
             lens=False, textured=False),
        # a thin-lens camera
        dict(name="lens_540x600", kind="views", width=540, height=600, msaa=8, meshes=1024, count=1, bits=32,
             lens=True, textured=False),
        # dense scenes of 1M and 2M triangles
        dict(name="dense_1m_1080x1200", kind="views", width=1080, height=1200, msaa=4, meshes=4096, count=1, bits=16,
             lens=False, textured=False),
        dict(name="dense_2m_760x840", kind="views", width=760, height=840, msaa=2, meshes=8192, count=1, bits=16,
             lens=False, textured=False),
        # foveated eye with a lens, jittered, the gaze moving: 315k polar samples to a headset eye
        dict(name="foveated_lens_1080x1200", kind="foveated", width=1080, height=1200, msaa=4, meshes=1024, bits=32,
             lens=True),
        # foveated eye of a dense scene, as served
        dict(name="foveated_1m_1080x1200", kind="foveated", width=1080, height=1200, msaa=2, meshes=4096, bits=16,
             lens=False),
        # animated models: new transforms, refit, and the refitted scene fetched
        dict(name="animate_262k", kind="animate", meshes=1024),
        # many views of a 1M-triangle scene per launch, 10% of its vertices displaced and the
        # BVH refitted in the replayed graph
        dict(name="batch_16_1m", kind="batch", views=16, meshes=4096, mix=0),
        # a burst of requests of mixed sizes, rates and foveation over two resident scenes
        dict(name="serving_16", kind="serving", requests=16, meshes=391, more_meshes=1024, mix=0),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["depth", "views", "views", "views", "foveated", "animate", "batch", "serving"])
    if kind == "depth":
        return dict(kind=kind, width=_spread(rng, 33, 640), height=_spread(rng, 25, 480), msaa=rng.choice([1, 2]),
                    cells=_spread(rng, 7, 64))
    if kind == "views":
        lens = rng.random() < 0.25
        meshes = _spread(rng, 16, 1024 if lens else 4096)
        return dict(kind=kind, width=_spread(rng, 99, 1080), height=_spread(rng, 101, 1200),
                    msaa=rng.choice([1, 2, 4, 8]), meshes=meshes, count=1 if meshes > 1024 else rng.choice([1, 2, 3]),
                    bits=rng.choice([16, 32]), lens=lens, textured=rng.random() < 0.25)
    if kind == "foveated":
        return dict(kind=kind, width=_spread(rng, 270, 1080), height=_spread(rng, 300, 1200),
                    msaa=rng.choice([1, 2, 4]), meshes=_spread(rng, 64, 2048), bits=rng.choice([16, 32]),
                    lens=rng.random() < 0.3)
    if kind == "animate":
        return dict(kind=kind, meshes=_spread(rng, 16, 1024))
    if kind == "batch":
        return dict(kind=kind, views=_spread(rng, 2, 16), meshes=_spread(rng, 64, 2048), mix=rng.randrange(1, 1 << 20))
    return dict(kind=kind, requests=_spread(rng, 3, 16), meshes=_spread(rng, 64, 1024),
                more_meshes=_spread(rng, 64, 1024), mix=rng.randrange(1, 1 << 20))


# ---------------------------------------------------------------------------------------
# assets, shared by the states: a program loads them once
# ---------------------------------------------------------------------------------------
@functools.lru_cache(None)
def _context():
    return H.GpuContext(0)


@functools.lru_cache(maxsize=6)
def _room(meshes):
    return H.HostScene(H.SCENE_ROOM, 0, meshes)


@functools.lru_cache(maxsize=2)
def _textured_room(meshes):
    """The room with half its materials naming a diffuse texture and a third a glossy one."""
    scene = H.HostScene(H.SCENE_ROOM, 0, meshes)
    none = 0xFFFF
    for i in range(len(scene.materials)):
        model = int(scene.materials["textureIDsAndShadingModel"][i]) & 0xFFFF
        diffuse = i % 3 if i % 2 else none
        glossy = 3 if i % 3 == 0 else none
        scene.materials["textureIDsAndShadingModel"][i] = model | (glossy << 16) | (none << 32) | (diffuse << 48)
    return scene


@functools.lru_cache(maxsize=64)
def _view(width, height, eye=0):
    return H.HostView(H.VIEW_PRESET_ROOM_EYE, eye, width, height)


@functools.lru_cache(maxsize=2)
def _polar():
    return H.HostFoveated(H.HostFoveated.FEB2017)


def _terrain_meshes(cells):
    """(positions [n, 3], triangles [m, 3]) of a 16 x 16 m heightfield of cells x cells quads,
    4 boxes per cell row on it, and one large triangle beneath, which every ray that nothing
    else stops ends on."""
    rng = np.random.default_rng(cells)
    n = cells + 1
    x, z = np.meshgrid(np.arange(n) * (16.0 / cells), np.arange(n) * (16.0 / cells))
    pos = [np.stack([x, rng.uniform(0, 1, (n, n)), z], -1).reshape(-1, 3)]
    a = (np.arange(cells)[:, None] * n + np.arange(cells)[None, :]).reshape(-1)
    tri = [np.stack([a, a + n, a + n + 1], -1), np.stack([a, a + n + 1, a + 1], -1)]
    corner = np.array([[i & 1, (i >> 1) & 1, i >> 2] for i in range(8)], np.float64) - 0.5
    quads = [(1, 3, 7, 5), (0, 4, 6, 2), (2, 6, 7, 3), (0, 1, 5, 4), (4, 5, 7, 6), (0, 2, 3, 1)]
    base = n * n
    for _ in range(4 * cells):
        centre = np.array([rng.uniform(2, 14), rng.uniform(0.5, 1.2), rng.uniform(2, 14)])
        edge = 0.1 * 20.0 ** rng.uniform(0, 1, 3)
        pos.append(centre + corner * edge)
        q = np.array(quads) + base
        tri += [q[:, [0, 1, 2]], q[:, [0, 2, 3]]]
        base += 8
    pos.append(np.array([[-400.0, -3.0, -400.0], [0.0, -3.0, 800.0], [400.0, -3.0, -400.0]]))
    tri.append(np.array([[base, base + 1, base + 2]]))
    return np.concatenate(pos).astype(np.float32), np.concatenate(tri).astype(np.uint32)


@functools.lru_cache(maxsize=4)
def _terrain(cells):
    pos, tri = _terrain_meshes(cells)
    rng = np.random.default_rng(cells + 1)
    p = pos[tri].astype(np.float64)
    face = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
    normal = np.zeros((len(pos), 3))
    for k in range(3):
        np.add.at(normal, tri[:, k], face)
    normal /= np.linalg.norm(normal, axis=1, keepdims=True)
    verts = np.zeros(len(pos), H.DTYPES["vertex"])
    verts["pos"] = pos
    verts["normal"][:, :3] = normal.astype(np.float16).view(np.uint16)
    mats = np.zeros(16, H.DTYPES["material"])
    mats["diffuse"] = np.concatenate([rng.uniform(0, 1, (16, 3)), np.ones((16, 1))], 1)
    mats["specular"] = (0.04, 0.04, 0.04, 1.0)
    mats["glossiness"] = rng.uniform(0.1, 0.9, 16)
    mats["opacity"] = 1.0
    mats["textureIDsAndShadingModel"] = 1 | (0xFFFF << 16) | (0xFFFF << 32) | (0xFFFF << 48)
    light = np.zeros(1, H.DTYPES["light"])
    light["type"] = 1
    light["body"][0, :6] = (0.4, 0.8, 0.45, 2.5, 2.4, 2.2)
    light["body"][0, :3] /= np.linalg.norm(light["body"][0, :3])
    return H.HostScene.from_meshes([(verts, tri, rng.integers(0, 16, len(tri)), None)], mats, light)


@functools.lru_cache(maxsize=4)
def _terrain_view(width, height):
    """A 60 degree camera's samples."""
    t = math.tan(math.radians(30.0))
    s = t * width / height
    return H.HostView.from_samples(H.grid_samples(width, height), width, height, (-s, -t, s, t))


# ---------------------------------------------------------------------------------------
# what a program holds
# ---------------------------------------------------------------------------------------
def _check(rc):
    if rc < 0:
        raise H.HvvrError(H.load_gpu().hvvr_gpu_last_error().decode())


class _Pinned:
    """Page-locked host memory as arrays; freed with the last of them."""

    def __init__(self, nbytes):
        lib = H.load_gpu()
        lib.hvvr_gpu_host_alloc.restype = ctypes.c_void_p
        lib.hvvr_gpu_host_alloc.argtypes = [ctypes.c_uint64]
        lib.hvvr_gpu_host_free.argtypes = [ctypes.c_void_p]
        address = lib.hvvr_gpu_host_alloc(nbytes)
        if not address:
            raise MemoryError("page-locked host memory: out of memory")
        self.pointer = ctypes.c_void_p(address)
        self.__array_interface__ = dict(shape=(nbytes,), typestr="|u1", data=(address, False), version=3)
        weakref.finalize(self, lib.hvvr_gpu_host_free, address)


def _pinned(nbytes):
    p = _Pinned(nbytes)
    return np.asarray(p), p.pointer


class _State:
    """Closes what it holds, views before scenes."""

    def __init__(self, case, seed):
        self.case, self.rng, self.closing = case, np.random.default_rng(seed), []

    def hold(self, x):
        self.closing.append(x)
        return x

    def __del__(self):
        try:
            _context().synchronize()
            for x in reversed(self.closing):
                x.close()
        except Exception:
            pass


def _camera(rng):
    """A pose near the room's entrance: (position, rotation quaternion)."""
    pos = np.array(ROOM_CENTRE) + rng.uniform(-1, 1, 3) * (2.0, 1.0, 0.5)
    yaw, pitch = np.radians(rng.uniform(-12, 12)) / 2, np.radians(rng.uniform(-6, 6)) / 2
    cy, sy, cp, sp = math.cos(yaw), math.sin(yaw), math.cos(pitch), math.sin(pitch)
    return pos, np.array([cy * sp, sy * cp, -sy * sp, cy * cp])


def _eye_matrix(pos, q, eye):
    m = H.transform_matrix(pos, q).reshape(4, 4)
    return H.transform_matrix(pos + (eye - 0.5) * 0.064 * m[0, :3].astype(np.float64), q)


def _fit(view, render):
    """Renders until the view's lists hold the frame, as list_demand asks."""
    for _ in range(3):
        render()
        need, have, overflowed = view.list_demand()
        if not overflowed:
            return
        view.reserve_lists(need + need // 4)


def _image_buffer(view):
    data, pointer = _pinned(view.view.height * view.view.width * 4)
    return data.reshape(view.view.height, view.view.width, 4), pointer


def _read_image(view, pointer):
    _check(view.lib.hvvr_gpu_view_read_image(view.handle, pointer, ctypes.c_uint32(view.view.width)))


def prepare(case, seed):
    s = _State(case, seed)
    globals()["_prepare_" + case["kind"]](s, case)
    _context().synchronize()
    return s


def run(state):
    return globals()["_run_" + state.case["kind"]](state)


# ---- depth: one small camera, its image and every sample's (t, u, v, w) ----
def _terrain_camera(rng):
    """Above the terrain, looking down."""
    pos = np.array([8.0, 7.0, 8.0]) + rng.uniform(-1, 1, 3)
    half = math.radians(-85.0 + rng.uniform(-5, 5)) / 2
    return H.transform_matrix(pos, (math.sin(half), 0.0, 0.0, math.cos(half)))


def _prepare_depth(s, case):
    hv = _terrain_view(case["width"], case["height"])
    s.scene = s.hold(H.GpuScene(_context(), _terrain(case["cells"])))
    s.view = s.hold(H.GpuView(_context(), hv, case["msaa"]))
    s.view.set_hit_output(True)
    s.camera = _terrain_camera(s.rng)
    s.image, s.image_ptr = _image_buffer(s.view)
    s.hits, s.hits_ptr = _pinned(hv.sample_count * case["msaa"] * 16)
    s.hits = s.hits.view(np.float32).reshape(hv.sample_count, case["msaa"], 4)
    _fit(s.view, lambda: s.view.render(s.scene, s.camera))


def _run_depth(s):
    s.view.render(s.scene, s.camera)
    _check(s.view.lib.hvvr_gpu_view_read_hits(s.view.handle, s.hits_ptr))
    _read_image(s.view, s.image_ptr)
    return {"image": s.image, "hits": s.hits}


# ---- views: the frame of one or several cameras ----
def _prepare_views(s, case):
    ctx = _context()
    scene = _textured_room(case["meshes"]) if case["textured"] else _room(case["meshes"])
    s.scene = s.hold(H.GpuScene(ctx, scene))
    if case["textured"]:
        s.scene.set_textures([("srgb8", s.rng.integers(0, 256, (256, 256, 4), np.uint8)) for _ in range(3)] +
                             [("unorm8", s.rng.integers(0, 256, (128, 64, 4), np.uint8))])
    pos, q = _camera(s.rng)
    s.views, s.cameras, s.images = [], [], []
    for eye in range(case["count"]):
        hv = _view(case["width"], case["height"], eye & 1)
        if case["lens"]:
            hv = _lens_view(hv, 0.01, float(s.rng.uniform(1, 10)))
        v = s.hold(H.GpuView(ctx, hv, case["msaa"]))
        v.set_shading_precision(case["bits"])
        s.views.append(v)
        s.cameras.append(_eye_matrix(pos, q, eye))
        s.images.append(_image_buffer(v))
        _fit(v, lambda: v.render(s.scene, s.cameras[-1]))


class _lens_view:
    """A host view's samples with another lens (radius, focal distance)."""

    def __init__(self, hv, radius, focal):
        self._hv, self.lens = hv, np.array([radius, focal], np.float32)

    def __getattr__(self, name):
        return getattr(self._hv, name)


def _run_views(s):
    if len(s.views) == 1:
        s.views[0].render(s.scene, s.cameras[0])
    else:
        H.render_views(s.scene, s.views, s.cameras)
    for v, (_, pointer) in zip(s.views, s.images):
        _read_image(v, pointer)
    return [image for image, _ in s.images]


# ---- foveated: one eye's polar samples traced and reconstructed, frame after frame ----
def _prepare_foveated(s, case):
    ctx = _context()
    s.scene = s.hold(H.GpuScene(ctx, _room(case["meshes"])))
    s.screen = _view(case["width"], case["height"])
    lens = dict(lens_radius=0.01, focal_distance=float(s.rng.uniform(1, 10))) if case["lens"] else {}
    s.view = s.hold(H.GpuFoveatedView(ctx, _polar(), case["width"], case["height"], case["msaa"], **lens))
    s.view.set_shading_precision(case["bits"])
    s.view.set_jitter_spin(True)
    pos, q = _camera(s.rng)
    s.camera = _eye_matrix(pos, q, 0)
    s.gazes = np.radians(s.rng.uniform(-20, 20, (64, 2)))
    s.jitters = s.rng.uniform(0, 1, (64, 2)).astype(np.float32)
    s.image, s.image_ptr = _image_buffer(s.view)
    for k in range(0, 64, 8):
        s.frame, s.history = k, H.foveated_history()
        _fit(s.view, lambda: _foveated_frame(s))
    # the lists have room for gazes that were not tried
    need, have, _ = s.view.list_demand()
    s.view.reserve_lists(have + have // 2)
    s.frame, s.history = 0, H.foveated_history()


def _foveated_frame(s):
    yaw, pitch = s.gazes[s.frame % 64]
    eye = np.array([math.sin(yaw) * math.cos(pitch), math.sin(pitch), -math.cos(yaw) * math.cos(pitch)], np.float32)
    frame = H.foveated_frame(s.camera, eye, s.screen.sample_to_camera, s.screen.sample_bounds, s.history)
    s.view.render_foveated(s.scene, frame, s.jitters[s.frame % 64])


def _run_foveated(s):
    _foveated_frame(s)
    s.frame += 1
    _read_image(s.view, s.image_ptr)
    return s.image


# ---- animate: model transforms, refit, the refitted nodes and triangles fetched ----
def _animated(rng, transforms):
    """Every model moved by up to 10 cm and turned by up to 0.1 rad about the vertical axis."""
    t = np.array(transforms, np.float32).reshape(-1, 4, 4)  # rows are the matrices' columns
    a = rng.uniform(-0.1, 0.1, len(t))
    turn = np.zeros((len(t), 3, 3))
    turn[:, 0, 0] = turn[:, 2, 2] = np.cos(a)
    turn[:, 0, 2], turn[:, 2, 0] = -np.sin(a), np.sin(a)
    turn[:, 1, 1] = 1.0
    t[:, :3, :3] = t[:, :3, :3].astype(np.float64) @ turn
    t[:, 3, :3] += rng.uniform(-0.1, 0.1, (len(t), 3))
    return t.reshape(-1, 16)


def _prepare_animate(s, case):
    scene = _room(case["meshes"])
    s.scene = s.hold(H.GpuScene(_context(), scene))
    s.transforms = _animated(s.rng, scene.transforms)
    s.nodes, s.nodes_ptr = _pinned(scene.nodes.nbytes)
    s.bounds = s.nodes.view(H.DTYPES["node"])["bounds"]
    s.tris, s.tris_ptr = _pinned(36 * len(scene.triShade))
    s.tris = s.tris.view(np.float32).reshape(-1, 9)
    s.scene.update()


def _run_animate(s):
    s.scene.set_transforms(s.transforms)
    s.scene.update()
    _check(s.scene.lib.hvvr_gpu_scene_read_nodes(s.scene.handle, s.nodes_ptr))
    _check(s.scene.lib.hvvr_gpu_scene_read_triangles(s.scene.handle, s.tris_ptr))
    return {"bounds": s.bounds, "triangles": s.tris}


# ---- batch: many views per launch, vertices displaced and the BVH refitted every frame ----
def _batch_specs(case):
    rng = np.random.default_rng(case["mix"])
    specs = []
    for _ in range(case["views"]):
        area = math.exp(rng.uniform(math.log(128 * 128), math.log(960 * 540)))
        h = int(round(math.sqrt(area * 9 / 16)))
        specs.append((max(int(round(h * 16 / 9)), 8), max(h, 8), int(rng.choice([1, 2, 4, 8]))))
    return specs


def _prepare_batch(s, case):
    ctx = _context()
    scene = _room(case["meshes"])
    s.scene = s.hold(H.GpuScene(ctx, scene))
    s.views, s.images, s.cameras = [], [], []
    for k, (w, h, a) in enumerate(_batch_specs(case)):
        v = s.hold(H.GpuView(ctx, _view(w, h, k & 1), a))
        v.set_shading_precision(16)
        s.views.append(v)
        s.images.append(_image_buffer(v))
        s.cameras.append(_eye_matrix(*_camera(s.rng), k & 1))
    n = len(scene.verts) // 10
    s.first = int(s.rng.integers(0, len(scene.verts) - n))
    s.moved = scene.verts[s.first:s.first + n].copy()
    s.moved["pos"] += s.rng.normal(0, 0.02, (n, 3)).astype(np.float32)
    s.batch = s.hold(H.GpuBatch(ctx, s.views))
    s.batch.set_refit(True)
    for _ in range(2):
        s.scene.set_vertices(s.first, s.moved)
        s.batch.render(s.scene, s.cameras)
        s.batch.synchronize()
        for v in s.views:
            need, have, overflowed = v.list_demand()
            if overflowed:
                v.reserve_lists(need + need // 4)
    s.batch.set_graph(True)
    s.batch.render(s.scene, s.cameras)


def _run_batch(s):
    s.scene.set_vertices(s.first, s.moved)
    s.batch.render(s.scene, s.cameras)
    s.batch.synchronize()
    for v, (_, pointer) in zip(s.views, s.images):
        _read_image(v, pointer)
    return [image for image, _ in s.images]


# ---- serving: a burst of requests, submitted together and drained ----
def _requests(case):
    rng = np.random.default_rng(case["mix"])
    return [(int(rng.integers(2)), int(rng.integers(len(SERVED_SIZES))), int(rng.choice([1, 2, 4])), bool(k % 2))
            for k in range(case["requests"])]


def _prepare_serving(s, case):
    ctx = _context()
    s.scenes = [s.hold(H.GpuScene(ctx, _room(case[k]))) for k in ("meshes", "more_meshes")]
    for g in s.scenes:
        g.update()
    s.server = s.hold(H.Server(ctx, 16 << 30, 8, shading_bits=16))
    shapes = {}
    s.queue = []
    for scene, size, msaa, foveated in _requests(case):
        key = (size, msaa, foveated)
        hv = _view(*SERVED_SIZES[size])
        if key not in shapes:
            shapes[key] = (s.server.add_foveated_shape(_polar(), hv, msaa) if foveated
                           else s.server.add_shape(hv, msaa))
        yaw, pitch = np.radians(s.rng.uniform(-20, 20, 2))
        eye = np.array([math.sin(yaw) * math.cos(pitch), math.sin(pitch), -math.cos(yaw) * math.cos(pitch)],
                       np.float32) if foveated else None
        s.queue.append((s.scenes[scene], shapes[key], _eye_matrix(*_camera(s.rng), 0), eye))
    _run_serving(s)  # the pool's views exist, their lists sized


def _run_serving(s):
    images = [s.server.submit(scene, shape, camera, eye)[1] for scene, shape, camera, eye in s.queue]
    s.server.drain()
    return [i.view(np.uint8) for i in images]


# ---------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------
def _scene_bytes(meshes):
    # per mesh: 256 triangles (36 B geometry, 16 B indices and material), about 224 vertices of
    # 32 B, about 35 nodes of 128 B, a material
    return meshes * (256 * 52 + 224 * 32 + 35 * 128 + 64)


def _frame(samples, msaa, pixels, lights=5):
    """One frame's own bytes (beams in, image out) and operations (one accepted triangle test
    of each subsample, one shading of each sample by each light)."""
    return 36 * samples + 4 * pixels, samples * (80 + 16 * msaa) + samples * lights * 80


def work(case):
    kind = case["kind"]
    polar = 315202
    if kind == "depth":
        n = case["width"] * case["height"]
        b, f = _frame(n, case["msaa"], n, 1)
        tris = 2 * case["cells"] ** 2 + 48 * case["cells"] + 1
        return {"bytes": b + 16 * n * case["msaa"] + 100 * tris, "flops": f}
    if kind == "views":
        n = case["width"] * case["height"]
        b, f = _frame(n, case["msaa"], n)
        return {"bytes": case["count"] * b + _scene_bytes(case["meshes"]), "flops": case["count"] * f}
    if kind == "foveated":
        b, f = _frame(polar, case["msaa"], 2 * case["width"] * case["height"])  # the history is read too
        return {"bytes": b + _scene_bytes(case["meshes"]), "flops": f + 400 * case["width"] * case["height"]}
    if kind == "animate":
        # vertices read, triangles and nodes written; a 4x4 transform per vertex, 6 comparisons
        # per triangle vertex
        m = case["meshes"]
        return {"bytes": m * (224 * 32 + 256 * (16 + 36) + 35 * 128), "flops": m * (224 * 32 + 256 * 24)}
    if kind == "batch":
        total = [0, 0]
        for w, h, a in _batch_specs(case):
            b, f = _frame(w * h, a, w * h)
            total[0] += b
            total[1] += f
        return {"bytes": total[0] + 2 * _scene_bytes(case["meshes"]), "flops": total[1]}
    total = [_scene_bytes(case["meshes"]) + _scene_bytes(case["more_meshes"]), 0]
    for _, size, a, foveated in _requests(case):
        w, h = SERVED_SIZES[size]
        b, f = _frame(polar if foveated else w * h, a, w * h)
        total[0] += b
        total[1] += f
    return {"bytes": total[0], "flops": total[1]}


# Bytes of an image are truncated 8-bit codes: a value near a code's edge falls on either side
# under another correct rounding. Against an FP64 shading of the same hits (270x300 room views,
# 1 to 8 subsamples) at most 1.3e-5 of the FP32 frames' bytes differ and 4.4e-3 of the frames'
# with packed-FP16 light terms; a foveated frame encodes its image several times over. Hits are
# the ray test's own FP32 values.
def tolerance(case):
    kind = case["kind"]
    if kind == "animate":
        return {"rel": 1e-6, "max": 1e-4}
    if kind == "depth":
        return {"rel": 1e-5, "max": 1e-2, "differ": 1e-4}
    if kind in ("foveated", "serving") or case.get("bits", 16) == 16:
        return {"rel": 1e-5, "differ": 1e-2}
    return {"rel": 1e-5, "differ": 5e-5}


# ---------------------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "depth":
        return {"image": None, "hits": _exact_hits(case, seed)}
    if case["kind"] == "animate":
        return _exact_refit(case, seed)
    return None  # images: bytes


def _exact_hits(case, seed):
    """(t, u, v, w) of each subsample's nearest front-facing triangle, every ray against every
    triangle (Moller-Trumbore)."""
    hv = _terrain_view(case["width"], case["height"])
    m = np.asarray(_terrain_camera(np.random.default_rng(seed)), np.float64).reshape(4, 4)
    rot, origin = m[:3, :3], m[3, :3]  # rows are the matrix's columns
    a = case["msaa"]
    turns = {1: 1, 2: 1}[a] * 6.28
    alpha = (np.arange(a) + 0.5) / a
    ox, oy = np.cos(alpha * turns) * np.sqrt(alpha), np.sin(alpha * turns) * np.sqrt(alpha)
    c, du, dv = (hv.beams[k].astype(np.float64) @ rot for k in ("centerRay", "du", "dv"))
    dirs = c[:, None] + du[:, None] * ox[None, :, None] + dv[:, None] * oy[None, :, None]
    dirs = torch.from_numpy(dirs.reshape(-1, 3)).cuda()
    pos, tri = _terrain_meshes(case["cells"])
    p = torch.from_numpy(pos[tri.astype(np.int64)].astype(np.float64)).cuda()
    e1, e2 = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    s = torch.from_numpy(origin).cuda() - p[:, 0]
    n, q = torch.linalg.cross(e1, e2), torch.linalg.cross(s, e1)
    se2 = torch.linalg.cross(e2, s)
    tn = (s * n).sum(1)
    out = torch.empty(len(dirs), 4, dtype=torch.float64, device="cuda")
    step = max(64, (1 << 25) // len(tri))
    for k in range(0, len(dirs), step):
        d = dirs[k:k + step]
        det = -(d @ n.T)  # d . (e1 x e2) = -det
        b1 = (d @ se2.T) / det
        b2 = (d @ q.T) / det
        t = tn[None] / det
        hit = (det > 0) & (b1 >= 0) & (b2 >= 0) & (b1 + b2 <= 1) & (t > 0)
        t = torch.where(hit, t, math.inf)
        near, i = t.min(1)
        b1, b2 = b1.gather(1, i[:, None])[:, 0], b2.gather(1, i[:, None])[:, 0]
        out[k:k + step] = torch.stack([near, 1 - b1 - b2, b1, b2], 1)
    return out.reshape(-1, a, 4).cpu().numpy()


def _exact_refit(case, seed):
    """Triangles (a corner and two edges) of the transformed vertices, and every child box of
    the BVH from them, children before parents; an empty slot holds -inf."""
    scene = _room(case["meshes"])
    xf = _animated(np.random.default_rng(seed), scene.transforms).astype(np.float64).reshape(-1, 4, 4)
    xf = xf[scene.vertexToTransform]
    pos = (scene.verts["pos"].astype(np.float64)[:, None, :] @ xf[:, :3, :3])[:, 0] + xf[:, 3, :3]
    p = pos[scene.triShade["indices"].astype(np.int64)]
    tris = np.concatenate([p[:, 0], p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]], 1)
    hi, lo = p.max(1), p.min(1)
    nodes = scene.nodes
    leaf, data = nodes["leafMask"], nodes["data"].astype(np.int64)
    bounds = np.empty((len(nodes), 6, 4))
    for i in range(len(nodes) - 1, -1, -1):
        for k in range(4):
            if leaf[i] >> k & 1:
                first, last = data[i, k], data[i, k + 1]
                if last <= first:
                    bounds[i, :, k] = -math.inf
                    continue
                bounds[i, 0::2, k] = hi[first:last].max(0)
                bounds[i, 1::2, k] = -lo[first:last].min(0)
            else:
                bounds[i, :, k] = bounds[i + data[i, 1 + k]].max(1)
    return {"bounds": bounds, "triangles": tris}
