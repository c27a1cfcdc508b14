"""What users of this renderer wait for, as cases that can be timed.

A case is one whole request through the public interface: a scene rendered to
its host framebuffer (the update stage, the frame's launches and its copy
back, as QuadRay's rt_Scene::render), a path-traced still, a batch of frames,
a burst of requests to the serving loop, or a frame from caller tables
through the entry point that allocates nothing.  Scenes are the seeded
workloads of qrgen_create; a seed draws other surfaces, materials, lights and
cameras, so another seed is another scene.

Every output is a frame of packed ARGB8 pixels: whole numbers that must stay
the same bit for bit (the test suite holds them equal to the CPU oracle's),
so the tolerance is "exact" and there is no 64-bit value to compare with.
"""
import ctypes as C
import math
import os
import random
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "quadray-engine_amd", "python"))

import qrhip  # noqa: E402

SAMPLES = (1, 2, 4)             # camera samples per pixel by AA mode

# fp32 operations one camera sample cannot do without, per workload at
# secondary-ray depths 0, 1, 2, 4 and 8: the CPU oracle's count of the
# operations along each ray when it skips what its own box tests rule out
# (160x90, seed 1; the median of seeds 1-8 for 7 and 8)
OPS_DEPTHS = (0, 1, 2, 4, 8)
OPS = {
    1: (320, 320, 320, 320, 320),
    2: (2227, 2505, 2655, 2815, 2926),
    4: (6843, 8871, 10046, 11262, 12803),
    5: (13824, 15980, 16806, 18031, 20188),
    6: (2361, 3371, 4226, 5767, 9499),
    7: (2295, 2599, 2788, 2954, 3111),
    8: (3911, 4292, 4479, 4699, 4926),
    9: (2229, 2400, 2489, 2504, 2507),
}
# the same per path-traced sample at depths 2, 4, 8 and 10
PT_DEPTHS = (2, 4, 8, 10)
PT_OPS = (1342, 1761, 3342, 4876)
PT_BOX = 3                      # the path-traced box's workload

SERVE_RES = ((640, 360), (1280, 720), (1920, 1080))


def listed():
    return [
        # the smallest call: a thumbnail, where launches and latency count
        {"name": "thumb_64", "kind": "still", "config": 7, "x": 64, "y": 64, "fsaa": 0,
         "depth": 1, "time": 0, "animated": False},
        # the plain scene (a plane and a few quadrics) at its own size
        {"name": "plain_800x480", "kind": "still", "config": 1, "x": 800, "y": 480, "fsaa": 0,
         "depth": 4, "time": 0, "animated": False},
        # an interactive viewer: a small animated frame, updated every time
        {"name": "animated_360p", "kind": "still", "config": 8, "x": 640, "y": 360, "fsaa": 0,
         "depth": 4, "time": 40, "animated": True},
        # every surface kind with clippers and gamma, odd sizes, 4X
        {"name": "kinds_321x181_4x", "kind": "still", "config": 9, "x": 321, "y": 181,
         "fsaa": 2, "depth": 6, "time": 0, "animated": False},
        # a dense scene (256 quadrics) at an odd size, 2X
        {"name": "dense_1281x719_2x", "kind": "still", "config": 4, "x": 1281, "y": 719,
         "fsaa": 1, "depth": 3, "time": 0, "animated": False},
        # glass everywhere, deep secondary rays: the largest ray trees
        {"name": "glass_641x359_4x", "kind": "still", "config": 6, "x": 641, "y": 359,
         "fsaa": 2, "depth": 8, "time": 0, "animated": False},
        # the headline frame: 64 quadrics, 4 lights, Fresnel, 1080p 4X
        {"name": "whitted_1080p_4x", "kind": "still", "config": 2, "x": 1920, "y": 1080,
         "fsaa": 2, "depth": 4, "time": 0, "animated": False},
        # frames of uneven scene, size, AA and depth traced together
        {"name": "batch_24", "kind": "batch", "frames": 24, "scenes": 6},
        # requests that arrive together at the serving loop
        {"name": "serve_16", "kind": "serve", "requests": 16, "scenes": 6},
        # a path-traced preview: one pass of a small frame, deep paths, 4X
        {"name": "pt_321x179_1spp", "kind": "pt", "x": 321, "y": 179, "fsaa": 2,
         "depth": 10, "spp": 1},
        # a path-traced still: the box at 720p, 64 samples per pixel
        {"name": "pt_720p_64spp", "kind": "pt", "x": 1280, "y": 720, "fsaa": 0,
         "depth": 8, "spp": 64},
        # caller tables through the entry point that allocates nothing
        {"name": "noalloc_640x360_2x", "kind": "noalloc", "config": 2, "x": 640, "y": 360,
         "fsaa": 1, "depth": 4},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("still", "still", "still", "still", "pt", "pt", "batch", "serve",
                       "noalloc"))
    if kind == "batch":
        return {"kind": kind, "frames": rng.randint(5, 24), "scenes": rng.randint(2, 6)}
    if kind == "serve":
        return {"kind": kind, "requests": rng.randint(5, 16), "scenes": rng.randint(2, 6)}
    x = _log(rng, 64, 1920)
    y = max(33, min(1080, int(x * rng.uniform(0.4, 0.8))))
    fsaa = rng.randrange(3)
    if kind == "pt":
        depth = rng.randint(2, 10)
        x, y = min(x, 1280), min(y, 720)
        most = max(1, min(64, int(2.0e7 / (x * y * SAMPLES[fsaa]))))
        return {"kind": kind, "x": x, "y": y, "fsaa": fsaa, "depth": depth,
                "spp": _log(rng, 1, most)}
    if kind == "noalloc":
        return {"kind": kind, "config": rng.choice((1, 2, 6, 9)), "x": min(x, 900),
                "y": min(y, 600), "fsaa": fsaa, "depth": rng.randint(0, 6)}
    return {"kind": kind, "config": rng.choice((1, 2, 2, 4, 5, 6, 7, 7, 8, 9)), "x": x,
            "y": y, "fsaa": fsaa, "depth": rng.choice((0, 1, 2, 3, 4, 4, 4, 6, 8)),
            "time": rng.choice((0, 40, 80, 120)), "animated": rng.random() < 0.3}


class _Handles:
    """The library handles a program holds between frames; released with the
    object."""

    def __init__(self, fsaa):
        self.dev = qrhip.Device(0)
        self.dev.set_fsaa(fsaa)
        self.works, self.scenes = [], []
        self.batch = self.server = None

    def scene(self, config, seed, x, y, animated=False):
        w = qrhip.Workload(config, seed, animated=animated)
        self.works.append(w)
        s = qrhip.Scene(self.dev, w.ptr, x, y)
        self.scenes.append(s)
        return s

    def __del__(self):
        for h in (self.batch, self.server):
            if h is not None:
                h.destroy()
        for s in self.scenes:
            s.destroy()
        for w in self.works:
            w.close()
        self.dev.close()


class _State:
    """A case's handles and inputs."""

    def __init__(self, case):
        self.case = case
        self.handles = _Handles(case.get("fsaa", 0))


def _framebuffer(handles, s):
    """The scene's host framebuffer as an array over the same memory, which
    keeps the scene alive while the array is."""
    p = qrhip.lib().qrhip_scene_get_frame(s.h)
    buf = (C.c_int32 * (s.x_res * s.y_res)).from_address(C.addressof(p.contents))
    buf.handles = handles
    return np.ctypeslib.as_array(buf).reshape(s.y_res, s.x_res)


def _batch_frames(case):
    """(scene, x, y, fsaa, depth) per frame: sizes log-uniform 64x64 to
    1920x1080; the first three are of the smallest, a middle and the largest
    size, so every batch has the range.  (A seed changes the scenes.)"""
    rng = random.Random(case["frames"] * 7919 + case["scenes"])
    out = []
    for k in range(case["frames"]):
        t = (0.0, 0.5, 1.0)[k] if k < 3 else rng.random()
        out.append((rng.randrange(case["scenes"]), int(round(64 * (1920 / 64) ** t)),
                    int(round(64 * (1080 / 64) ** t)), rng.randrange(3), rng.randint(1, 4)))
    return out


def _requests(case):
    """(scene, x, y, fsaa, spp, time, yaw) per request; the last scene is the
    path-traced box, which one request in seven asks for."""
    rng = random.Random(case["requests"] * 104729 + case["scenes"])
    out = []
    for k in range(case["requests"]):
        pt = k % 7 == 6
        x, y = SERVE_RES[k % 3]
        out.append((case["scenes"] - 1 if pt else rng.randrange(case["scenes"] - 1), x, y,
                    0 if pt else rng.randrange(3), 16 if pt else 0, rng.randrange(4) * 40,
                    rng.uniform(-0.5, 0.5)))
    return out


def prepare(case, seed):
    kind = case["kind"]
    st = _State(case)
    h = st.handles
    if kind in ("still", "pt"):
        s = h.scene(PT_BOX if kind == "pt" else case["config"], seed, case["x"], case["y"],
                    case.get("animated", False))
        s.set_depth(case["depth"])
        st.scene = s
        st.frame = _framebuffer(h, s)
    elif kind == "batch":
        for k in range(case["scenes"]):
            h.scene(7, seed * 64 + k, 64, 64).update(0)
        h.batch = qrhip.Batch(h.dev)
        h.batch.set([(h.scenes[i], x, y, a, d) for i, x, y, a, d in _batch_frames(case)])
    elif kind == "serve":
        for k in range(case["scenes"] - 1):
            h.scene(8, seed * 64 + k, 64, 64, animated=True).update(0)
        h.scene(PT_BOX, seed * 64 + 63, 64, 64).update(0)
        st.reqs = []
        for k, (i, x, y, a, spp, t, yaw) in enumerate(_requests(case)):
            c, s_ = math.cos(yaw), math.sin(yaw)
            rz = np.array([[c, -s_, 0.0], [s_, c, 0.0], [0.0, 0.0, 1.0]])
            pose = (h.scenes[i].pose().astype(np.float64).reshape(4, 3) @ rz.T).reshape(12)
            st.reqs.append(qrhip.Server.request(k, i, x, y, a, 4, spp=spp, time=t, pose=pose))
        # bounded by memory and by the samples a step takes; a serving loop
        # runs for long, so its buffers are at their working sizes
        h.server = qrhip.Server(h.dev, h.scenes, 64 << 30, 64, 1 << 24)
        for _ in range(3):
            _serve(h.server, st.reqs)
    elif kind == "noalloc":
        s = h.scene(case["config"], seed, case["x"], case["y"])
        s.set_depth(case["depth"])
        s.update(0)
        st.tables, st.fd = s.tables()
    else:
        raise ValueError(kind)
    return st


def _serve(srv, reqs):
    """Submit the requests at once and wait for their frames."""
    frames = [srv.submit(r) for r in reqs]
    left = len(frames)
    while left > 0:
        got = srv.poll(wait_ms=1000)
        if any(r["status"] != 0 for r in got):
            raise RuntimeError("a request failed")
        left -= len(got)
    srv.frames.clear()
    return [f.view(np.int32) for f in frames]


def run(state):
    kind, h = state.case["kind"], state.handles
    L = qrhip.lib()
    if kind == "still":
        qrhip.check(L.qrhip_scene_render(state.scene.h, state.case["time"]))
        return state.frame
    if kind == "pt":
        # a still from the first sample on: switching the path tracer on
        # restarts the accumulation
        state.scene.set_pton(0)
        state.scene.set_pton(state.case["spp"])
        qrhip.check(L.qrhip_scene_render(state.scene.h, 0))
        return state.frame
    if kind == "batch":
        h.batch.launch(qrhip.BATCH_GRAPH)
        qrhip.check(L.qrhip_batch_download(h.batch.h, -1))
        return [b.view(np.int32) for b in h.batch.bufs]
    if kind == "serve":
        return _serve(h.server, state.reqs)
    frame, _ = h.dev.render_tables_noalloc(state.tables, state.fd)
    return frame.view(np.int32)


def _at(depths, ops, depth):
    """ops at a depth, linear between the counted depths."""
    if depth >= depths[-1]:
        return ops[-1] * (depth + 1) / (depths[-1] + 1)
    for k in range(len(depths) - 1):
        if depth <= depths[k + 1]:
            t = (depth - depths[k]) / (depths[k + 1] - depths[k])
            return ops[k] + (ops[k + 1] - ops[k]) * t
    return ops[-1]


def work(case):
    """The operations along each ray and the pixels written: tables and
    textures (tens of kilobytes) are read once, queues are not counted."""
    kind = case["kind"]
    if kind == "batch":
        parts = [(x * y, x * y * SAMPLES[a] * _at(OPS_DEPTHS, OPS[7], d))
                 for _, x, y, a, d in _batch_frames(case)]
    elif kind == "serve":
        parts = [(x * y, x * y * (spp * _at(PT_DEPTHS, PT_OPS, 4) if spp else
                                  SAMPLES[a] * _at(OPS_DEPTHS, OPS[8], 4)))
                 for _, x, y, a, spp, _, _ in _requests(case)]
    else:
        px = case["x"] * case["y"]
        n = px * SAMPLES[case["fsaa"]]
        if kind == "pt":
            n *= case["spp"] * _at(PT_DEPTHS, PT_OPS, case["depth"])
        else:
            n *= _at(OPS_DEPTHS, OPS[case["config"]], case["depth"])
        parts = [(px, n)]
    return {"bytes": 4.0 * sum(p for p, _ in parts) + 65536.0 * len(parts),
            "flops": float(sum(f for _, f in parts))}


def tolerance(case):
    """Packed 8-bit pixels: whole numbers, the same on every correct run."""
    return "exact"


def exact(case, seed):
    """None: pixels are whole numbers, held equal bit for bit."""
    return None
