"""HIP Whitted kernel against the oracle and QuadRay's golden frames, through
the C ABI (rt_Scene-style scenes and caller-built tables).

Bar: ARGB8 within +-1 per channel on >= 99.9% of the pixels, which these
kernels meet with every pixel identical (they apply QuadRay's operations in
its order), so frames are required bit-identical; first-hit ids identical
except on rays the oracle flags as near-zero discriminant (|D| < 1e-5, where
fp32 root selection is ill-conditioned)."""
import ctypes as C

import numpy as np
import pytest

import qr_oracle
import qrhip
from helpers import (GoldenTables, HostScene, assert_frame_exact, channels, frame_stats,
                     golden_camera_cases, golden_cases, golden_frame, golden_table_cases,
                     replay_actions)

pytestmark = pytest.mark.gpu

CASES = golden_cases()
TABLE_CASES = golden_table_cases()
PATHS = [qrhip.PATH_LEVELS, qrhip.PATH_ONE_KERNEL]


@pytest.fixture(params=PATHS, ids=["levels", "onekernel"])
def path_dev(device, request):
    """The device with one of its two tracing paths selected."""
    device.set_path(request.param)
    yield device
    device.set_path(qrhip.PATH_LEVELS)


def gpu_scene(device, config, seed, x, y, fsaa, depth, ids=False, x_row=None):
    device.set_fsaa(fsaa)
    w = qrhip.Workload(config, seed, ids=ids)
    s = qrhip.Scene(device, w.ptr, x, y, x_row=x_row)
    s.set_depth(depth)
    return w, s


@pytest.mark.parametrize("name", sorted(CASES))
def test_gpu_matches_reference_golden(path_dev, name):
    c = CASES[name]
    print(f"case {name} path {qrhip.lib().qrhip_device_get_path(path_dev.h)}", flush=True)
    w, s = gpu_scene(path_dev, c["config"], c["seed"], c["x_res"], c["y_res"],
                     c["fsaa"], c["depth"], ids=c["ids"])
    try:
        got = s.render(0)
    finally:
        s.destroy()
        w.close()
    exact, within, dmax = assert_frame_exact(got, golden_frame(name), name)
    print(f"{name}: exact {exact:.6f} within1 {within:.6f} max {dmax}")


@pytest.mark.parametrize("name", sorted(TABLE_CASES))
def test_gpu_matches_reference_test_scene(path_dev, name):
    """QuadRay's own test scenes (test/scenes/scn_test01..18: every surface
    kind, two-plane solver, gamma, array relations, textures), replayed from
    their stored tables, against QuadRay's frames bit for bit; the distance
    to its fp64 build is reported."""
    print(f"case {name} path {qrhip.lib().qrhip_device_get_path(path_dev.h)}", flush=True)
    g = GoldenTables(name)
    got, _ = path_dev.render_tables(g.ptr, g.fd)
    assert_frame_exact(got, g.frame, name)
    d = np.abs(channels(got) - channels(g.frame64)).max(-1)
    print(f"{name}: vs fp64 within1 {(d <= 1).mean():.5f} max {int(d.max())}")


@pytest.mark.parametrize("name", sorted(golden_camera_cases()))
def test_gpu_camera_actions(path_dev, name):
    """Camera actions between renders (rt_Scene::update(time, action)) on
    the device scene, against QuadRay's frame after the same calls."""
    c = golden_camera_cases()[name]
    print(f"case {name}", flush=True)
    w, s = gpu_scene(path_dev, c["config"], c["seed"], c["x_res"], c["y_res"],
                     c["fsaa"], c["depth"])
    try:
        got = replay_actions(s, c["actions"], s.render)
    finally:
        s.destroy()
        w.close()
    assert_frame_exact(got, golden_frame(name), name)


@pytest.mark.parametrize("config,seed,x,y,fsaa,depth", [
    (1, 11, 160, 96, 0, 1),
    (2, 12, 192, 108, 2, 0),
    (2, 13, 192, 108, 0, 14),
    (3, 14, 160, 90, 1, 8),
    (4, 15, 128, 72, 0, 4),
    (5, 16, 96, 54, 0, 4),
    (9, 17, 321, 181, 0, 6),
    (9, 18, 200, 120, 1, 10),
    (10, 19, 160, 90, 2, 10),
])
def test_gpu_matches_oracle(path_dev, config, seed, x, y, fsaa, depth):
    print(f"case config {config} seed {seed} {x}x{y} fsaa {fsaa} depth {depth}",
          flush=True)
    hs = HostScene(config, seed, x, y, fsaa, depth)
    try:
        want = hs.oracle()[0]
        got, _ = path_dev.render_tables(hs.tables, hs.fd)
    finally:
        hs.close()
    assert_frame_exact(got, want)


@pytest.mark.parametrize("config,seed", [(1, 21), (2, 22), (3, 23), (4, 24), (9, 25),
                                         (10, 26)])
def test_gpu_first_hit_ids(path_dev, config, seed):
    print(f"case ids config {config} seed {seed}", flush=True)
    hs = HostScene(config, seed, 192, 108, 2, 4)
    try:
        _, ids_o, flags, _, _ = hs.oracle(want_ids=True)
        _, ids_g = path_dev.render_tables(hs.tables, hs.fd, want_ids=True)
    finally:
        hs.close()
    diff = ids_o != ids_g
    assert not np.any(diff & (flags == 0)), int((diff & (flags == 0)).sum())
    print(f"ids differ on {int(diff.sum())} of {diff.size} samples "
          f"({int(flags.sum())} flagged)")


def test_gpu_rejects_malformed_culling_programs(device):
    """Caller tables are checked on the host before any launch: a box step
    whose range leaves the program, and a local box on a transform node
    (whose step must carry its group end), are refused."""
    hs = HostScene(2, 3, 64, 48, 0, 2)
    try:
        snap = qrhip.tables_snapshot(hs.tables, hs.fd)
    finally:
        hs.close()
    steps = snap["steps"].view(np.int32).reshape(-1, 8)
    n_step = steps.shape[0]
    srf_tag = snap["surfaces"].view(np.int32).reshape(-1, qrhip.C.sizeof(qrhip.QrSurface) // 4)
    elem_srf = snap["elems"].view(np.int32).reshape(-1, 2)[:, 0]
    box = np.nonzero(steps[:, 6] < 0)[0]
    node = [p for p in np.nonzero(steps[:, 6] >= 0)[0]
            if srf_tag[elem_srf[steps[p, 6]], qrhip.QrSurface.tag.offset // 4] < 0]
    assert len(box) and len(node)

    def attempt(edit, message):
        bad = {k: v.copy() for k, v in snap.items()}
        edit(bad["steps"].view(np.int32).reshape(-1, 8))
        t = qrhip.TablesFromSnapshot(bad)
        with pytest.raises(qrhip.QrError, match=message):
            device.render_tables(t.ptr, t.fd)

    def past_end(st):
        st[box[0], 7] = n_step + 1

    def node_box(st):
        st[node[0], 7] = -2

    attempt(past_end, "culling program out of range")
    attempt(node_box, "local box")


def test_gpu_more_lights_than_visibility_bytes(path_dev):
    """A hit's visibility is a byte per light with up to four lights and a
    bit per light (set by atomics) with more: config 2's four lights plus
    three moved copies of them, seven in all, give the oracle's frame."""
    import qr_oracle
    hs = HostScene(2, 1, 160, 96, 2, 4)
    try:
        snap = qrhip.tables_snapshot(hs.tables, hs.fd)
        four = hs.oracle()[0]
    finally:
        hs.close()
    words = qrhip.C.sizeof(qrhip.QrLight) // 4
    lights = snap["lights"].view(np.float32).reshape(-1, words)
    assert lights.shape[0] == 4
    extra = lights[:3].copy()
    extra[:, 0:3] += np.array([[3.0, 1.0, -2.0], [-4.0, 2.0, 1.5], [1.0, 3.5, 2.5]],
                              np.float32)
    more = np.concatenate([lights, extra])
    snap = dict(snap)
    snap["lights"] = np.ascontiguousarray(more).view(np.uint8).reshape(-1)
    counts = snap["counts"].copy()
    counts[qrhip.TABLE_COUNTS.index("n_lgt")] = more.shape[0]
    snap["counts"] = counts
    t = qrhip.TablesFromSnapshot(snap)
    want = qr_oracle.render(t.ptr, t.fd)[0]
    got, _ = path_dev.render_tables(t.ptr, t.fd)
    assert np.array_equal(got, want), int((got != want).sum())
    assert not np.array_equal(want, four), "the extra lights change the frame"


def test_gpu_plain_full_frame_bit_exact(path_dev):
    """The plain scene's infinite ground sends shadow rays from hits
    thousands of units away, whose fp32 cancellation makes false roots near
    surfaces; culling must keep every one of them: bit-identical frame."""
    hs = HostScene(1, 1, 800, 480, 0, 4)
    try:
        want = hs.oracle()[0]
        got, _ = path_dev.render_tables(hs.tables, hs.fd)
    finally:
        hs.close()
    assert np.array_equal(got, want), int((got != want).sum())


def test_gpu_full_1080p_whitted_rows(path_dev):
    """The benchmark frame itself (1920x1080, 4X AA, depth 4, 64 quadrics):
    the whole GPU frame against the oracle on 24 rows spread over it."""
    print("case full 1080p rows", flush=True)
    w, s = gpu_scene(path_dev, 2, 1, 1920, 1080, 2, 4)
    try:
        got = s.render(0)
        t, fd = s.tables()
        rows = list(range(3, 1080, 45))
        import qr_oracle
        want = qr_oracle.render(t, fd, rows=rows)[0]
    finally:
        s.destroy()
        w.close()
    assert_frame_exact(got[rows], want[rows], "1080p rows")


@pytest.mark.parametrize("seed,depth", [(41, 4), (42, 8)])
def test_gpu_queue_growth_all_glass(device, seed, depth):
    """Glass everywhere: every hit spawns two children, so the level queues
    overflow their first sizing; the frame is traced again after they grow
    and must still equal the oracle and the one-kernel path."""
    print(f"case all-glass seed {seed} depth {depth}", flush=True)
    hs = HostScene(6, seed, 160, 90, 2, depth)
    try:
        want = hs.oracle()[0]
        device.set_path(qrhip.PATH_LEVELS)
        got, _ = device.render_tables(hs.tables, hs.fd)
        device.set_path(qrhip.PATH_ONE_KERNEL)
        one, _ = device.render_tables(hs.tables, hs.fd)
    finally:
        device.set_path(qrhip.PATH_LEVELS)
        hs.close()
    assert_frame_exact(got, want, "levels")
    assert np.array_equal(got, one)


def test_gpu_repeat_and_bottom_up_frame(device):
    """Renders repeat bit for bit; a negative x_row stores rows bottom-up."""
    w, s = gpu_scene(device, 2, 31, 160, 90, 2, 4)
    w2, s2 = None, None
    try:
        a = s.render(0)
        b = s.render(1)
        assert np.array_equal(a, b)
        s.destroy()
        w2 = qrhip.Workload(2, 31)
        s2 = qrhip.Scene(device, w2.ptr, 160, 90, x_row=-192)
        s2.set_depth(4)
        c = s2.render(0)
        assert np.array_equal(a, c)
    finally:
        s.destroy()
        w.close()
        if s2 is not None:
            s2.destroy()
        if w2 is not None:
            w2.close()


def test_gpu_split_render_and_timing(device):
    w, s = gpu_scene(device, 1, 1, 800, 480, 0, 4)
    try:
        ref = s.render(0)
        s.update(0)
        assert qrhip.lib().qrhip_scene_launch(s.h) == 0
        assert qrhip.lib().qrhip_scene_download(s.h) == 0
        assert np.array_equal(s.frame(), ref)
        ms = s.time_launches(3)
        assert 0.0 < ms < 1000.0
    finally:
        s.destroy()
        w.close()


def test_gpu_rejects_bad_depth_and_tables(device):
    hs = HostScene(1, 1, 64, 32, 0, 4)
    try:
        fd = hs.fd
        fd.depth = 15
        with pytest.raises(qrhip.QrError):
            device.render_tables(hs.tables, fd)
        fd.depth = 4
        t = hs.tables.contents
        keep = t.surfaces[0].clip_cnt
        t.surfaces[0].clip_cnt = t.n_clip + 5
        with pytest.raises(qrhip.QrError, match="clip list"):
            device.render_tables(hs.tables, fd)
        t.surfaces[0].clip_cnt = keep
    finally:
        hs.close()


def test_gpu_texture_files_render_as_texel_arrays(device, tmp_path):
    """Materials that name BMP files under data/textures/ render the frame of
    the same materials with the texel arrays in place."""
    (tmp_path / "data" / "textures").mkdir(parents=True)
    qrhip.set_data_path(str(tmp_path) + "/")
    frames = []
    try:
        for files in (False, True):
            device.set_fsaa(1)
            w = qrhip.Workload(2, 79, texture_files=files)
            s = qrhip.Scene(device, w.ptr, 160, 90)
            try:
                s.set_depth(3)
                frames.append(s.render(0))
            finally:
                s.destroy()
                w.close()
    finally:
        qrhip.set_data_path("../")
    assert len(list((tmp_path / "data" / "textures").iterdir())) > 0
    assert np.array_equal(frames[0], frames[1])


@pytest.mark.parametrize("config,seed", [(9, 3), (2, 5)])
@pytest.mark.parametrize("d_eps,zero", [(0.0, 0.0), (1.0e-30, -0.0), (1.0, 0.0),
                                        (1.2621774e-29, -0.0)])
def test_gpu_root_forms(path_dev, config, seed, d_eps, zero):
    """Each way the walks form a surface's roots, on caller tables: no
    near-zero discriminants, thresholds below and at the smallest value the
    short square root takes, many of them, and linear terms of either zero
    (only +0 leaves them out); bit for bit the oracle's frame."""
    hs = HostScene(config, seed, 97, 61, 1, 3)
    try:
        snap = qrhip.tables_snapshot(hs.tables, hs.fd)
    finally:
        hs.close()
    t = qrhip.TablesFromSnapshot(snap)
    for i in range(t.tables.n_surf):
        s = t.tables.surfaces[i]
        s.d_eps = d_eps
        for a in range(3):
            if s.scj[a] == 0.0:
                s.scj[a] = zero
    want, ids_o, flags, _, _ = qr_oracle.render(t.ptr, t.fd, want_ids=True)
    got, ids = path_dev.render_tables(t.ptr, t.fd, want_ids=True)
    assert_frame_exact(got, want, f"config {config} d_eps {d_eps} zero {zero}")
    assert np.array_equal(ids[flags == 0], ids_o[flags == 0])


def _snapshot(config, seed, x, y, fsaa, depth):
    hs = HostScene(config, seed, x, y, fsaa, depth)
    try:
        return qrhip.tables_snapshot(hs.tables, hs.fd)
    finally:
        hs.close()


def _render_every_way(path_dev, t):
    """A table's (frame, ids) through the allocating and the no-alloc entry
    points."""
    return [path_dev.render_tables(t.ptr, t.fd, want_ids=True),
            path_dev.render_tables_noalloc(t.ptr, t.fd, want_ids=True)]


@pytest.mark.parametrize("config,depth", [(1, 0), (1, 4), (9, 0), (9, 5)])
def test_gpu_world_surfaces_with_a_transform(path_dev, config, depth):
    """Caller tables whose surfaces are traced in world coordinates (shift 0)
    though they carry a transform (trm): their transform node, an identity
    rotation, turns their normals; their own matrix is read by nothing.  The
    frame and the first-hit ids are those of the tables without transforms."""
    snap = _snapshot(config, 21, 95, 63, 1, depth)
    t = qrhip.TablesFromSnapshot(snap)
    want, ids_o, flags, _, _ = qr_oracle.render(t.ptr, t.fd, want_ids=True)
    t = qrhip.TablesFromSnapshot(snap)
    world = [i for i in range(t.tables.n_surf)
             if t.tables.surfaces[i].tag >= 0 and t.tables.surfaces[i].trm == 0]
    assert len(world) >= 5
    rng = np.random.default_rng(config)
    for k, i in enumerate(world):
        s = t.tables.surfaces[i]
        s.trm = 2 if k == 0 else 1 + k % 3
        s.trnode = world[0]
        for r in range(3):
            for c in range(3):
                s.tc[r][c] = float(r == c) if k == 0 else float(rng.uniform(-2.0, 2.0))
    for got, ids in _render_every_way(path_dev, t):
        assert_frame_exact(got, want, f"config {config} depth {depth}")
        assert np.array_equal(ids[flags == 0], ids_o[flags == 0])


@pytest.mark.parametrize("config,depth", [(2, 0), (2, 4), (9, 0), (9, 5)])
def test_gpu_world_surfaces_in_a_group(path_dev, config, depth):
    """Caller tables with surfaces traced in world coordinates (shift 0)
    inside a transform node's group: the ray's direction stays the world's
    and its origin is the one the node left, as in QuadRay's list walk; bit
    for bit the oracle's frame.  (No culling program: its local boxes are for
    surfaces in the node's frame.)"""
    snap = _snapshot(config, 22, 93, 59, 1, depth)
    t = qrhip.TablesFromSnapshot(snap)
    t.tables.n_step = t.tables.n_step_any = 0
    changed = 0
    for i in range(t.tables.n_surf):
        s = t.tables.surfaces[i]
        if s.tag >= 0 and s.shift != 0 and s.trnode not in (-1, i):
            changed += 1
            if changed % 2 == 1:
                s.shift = s.trm = s.apex = 0
                s.trnode = -1
    assert changed >= 4
    want, ids_o, flags, _, _ = qr_oracle.render(t.ptr, t.fd, want_ids=True)
    for got, ids in _render_every_way(path_dev, t):
        assert_frame_exact(got, want, f"config {config} depth {depth}")
        assert np.array_equal(ids[flags == 0], ids_o[flags == 0])


@pytest.mark.parametrize("config,depth", [(1, 2), (9, 2), (2, 2)])
def test_gpu_planes_have_no_apex(path_dev, config, depth):
    """An apex kind in a plane's record changes nothing, whatever its
    thresholds: bit for bit the oracle's frame."""
    t = qrhip.TablesFromSnapshot(_snapshot(config, 25, 95, 61, 1, depth))
    for i in range(t.tables.n_surf):
        s = t.tables.surfaces[i]
        if s.solver == 1:
            s.apex, s.d_eps, s.t_eps = 1 + i % 2, 1.0e6, 1.0e6
    want, ids_o, flags, _, _ = qr_oracle.render(t.ptr, t.fd, want_ids=True)
    for got, ids in _render_every_way(path_dev, t):
        assert_frame_exact(got, want, f"config {config}")
        assert np.array_equal(ids[flags == 0], ids_o[flags == 0])


@pytest.mark.parametrize("config,depth", [(1, 0), (1, 3), (9, 0), (9, 3)])
@pytest.mark.parametrize("back", [False, True])
def test_gpu_equal_distances(path_dev, config, depth, back):
    """Coincident surfaces, whose roots are equal: the later one of the list
    is seen, also at distances below zero ("back": a camera turned away, with
    a near clip behind it); bit for bit the oracle's frame."""
    snap = _snapshot(config, 23, 95, 61, 1, depth)
    t = qrhip.TablesFromSnapshot(snap)
    t.tables.n_step = t.tables.n_step_any = 0
    world = [i for i in range(t.tables.n_surf)
             if t.tables.surfaces[i].tag >= 0 and t.tables.surfaces[i].shift == 0]
    assert len(world) >= 5
    for a, b in zip(world[0::2], world[1::2]):
        keep = {k: list(getattr(t.tables.surfaces[b], k)) for k in ("mat", "props")}
        own = t.tables.surfaces[b].id
        C.memmove(C.byref(t.tables.surfaces[b]), C.byref(t.tables.surfaces[a]),
                  C.sizeof(qrhip.QrSurface))
        t.tables.surfaces[b].id = own
        for k, v in keep.items():
            for side in range(2):
                getattr(t.tables.surfaces[b], k)[side] = v[side]
    if back:
        t.fd.t_min = -1.0e30
        for field in ("dir", "hor", "ver"):
            v = getattr(t.fd, field)
            for k in range(len(v)):
                v[k] = -v[k]
    want, ids_o, flags, _, _ = qr_oracle.render(t.ptr, t.fd, want_ids=True)
    assert (ids_o >= 0).any()
    for got, ids in _render_every_way(path_dev, t):
        assert_frame_exact(got, want, f"config {config} depth {depth} back {back}")
        assert np.array_equal(ids[flags == 0], ids_o[flags == 0])


@pytest.mark.parametrize("config,x,y,fsaa,depth", [
    # 16 lanes to a sample: the smallest frame, ragged edges of every tile
    # shape, the largest number of samples; then 4, 2 and 1 lanes
    (2, 1, 1, 0, 4), (4, 37, 23, 1, 4), (6, 29, 31, 2, 8), (2, 512, 512, 0, 2),
    (4, 513, 513, 0, 2), (2, 363, 367, 1, 3), (6, 259, 257, 2, 4),
    (2, 1801, 1203, 0, 2), (2, 1449, 733, 1, 2), (2, 751, 749, 2, 2),
    (2, 2063, 2049, 0, 1), (2, 1451, 1449, 1, 1), (2, 1025, 1031, 2, 1),
    # without secondary rays a sixteenth of the samples takes each of them
    (1, 128, 128, 0, 4), (1, 131, 127, 0, 4), (2, 363, 367, 0, 0), (4, 363, 367, 1, 0),
])
def test_gpu_one_kernel_lanes_per_sample(device, config, x, y, fsaa, depth):
    """However many lanes trace a sample, and over ragged tiles, the frame and
    the first-hit ids are those of the level pipeline, or of the oracle where
    a frame without secondary rays would take the one kernel on both paths."""
    device.set_fsaa(fsaa)
    hs = HostScene(config, 51, x, y, fsaa, depth)
    try:
        same = np.ones(1, dtype=bool)
        if config == 1 or depth == 0:
            want, wid, flags, _, _ = hs.oracle(want_ids=True)
            same = flags == 0
        else:
            want, wid = device.render_tables(hs.tables, hs.fd, want_ids=True)
        device.set_path(qrhip.PATH_ONE_KERNEL)
        got, gid = device.render_tables(hs.tables, hs.fd, want_ids=True)
    finally:
        device.set_path(qrhip.PATH_LEVELS)
        hs.close()
    assert np.array_equal(got, want)
    assert not np.any((gid != wid) & same)


@pytest.mark.parametrize("config,x,y,fsaa,depth", [
    # without secondary rays: 16, 4 and 1 lanes to a sample, ragged tiles, one
    # light and four, and either side of the size a dense scene changes path at
    (1, 1, 1, 2, 4), (1, 127, 129, 0, 4), (1, 131, 127, 0, 4), (1, 181, 187, 1, 4),
    (1, 363, 367, 0, 4), (2, 257, 259, 1, 0), (4, 37, 23, 2, 0), (4, 91, 95, 2, 0),
    (11, 363, 361, 0, 0), (11, 363, 363, 0, 0),
])
def test_gpu_frames_without_secondary_rays(path_dev, config, x, y, fsaa, depth):
    hs = HostScene(config, 52, x, y, fsaa, depth)
    try:
        want, wid, flags, _, _ = hs.oracle(want_ids=True)
        got, gid = path_dev.render_tables(hs.tables, hs.fd, want_ids=True)
    finally:
        hs.close()
    assert_frame_exact(got, want, "frame")
    assert not np.any((gid != wid) & (flags == 0))


def test_gpu_scene_creation_waits_for_no_other_work(device):
    """A scene with a frame of its own is made, blank, while the program's
    default stream is busy, or the device's own."""
    rt, n = qrhip.lib(), 1 << 31
    buf = C.c_void_p()
    assert rt.hipMalloc(C.byref(buf), C.c_size_t(n)) == 0
    works = [qrhip.Workload(2, 54 + k) for k in range(3)]
    scenes = [qrhip.Scene(device, works[0].ptr, 1920, 1080)]
    try:
        scenes[0].set_depth(8)
        scenes[0].render(0)
        assert rt.hipMemset(buf, 0, C.c_size_t(n)) == 0
        for _ in range(100):            # tens of milliseconds
            assert rt.hipMemsetAsync(buf, 0, C.c_size_t(n), None) == 0
        scenes.append(qrhip.Scene(device, works[1].ptr, 1281, 719))
        busy = rt.hipStreamQuery(None)
        assert not scenes[1].frame().any()
        assert rt.hipDeviceSynchronize() == 0
        for _ in range(20):
            qrhip.check(rt.qrhip_scene_launch(scenes[0].h))
        scenes.append(qrhip.Scene(device, works[2].ptr, 1281, 719))
        assert not scenes[2].frame().any()
        qrhip.check(rt.qrhip_scene_sync(scenes[0].h))
    finally:
        assert rt.hipFree(buf) == 0
        for s in scenes:
            s.destroy()
        for w in works:
            w.close()
    assert busy == 600      # hipErrorNotReady: the fills were still running


def test_gpu_depth_changes_path_between_frames(device):
    """A scene's frames with and without secondary rays in turn: queues that
    overflow in the one kind leave nothing to check in the other."""
    w, s = gpu_scene(device, 6, 53, 160, 90, 2, 8)
    got = []
    try:
        for depth in (0, 8, 0, 8):
            s.set_depth(depth)
            got.append(s.render(0).copy())
    finally:
        s.destroy()
        w.close()
    for depth, frame in zip((0, 8, 0, 8), got):
        hs = HostScene(6, 53, 160, 90, 2, depth)
        try:
            assert_frame_exact(frame, hs.oracle()[0], depth)
        finally:
            hs.close()
