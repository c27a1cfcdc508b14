"""Seeded random frames over every tracing kernel, bit for bit: the level
pipeline, the one-kernel tracer with and without a tree at each number of
lanes per sample, the no-alloc entry point and the path tracer, against the
oracle (whole frames of small ones, sampled rows of large ones).  Scenes,
sizes, anti-aliasing and depths are drawn, so a kernel that a compiler or an
edit breaks for some of them is met (a seed's frames stay the same)."""
import math
import random

import numpy as np
import pytest

import qr_oracle
import qrhip
from helpers import HostScene, assert_frame_exact

pytestmark = pytest.mark.gpu

CONFIGS = (1, 2, 2, 4, 6, 6, 7, 9, 9, 10)


def draw(rng, lo, hi):
    x = int(round(lo * (hi / lo) ** rng.random()))
    y = max(lo // 2, int(x * rng.uniform(0.4, 0.9)))
    return (rng.choice(CONFIGS), rng.randrange(1, 10000), x, y, rng.randrange(3),
            rng.choice((0, 0, 1, 2, 3, 4, 6, 9)))


def each_way(device, hs):
    """(name, frame, ids) of a host scene's tables through each Whitted path."""
    for name, path in (("levels", qrhip.PATH_LEVELS), ("one kernel", qrhip.PATH_ONE_KERNEL)):
        device.set_path(path)
        try:
            yield (name, *device.render_tables(hs.tables, hs.fd, want_ids=True))
        finally:
            device.set_path(qrhip.PATH_LEVELS)
    yield ("no-alloc", *device.render_tables_noalloc(hs.tables, hs.fd, want_ids=True))


@pytest.mark.parametrize("seed", range(6))
def test_random_small_frames(device, seed):
    rng = random.Random(seed)
    for _ in range(25):
        case = draw(rng, 6, 110)
        print(f"case {case}", flush=True)
        hs = HostScene(*case)
        try:
            want, ids_o, flags, _, _ = hs.oracle(want_ids=True)
            for name, got, ids in each_way(device, hs):
                assert_frame_exact(got, want, f"{case} {name}")
                assert np.array_equal(ids[flags == 0], ids_o[flags == 0]), (case, name)
        finally:
            hs.close()


@pytest.mark.parametrize("seed", range(4))
def test_random_large_frames(device, seed):
    """Frames of every number of lanes per sample (they change at 2^14 and
    2^17 samples without a tree, 2^18, 2^21 and 2^22 with one)."""
    rng = random.Random(100 + seed)
    for k in range(8):
        config, s, _, _, fsaa, depth = draw(rng, 6, 110)
        n = 2.0 ** rng.uniform(14.5 + k, 15.5 + k)
        x = int(math.sqrt(n / (1, 2, 4)[fsaa] * rng.uniform(1.0, 2.0)))
        y = max(1, int(n / (1, 2, 4)[fsaa] / x))
        case = (config, s, x, y, fsaa, depth)
        print(f"case {case}", flush=True)
        hs = HostScene(*case)
        try:
            rows = sorted(set(rng.randrange(y) for _ in range(3)))
            want = hs.oracle(rows=rows)[0]
            frames = list(each_way(device, hs)) if n < 1 << 21 else list(each_way(device, hs))[:2]
            for name, got, ids in frames:
                for r in rows:
                    assert np.array_equal(got[r], want[r]), (case, name, r)
                assert np.array_equal(got, frames[0][1]), (case, name)
                assert np.array_equal(ids, frames[0][2]), (case, name)
        finally:
            hs.close()


@pytest.mark.parametrize("seed", range(4))
def test_random_path_traced_frames(device, seed):
    """Two passes of small frames from random planes' seeds: planes, seeds
    and frame."""
    rng = random.Random(200 + seed)
    for _ in range(8):
        _, s, x, y, fsaa, _ = draw(rng, 6, 90)
        case = (rng.choice((2, 3, 3, 3, 6, 9, 10)), s, x, y, fsaa, rng.choice((0, 1, 3, 5, 8, 10)))
        print(f"case {case}", flush=True)
        hs = HostScene(*case)
        try:
            slots = x * y * (1, 2, 4)[fsaa]
            hs.fd.pt_on = 1
            out = []
            for render in (qr_oracle.render_pt, device.render_tables_pt):
                planes = np.zeros((3, slots), dtype=np.float32)
                seeds = np.random.default_rng(seed).integers(0, 1 << 32, slots, dtype=np.uint32)
                for p in (1.0, 2.0):
                    hs.fd.pts_c = p
                    frame = render(hs.tables, hs.fd, planes, seeds)
                out.append((frame, planes, seeds))
        finally:
            hs.close()
        for a, b in zip(*out):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), case
