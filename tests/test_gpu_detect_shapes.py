"""GPU: launch shapes of the collision query that the settings and the front
lengths choose, against the oracle."""
import numpy as np
import pytest

from oibvh_amd import meshgen as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from oibvh_amd import api as A

    return A


def scene_of(api, ctx, meshes):
    trees = [api.OibvhTree(ctx, *m) for m in meshes]
    scene = api.Scene(ctx)
    for t in trees:
        t.build()
        scene.addOibvhTree(t)
    return scene, trees


@pytest.mark.parametrize("blocks", [1, 3, 64, 513])
@pytest.mark.parametrize("entry, expand", [(0, 1), (4, 2), (4, 3)])
def test_walks_by_few_workgroups(api, ctx, orc, blocks, entry, expand):
    """Walks that traverse_blocks holds to 1 to 513 workgroups: every workgroup
    takes several shares of the front. Pairs, statistics and front lengths are
    those of the default."""
    print(f"walk by {blocks} workgroups, entry {entry}, expand {expand}", flush=True)
    a, b = M.icosphere(4, 1.0, 0.02, 5), M.icosphere(4, 1.0, 0.02, 6, center=(0.2, 0.1, 0.0))
    scene, _ = scene_of(api, ctx, [a, b])
    want = orc.detect([orc.Tree(*a), orc.Tree(*b)])
    assert len(want) > 500
    scene.detectCollision(entry, expand)
    tests, levels = scene.stats()["bvtt_tests"], scene.level_counts()
    base = ctx.get_tuning()
    ctx.set_tuning(traverse_blocks=blocks)
    try:
        scene.detectCollision(entry, expand)
        assert np.array_equal(scene.getIntTriPairs(), want)
        assert scene.stats()["bvtt_tests"] == tests
        assert np.array_equal(scene.level_counts(), levels)
    finally:
        ctx.set_tuning(**base)


def cloud(n, size, seed, spread=1.0):
    r = np.random.default_rng(seed)
    xyz = r.uniform(-spread, spread, (n, 1, 3)) + r.uniform(-size, size, (n, 3, 3))
    return xyz.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)


@pytest.mark.parametrize("mode", ["fp32", "separate", "fp64"])
def test_steps_that_keep_every_pair(api, ctx, orc, mode):
    """Three-level steps (after a head walk of one step, so that none is a walk) over
    clouds in which every box meets every other: 64 pairs kept per front pair, many
    times what the rings in LDS hold, all of one kind, both kinds in one tile (trees of
    unequal depth), and against itself: the oracle's pairs."""
    print(f"steps that keep every pair, {mode}", flush=True)
    fp64 = mode == "fp64"
    a, b, small = cloud(700, 2.0, 1, 0.1), cloud(650, 2.0, 2, 0.1), cloud(40, 2.0, 3, 0.1)
    base = ctx.get_tuning()
    ctx.set_tuning(traverse_local=1, traverse_local_levels=1, narrow_separate=1 if mode == "separate" else 0)
    try:
        for meshes, entry, self_collide in (([a, b], 1, False), ([a, small], 1, False), ([a, b, small], 3, False),
                                            ([b], 3, True)):
            scene, trees = scene_of(api, ctx, meshes)
            scene.detectCollision(entry, 3, self_collide=self_collide, fp64_fallback=fp64)
            want = orc.detect([orc.Tree(x, f, order=t.perm()) for (x, f), t in zip(meshes, trees)],
                              self_collide=self_collide, fp64=fp64)
            assert len(want) > 5000
            assert np.array_equal(scene.getIntTriPairs(), want), (len(meshes), entry)
            if len(meshes) == 2 and meshes[1] is b:
                # nodes of the levels 1, 4 and 7 over 700 and 650 leaves
                levels = scene.level_counts()
                assert list(levels[:2]) == [2 * 2, 11 * 11] and levels[2] > 0.9 * 88 * 82
    finally:
        ctx.set_tuning(**base)


@pytest.mark.parametrize("batched", [False, True])
def test_walks_over_clouds_that_meet_and_part(api, ctx, orc, batched):
    """Two clouds whose fronts grow far faster than guessed: the steps are planned
    again after the first query, and back after the clouds have parted. Always the
    oracle's pairs, front lengths and statistics of the first query."""
    print(f"walks over clouds, batched={batched}", flush=True)
    a, b = cloud(20000, 0.1, 1), cloud(20000, 0.1, 2)
    far = (b[0] + np.float32(1.9), b[1])
    on = {"near": b, "far": far}
    device = {k: api.DeviceBuffer.from_array(v[0]) for k, v in on.items()}
    if batched:
        obj = api.Batch(ctx)
        for m in (a, b):
            obj.add_mesh(0, *m)
        obj.build()
    else:
        obj, trees = scene_of(api, ctx, [a, b])
        order = trees[1].perm()
    want, seen = {}, {}
    for k, (xyz, f) in on.items():
        order = obj.perm(1) if batched else order
        want[k] = orc.detect([orc.Tree(*a), orc.Tree(xyz, f, order=order)])
    assert len(want["near"]) > 20000 > len(want["far"])
    for k in ("near", "near", "near", "far", "far", "near", "near"):
        if batched:
            obj.set_positions_device(1, device[k].ptr.value)
            obj.frame(4, 3)
            got = obj.pairs()
        else:
            trees[1].set_positions_device(device[k].ptr.value)
            obj.frame(None, 4, 3)
            got = obj.getIntTriPairs()
        assert np.array_equal(got, want[k]), k
        levels, stats = obj.level_counts(), obj.stats()
        if k not in seen:
            seen[k] = levels, stats["bvtt_tests"], stats["candidates"]
        assert np.array_equal(levels, seen[k][0]) and (stats["bvtt_tests"], stats["candidates"]) == seen[k][1:], k
    assert seen["near"][0].max() > 1 << 17 > seen["far"][0].max()


def test_checks_with_blocking_waits(api, ctx, orc):
    """The same results in a program whose waits block (hipDeviceScheduleBlockingSync)."""
    from oibvh_amd import _lib

    print("checks with blocking waits", flush=True)
    a, b = M.icosphere(4, 1.0, 0.02, 5), M.icosphere(4, 1.0, 0.02, 6, center=(0.2, 0.1, 0.0))
    scene, _ = scene_of(api, ctx, [a, b])
    want = orc.detect([orc.Tree(*a), orc.Tree(*b)])
    hip = _lib.hip()
    hip.hipSetDeviceFlags.argtypes = [_lib.C.c_uint]
    assert hip.hipSetDeviceFlags(4) == 0
    try:
        for _ in range(3):
            scene.detectCollision(4, 3)
            assert np.array_equal(scene.getIntTriPairs(), want)
            assert scene.pairs_device()[1] == len(want)
    finally:
        assert hip.hipSetDeviceFlags(0) == 0
