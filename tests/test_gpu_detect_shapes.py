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
