"""GPU: builds at the sizes where the Morton launch changes its shape."""
import numpy as np
import pytest

from oibvh_amd import meshgen as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m63", [False, True])
@pytest.mark.parametrize("F", [512 * 1024, 512 * 1024 + 1, 1024 * 1024, 1024 * 1024 + 1, 2 * 1024 * 1024 + 1])
def test_build_morton_shapes(ctx, orc, F, m63):
    """2, 4 and again 2 faces a thread: the leaf order is the oracle's."""
    from oibvh_amd import api

    print(f"build of {F} faces, m63={m63}", flush=True)
    r = M.Rng(F)
    xyz = r.uniform((F + 2) * 3, -1.0, 1.0).reshape(-1, 3).astype(np.float32)
    f = r.integers(F * 3, 0, F + 1).reshape(F, 3).astype(np.uint32)
    t = api.OibvhTree(ctx, xyz, f)
    t.set_morton_bits(63 if m63 else 30)
    t.build()
    assert np.array_equal(t.perm(), orc.Tree(xyz, f, order="morton63" if m63 else "morton").order)
