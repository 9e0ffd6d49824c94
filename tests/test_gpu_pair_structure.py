"""The pair structure of worlds of many body pairs and few bodies: two crossed
layers of rods, every rod of one in contact with every rod of the other, around
the number of pairs (8192) from which several workgroups build it.  The
direction, with the residual of the system that adb_assemble returns: 1e-9 of
the gradient, a thousand times the solver's relative tolerance."""
import numpy as np
import pytest

from adb_amd import scenes
from adb_amd.capi import default_params
from adb_amd.world import World

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

D_HAT = 1e-3


@pytest.mark.parametrize("a,b", [(64, 128), (83, 99), (1, 1), (150, 150)])
def test_direction_of_crossed_rods(a, b):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    along_x, along_z = scenes.cube_mesh((0.4 * b, 0.1, 0.1)), scenes.cube_mesh((0.1, 0.1, 0.4 * a))
    bodies = [dict(verts=along_x[0], tris=along_x[1], edges=along_x[2], p=(0.0, 0.0, 0.3 * (i - 0.5 * (a - 1)))) for i in range(a)]
    bodies += [dict(verts=along_z[0], tris=along_z[1], edges=along_z[2], p=(0.3 * (j - 0.5 * (b - 1)), 0.1 + 0.5 * np.sqrt(D_HAT), 0.0))
               for j in range(b)]
    w = World(scenes.build_scene(bodies), default_params(d_hat=D_HAT, mu=0.4, enable_ground=0))
    pt, ee, _ = w.collision_set()
    pairs = np.unique(np.concatenate([pt[:, [0, 2]], ee[:, [0, 2]]]), axis=0)
    assert np.array_equal(pairs, [(i, a + j) for i in range(a) for j in range(b)])
    g, H = w.assemble()
    rc, dq = w.newton_direction()
    assert rc == 0
    assert np.linalg.norm(H @ dq + g) <= 1e-9 * np.linalg.norm(g)
    # every pair's block, and none elsewhere
    n = a + b
    blocks = np.abs(H.reshape(n, 12, n, 12)).max(axis=(1, 3)) > 0
    want = np.eye(n, dtype=bool)
    want[:a, a:] = want[a:, :a] = True
    assert np.array_equal(blocks, want)
