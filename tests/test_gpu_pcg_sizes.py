"""The PCG at the world sizes where its sums and loops change form: up to 64,
512 and more partials per kernel, more groups than update workgroups (2048)
and more rows than one pass of the product (4096), single worlds and batched.
Stacks of 20 touching cubes (one component larger than a preconditioner
group) among single cubes.  Nothing couples the components, so each stack's
direction is the oracle's for the stack alone, and a single cube's the
oracle's for it.  1e-7 of the largest entry: both solve to 1e-12 of the
residual, and the stiffness of the touching cubes amplifies that by up to 1e5."""
import numpy as np
import pytest

import oracle_lib as O
from adb_amd import scenes
from adb_amd.capi import default_params
from adb_amd.world import World

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

D_HAT, STACK = 1e-3, 20


@pytest.mark.parametrize("B,batched", [(64, False), (65, False), (257, False), (512, False), (513, False), (2049, False),
                                       (4100, False), (8300, False), (65, True), (600, True), (4500, True)])
def test_direction_of_independent_stacks(B, batched):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    v, f, e = scenes.cube_mesh()
    rng = np.random.default_rng(B)
    p = default_params(d_hat=D_HAT, mu=0.4, enable_ground=0)
    n_stack = 3
    bodies = []
    jit = rng.uniform(-0.05, 0.05, (STACK, 2))
    for s in range(n_stack):
        for i in range(STACK):
            bodies.append(dict(verts=v, tris=f, edges=e, R=np.eye(3), v=(0.0, -0.1 * i, 0.0),
                               p=(4.0 * s + jit[i, 0], (1.0 + 0.5 * np.sqrt(D_HAT)) * i, jit[i, 1])))
    for k in range(B - n_stack * STACK):
        bodies.append(dict(verts=v, tris=f, edges=e, R=np.eye(3), v=(0.0, 0.3, 0.1), p=(3.0 * (k % 100), 3.0 * (k // 100), 10.0)))
    cube = scenes.build_scene(bodies[-1:])
    off = [0] + [STACK * (s + 1) for s in range(n_stack)] + ([] if B == n_stack * STACK else [B])
    w = World(scenes.build_scene(bodies), p, scene_offsets=off) if batched else World(scenes.build_scene(bodies), p)
    rc, dq = w.newton_direction()
    dq = dq.reshape(B, 12)
    rs, ds = O.OracleWorld(cube, p).newton_direction()
    assert rc == rs == 0
    for s in range(n_stack):
        # the oracle of this very stack: where the edges are exactly parallel, a
        # translation's rounding decides which features are nearest (2e-3 of
        # the direction between the oracle's own answers)
        ow = O.OracleWorld(scenes.build_scene(bodies[STACK * s:STACK * (s + 1)]), p)
        pt, ee, _ = ow.collision_set()
        assert len(pt) + len(ee) > 10 * STACK
        ro, do = ow.newton_direction()
        assert ro == 0
        do = do.reshape(STACK, 12)
        tol = 1e-7 * np.abs(do).max()
        np.testing.assert_allclose(dq[STACK * s:STACK * (s + 1)], do, rtol=0, atol=tol)
    np.testing.assert_allclose(dq[n_stack * STACK:], np.repeat(ds.reshape(1, 12), B - n_stack * STACK, axis=0), rtol=0, atol=tol)


def column(n, rng):
    gap = 0.5 * np.sqrt(D_HAT)
    return [(rng.uniform(-0.05, 0.05), (1.0 + gap) * i, rng.uniform(-0.05, 0.05)) for i in range(n)], []


def wall(w, h, d):
    def make(rng):
        step = 1.0 + 0.5 * np.sqrt(D_HAT)
        return [(step * i, step * j, step * k) for k in range(d) for j in range(h) for i in range(w)], []
    return make


def shelf(n, rng):
    # columns of 10 cubes, each on a static cube of its own
    gap = 0.5 * np.sqrt(D_HAT)
    pos = [(3.0 * c, (1.0 + gap) * i, 0.0) for c in range(n) for i in range(11)]
    return pos, [11 * c for c in range(n)]


SHAPES = {
    # a path one body longer than an explicit inverse takes; the shortest and
    # the longest that a component's factors take, and one more or less (which
    # keep the small groups)
    "path9": lambda rng: column(9, rng), "path16": lambda rng: column(16, rng), "path17": lambda rng: column(17, rng), "path256": lambda rng: column(256, rng), "path257": lambda rng: column(257, rng),
    # cycles and fill: every cube of a wall touches its eight neighbours
    "wall3x4": wall(3, 4, 1), "wall4x10": wall(4, 10, 1),
    # too dense to eliminate: 26 neighbours
    "block4x4x4": wall(4, 4, 4),
    "static": lambda rng: shelf(3, rng),
}


@pytest.mark.parametrize("psd", [1, 0])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_direction_of_one_component(shape, psd):
    """Contact components as one preconditioner group (more than 8 bodies):
    the direction against the oracle's direct solve; tolerance as above."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    v, f, e = scenes.cube_mesh()
    rng = np.random.default_rng(7)
    pos, static = SHAPES[shape](rng)
    mass = rng.uniform(500.0, 2000.0, len(pos))
    mass[static] = -1.0
    bodies = [dict(verts=v, tris=f, edges=e, R=np.eye(3), p=q, mass=float(m)) for q, m in zip(pos, mass)]
    sc = scenes.build_scene(bodies)
    p = default_params(d_hat=D_HAT, mu=0.4, enable_ground=0, psd=psd)
    w, ow = World(sc, p), O.OracleWorld(sc, p)
    pt, ee, _ = ow.collision_set()
    assert len(pt) + len(ee) > 10 * len(pos)
    rg, dg = w.newton_direction()
    ro, do = ow.newton_direction()
    assert rg == ro == 0
    np.testing.assert_allclose(dg, do, rtol=0, atol=1e-7 * np.abs(do).max())
