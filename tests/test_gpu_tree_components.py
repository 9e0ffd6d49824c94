"""Contact components of more than 16 bodies, which are one preconditioner
group with block Cholesky factors where their elimination fills in little:
that these components take that path, seen in the PCG iterations of a step of
one Newton iteration, and what a lost pivot costs."""
import os
import re
import subprocess
import sys

import numpy as np
import pytest

import oracle_lib as O
from adb_amd import scenes
from adb_amd.capi import default_params
from adb_amd.world import World

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

D_HAT = 1e-3
GAP = 0.5 * np.sqrt(D_HAT)


def one_iteration(pos, **params):
    """Statistics of a step of one Newton iteration of unit cubes at pos."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    v, f, e = scenes.cube_mesh()
    sc = scenes.build_scene([dict(verts=v, tris=f, edges=e, R=np.eye(3), p=q) for q in pos])
    w = World(sc, default_params(d_hat=D_HAT, enable_ground=0, max_iter=1, **params))
    return w.step(allow_not_converged=True)[1]


def column(n, seed, gaps=()):
    rng = np.random.default_rng(seed)
    y, pos = 0.0, []
    for i in range(n):
        pos.append((rng.uniform(-0.05, 0.05), y, rng.uniform(-0.05, 0.05)))
        y += 1.0 + dict(gaps).get(i, GAP)
    return pos


@pytest.mark.parametrize("seed", range(4))
def test_a_lost_pivot_costs_a_few_iterations(seed):
    """Two bodies of a column of 40 at a distance of 1e-12: their contacts are
    4e21 against an inertia of 1e3, so pivots of the Schur complements are
    rounding errors of either sign.  Each changed pivot is a change of rank one
    to the preconditioner: a few iterations each by the theory, at most 67 for
    up to 3 of them in a NumPy model of the solve; 200 here, of a limit of 2000."""
    st = one_iteration(column(40, seed, {9: 1e-12}.items()), mu=0.0, kappa=1e-2)
    assert 0 < st.pcg_iters <= 200


CAPTURES = """
import sys
import numpy as np
sys.path[:0] = [%r, %r]
from test_gpu_tree_components import D_HAT, column
import oracle_lib as O
from adb_amd import scenes
from adb_amd.capi import default_params
from adb_amd.world import World

v, f, e = scenes.cube_mesh()
pos = [(x + 3.0 * c, y, z) for c in range(%d) for x, y, z in column(17, c)]
sc = scenes.build_scene([dict(verts=v, tris=f, edges=e, R=np.eye(3), p=q) for q in pos])
w = World(sc, default_params(d_hat=D_HAT, enable_ground=0))
apart = sc["q0"].copy()
apart[:17, 1] += 0.5 * np.arange(17)
for k in range(12):
    w.set_state(apart if k %% 2 else sc["q0"])
    w.newton_direction()
print("done")
"""


@pytest.mark.parametrize("columns", [1, 3])
def test_the_solver_graph_survives_a_changing_number_of_components(columns):
    """12 directions between which a column falls apart and forms again: its
    batch of PCG iterations is captured at most once per form of the update
    kernel (the runtime's own log of its calls, from a process of its own)."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    tests = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-c", CAPTURES % (os.path.dirname(tests), tests, columns)], capture_output=True,
                       text=True, env=dict(os.environ, AMD_LOG_LEVEL="3"))
    assert r.returncode == 0 and "done" in r.stdout, r.stderr[-2000:]
    calls = re.findall(r"\b(hip[A-Z]\w*) ?\(", r.stderr)
    assert calls.count("hipLaunchKernel") > 100
    assert 1 <= calls.count("hipGraphInstantiate") <= 2


def wall(w, h, d=1, at=(0.0, 0.0, 0.0)):
    s = 1.0 + GAP
    return [(at[0] + s * i, at[1] + s * j, at[2] + s * k) for k in range(d) for j in range(h) for i in range(w)]


LAUNCHES = """
import sys
sys.path[:0] = [%r, %r]
from test_gpu_tree_components import column, one_iteration, wall

st = one_iteration(column(17, 0) + wall(8, 8, at=(10.0, 0.0, 0.0)), mu=0.4)
print("iterations", st.pcg_iters)
"""


def test_components_are_solved_once_beside_a_slow_one():
    """A wall of 8 x 8 cubes, spread over several groups, takes hundreds of PCG
    iterations; the column of 17 beside it is solved after a few, and the
    update kernel that holds its solve (last template argument true or 1) is
    not launched again in the others (the runtime's log of its launches)."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    tests = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-c", LAUNCHES % (os.path.dirname(tests), tests)], capture_output=True, text=True,
                       env=dict(os.environ, AMD_LOG_LEVEL="3", ADB_PCG_GRAPH="0"))
    assert r.returncode == 0, r.stderr[-2000:]
    assert int(re.search(r"iterations (\d+)", r.stdout).group(1)) > 50
    updates = re.findall(r"ShaderName : .*k_pcg_update<([^>]*)>", r.stderr)
    trees = [u for u in updates if u.split(",")[-1].strip() in ("true", "1")]
    assert len(updates) > 50 and 1 <= len(trees) <= 8


@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("psd", [1, 0])
def test_direction_beside_other_components(batched, psd):
    """Columns of 17 and 40 (block factors), a wall of 8 x 8 and a block of 4 x 4
    x 2 (several groups each), a column of 12, single cubes: the direction
    against the oracle's direct solve of each component, 1e-7 of the largest
    entry as for components alone; batched, also with scenes that hold one kind
    only."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    parts = [column(17, 1), wall(8, 8), column(40, 2), wall(4, 4, 2), column(12, 3), [(0.0, 0.0, 0.0)]]
    v, f, e = scenes.cube_mesh()
    p = default_params(d_hat=D_HAT, enable_ground=0, mu=0.4, psd=psd)
    rng = np.random.default_rng(5)
    bodies, want = [], []
    for k, part in enumerate(parts):
        mine = [dict(verts=v, tris=f, edges=e, R=np.eye(3), p=(x + 16.0 * k, y, z), mass=rng.uniform(500.0, 2000.0)) for x, y, z in part]
        ro, do = O.OracleWorld(scenes.build_scene(mine), p).newton_direction()
        assert ro == 0
        bodies += mine
        want.append(do.reshape(-1, 12))
    n = np.cumsum([0] + [len(q) for q in parts])
    # scenes: the first column; the wall and the second column; the rest
    w = World(scenes.build_scene(bodies), p, [0, n[1], n[3], n[6]] if batched else None)
    rc, dq = w.newton_direction()
    assert rc == 0
    for a, b, d in zip(n[:-1], n[1:], want):
        np.testing.assert_allclose(dq.reshape(-1, 12)[a:b], d, rtol=0, atol=1e-7 * np.abs(d).max())


def bricks(w, h):
    """Running bond: each cube rests on two of the row below."""
    return [((1.0 + 3.0 * GAP) * i + (0.5 if j % 2 else 0.0), (1.0 + GAP) * j, 0.0) for j in range(h) for i in range(w)]


@pytest.mark.parametrize("pos,exact", [(column(17, 0), True), (column(256, 1), True), (wall(3, 6), True), (wall(4, 10), True), (bricks(6, 6), True),
                                       (column(16, 2), False), (column(257, 3), False), (wall(4, 4, 4), False)],
                         ids=["path17", "path256", "wall3x6", "wall4x10", "bricks6x6", "path16", "path257", "block4x4x4"])
def test_factored_components_are_solved_at_once(pos, exact):
    """A component with factors is solved exactly: 1 iteration in exact
    arithmetic, 3 allowed for the rounding of the stiff contacts (a NumPy model:
    at most 3 at distances down to 1e-9).  One that is spread over several
    groups of 8 is not solved in so few."""
    st = one_iteration(pos, mu=0.4)
    assert st.n_pt + st.n_ee > 0 and st.pcg_not_converged == 0
    assert 1 <= st.pcg_iters <= 3 if exact else st.pcg_iters > 6
