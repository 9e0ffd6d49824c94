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
