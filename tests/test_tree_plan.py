"""The elimination plan of contact components (adb_amd/csrc/tree.h) on the CPU:
its table describes a block Cholesky factorization of the component's matrix,
round by round of independent bodies, and the components it refuses are those
whose elimination fills in too much.  A NumPy factorization that follows the
table is compared with the matrix: 1e-12 of the largest entry, some thousand
roundings of blocks conditioned to 1e3."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "adb_amd", "csrc")

SHIM = r"""
#include <cstring>
#include "world.h"
using namespace adb;
extern "C" int limit(int what) { return what == 0 ? TREE_MIN : (what == 1 ? TREE_MAX : (what == 2 ? TREE_DEG : TREE_FILL)); }
// the table of the component of n bodies with m pairs; its size, 0: refused, -1: cap too small
extern "C" int plan(int n, int m, const int* pairs, const int* bodies, int* out, int cap) {
    static TreePlan p;          // reused, as a world's is
    std::vector<int> t(3, -7);
    p.start(n);
    for (int e = 0; e < m; e++) p.edge(pairs[2 * e], pairs[2 * e + 1], 2 * e);
    if (!p.finish(n, bodies, t)) return t.size() == 3 ? 0 : -2;
    if ((int)t.size() - 3 > cap) return -1;
    memcpy(out, t.data() + 3, (t.size() - 3) * sizeof(int));
    return (int)t.size() - 3;
}
extern "C" int solve_ints(int n, int nlev, int ne) { return tree_solve_ints(n, nlev, ne); }
// capacity left behind by a pinned buffer whose growth fails; -1: it did not fail
extern "C" int pinned_after_failure(int cap0) {
    int* p = nullptr;
    size_t cap = cap0;
    try { regrow_pinned(p, cap, (size_t)1 << 50); } catch (const HipError&) { return p ? -2 : (int)cap; }
    return -1;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    src, so = str(d / "shim.hip"), str(d / "shim.so")
    with open(src, "w") as fh:
        fh.write(SHIM)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.check_call([hipcc, "--offload-host-only", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, src, "-o", so])
    return C.CDLL(so)


def plan(lib, n, pairs, bodies):
    pairs = np.ascontiguousarray(pairs, dtype=np.int32).reshape(-1, 2)
    out = np.zeros(200000, dtype=np.int32)
    ptr = C.POINTER(C.c_int)
    bodies = np.ascontiguousarray(bodies, dtype=np.int32)
    k = lib.plan(n, len(pairs), pairs.ctypes.data_as(ptr), bodies.ctypes.data_as(ptr), out.ctypes.data_as(ptr), len(out))
    assert k >= 0
    return out[:k]


def fields(lib, t):
    n, nlev, ne, nc = t[:4]
    f, at = {"n": n, "nlev": nlev, "ne": ne, "nc": nc}, 4
    for name, size in (("lev", nlev + 1), ("body", n), ("up", n + 1), ("node", ne), ("own", ne), ("low", n + 1), ("lowe", ne)):
        f[name] = t[at:at + size]
        at += size
    assert at == lib.solve_ints(int(n), int(nlev), int(ne))
    for name, size in (("src", ne), ("con", ne + 1), ("cona", nc), ("conb", nc)):
        f[name] = t[at:at + size]
        at += size
    assert at == len(t)
    return f


def path(n):
    return n, [(i, i + 1) for i in range(n - 1)]


def cycle(n):
    return n, path(n)[1] + [(0, n - 1)]


def star(n):
    return n, [(0, i) for i in range(1, n)]


def random_tree(n):
    rng = np.random.default_rng(n)
    return n, [(int(rng.integers(i)), i) for i in range(1, n)]


def wall(w, h, diagonals=True):
    at = lambda i, j: j * w + i
    e = []
    for j in range(h):
        for i in range(w):
            for di, dj in ((1, 0), (0, 1)) + (((1, 1), (-1, 1)) if diagonals else ()):
                if 0 <= i + di < w and j + dj < h:
                    e.append((at(i, j), at(i + di, j + dj)))
    return w * h, e


def clique(n):
    return n, [(i, j) for j in range(n) for i in range(j)]


PLANNED = {"path17": path(17), "path256": path(256), "cycle40": cycle(40), "star100": star(100), "tree150": random_tree(150),
           "wall3x6": wall(3, 6), "wall4x10": wall(4, 10), "grid6x6": wall(6, 6, False), "clique9": clique(9)}
# more than 8 neighbours left, or more than 6 blocks a body
REFUSED = {"clique10": clique(10), "clique17": clique(17), "wall16x16": wall(16, 16), "grid16x16": wall(16, 16, False)}


def shuffled(n, pairs):
    """The graph with its bodies renumbered, the pairs sorted (lo, hi)."""
    perm = np.random.default_rng(len(pairs)).permutation(n)
    return sorted((min(perm[a], perm[b]), max(perm[a], perm[b])) for a, b in pairs)


@pytest.mark.parametrize("name", list(PLANNED))
def test_the_table_is_a_block_factorization(lib, name):
    n, pairs = PLANNED[name]
    pairs = shuffled(n, pairs)
    bodies = 5 + 3 * np.arange(n)
    f = fields(lib, plan(lib, n, pairs, bodies))
    assert f["n"] == n and sorted(f["body"]) == list(bodies) and f["ne"] <= lib.limit(3) * n
    local = (f["body"] - 5) // 3                      # body at a position
    # matrix: a Gram matrix of the pairs and the identity, b x b blocks
    b, rng = 3, np.random.default_rng(1)
    H = np.zeros((n, b, n, b))
    for i, j in pairs:
        u, v = rng.normal(size=(2, b, 4))
        H[i, :, i] += u @ u.T; H[j, :, j] += v @ v.T
        H[i, :, j] += u @ v.T; H[j, :, i] += v @ u.T
    for i in range(n):
        H[i, :, i] += 0.1 * np.eye(b)
    D, V = [None] * n, [None] * f["ne"]
    where = {}
    for l in range(f["nlev"]):
        cols = range(f["lev"][l], f["lev"][l + 1])
        assert len(cols) > 0
        done = f["lev"][l]
        for j in cols:
            A = H[local[j], :, local[j]].copy()
            for x in f["lowe"][f["low"][j]:f["low"][j + 1]]:
                # a round's columns need blocks of earlier rounds only
                assert f["node"][x] == j and f["own"][x] < done
                A -= V[x] @ V[x].T
            D[j] = np.linalg.cholesky(A)
            for e in range(f["up"][j], f["up"][j + 1]):
                i, s = f["node"][e], f["src"][e]
                assert f["own"][e] == j and i >= f["lev"][l + 1]
                pair = (min(local[i], local[j]), max(local[i], local[j]))
                if s >= 0:
                    assert pairs[s // 2] == pair and (s % 2 == 0) == (local[i] == pair[0])
                else:
                    assert pair not in pairs
                A = H[local[i], :, local[j]].copy()
                for x in range(f["con"][e], f["con"][e + 1]):
                    p, q = f["cona"][x], f["conb"][x]
                    assert f["own"][p] == f["own"][q] < done and f["node"][p] == i and f["node"][q] == j
                    A -= V[p] @ V[q].T
                V[e] = np.linalg.solve(D[j], A.T).T
                where[i, j] = e
    L = np.zeros((n, b, n, b))
    for j in range(n):
        L[j, :, j] = D[j]
    for (i, j), e in where.items():
        L[i, :, j] = V[e]
    L = L.reshape(n * b, n * b)
    P = H[local][:, :, local].reshape(n * b, n * b)
    np.testing.assert_allclose(L @ L.T, P, rtol=0, atol=1e-12 * np.abs(P).max())


@pytest.mark.parametrize("name", list(REFUSED))
def test_components_that_fill_in_are_refused(lib, name):
    n, pairs = REFUSED[name]
    assert len(plan(lib, n, shuffled(n, pairs), np.arange(n))) == 0


def test_a_path_takes_logarithmic_rounds(lib):
    n, pairs = path(256)
    assert fields(lib, plan(lib, n, pairs, np.arange(n)))["nlev"] <= 2 * 8 + 1


def test_a_failed_pinned_growth_leaves_no_capacity(lib):
    assert lib.pinned_after_failure(100) == 0
