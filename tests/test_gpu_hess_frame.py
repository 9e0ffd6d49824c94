"""The batched contact Hessians (five-coordinate frame, mollified pairs in
their own kernel) at the sizes where their launch can go wrong: one contact,
one below, at and above a 64-lane workgroup, and above one workgroup's scan of
the mollified kernel; every distance type; inputs that start at an odd double.
Against the oracle, 1e-9 of the largest entry: both sides project with
iterations that stop at off-diagonal entries of 1e-12, and log() differs from
the host's by rounding.  Gradients: 1e-10 of the largest entry, and what a
rounding of the points (coordinates up to 2) changes through the unprojected
Hessian, which is all there is on exactly parallel edges, whose mollified
gradient is zero."""
import numpy as np
import pytest

import oracle_lib as O
from adb_amd import abdtk
from adb_amd.capi import kernel_config

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DHAT = 1e-2


def contacts(kind, n, seed):
    """n configurations closer than sqrt(DHAT); a third of the edge pairs
    within 0.03 of parallel, some of them exactly parallel."""
    rng = np.random.default_rng(seed)
    X, T, D = [], [], []
    while len(X) < n:
        P = rng.uniform(-0.5, 0.5, (4, 3))
        if kind == "pt":
            w = rng.uniform(-0.3, 1.0, 3)
            P[0] = (w[:, None] * P[1:]).sum(0) / w.sum() + rng.uniform(-0.05, 0.05, 3)
            t, d = O.pt_distance(P.reshape(-1))
        else:
            u = P[1] - P[0]
            r = rng.random()
            if r < 0.33:
                v = u * rng.uniform(0.5, 1.5) + (rng.uniform(-0.02, 0.02, 3) if r < 0.28 else 0.0)
            else:
                v = rng.uniform(-1, 1, 3)
            P[2] = P[0] + rng.uniform(-0.2, 1.2) * u - rng.uniform(-0.2, 1.2) * v + rng.uniform(-0.05, 0.05, 3)
            P[3] = P[2] + v
            t, d = O.ee_distance(P.reshape(-1))
        if 1e-7 < d < DHAT:
            X.append(P.reshape(-1)); T.append(t); D.append(d)
    return np.array(X), np.array(T, dtype=np.int32), np.array(D)


def on_gpu(a, odd):
    """The array on the GPU, at a 16-byte boundary or 8 bytes past one."""
    t = torch.tensor(a, device="cuda")
    if not odd:
        return t
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
    view = buf[1:].view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize("kind", ["pt", "ee"])
@pytest.mark.parametrize("n,psd,odd", [(1, 1, False), (63, 1, True), (64, 0, False), (65, 1, False), (1025, 1, True),
                                       (1100, 0, True)])
def test_hess_sizes_and_types(kind, n, psd, odd):
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    X, T, D = contacts(kind, n, 100 + n + psd)
    if n > 1000:
        assert len(set(T.tolist())) == (7 if kind == "pt" else 9)
    old = abdtk.config
    abdtk.config = cfg = kernel_config(d_hat=DHAT, kappa=1e-3, eps_x=1e-3, psd=psd)
    try:
        f = abdtk.ipc_hess_pt_12x12_batched if kind == "pt" else abdtk.ipc_hess_ee_12x12_batched
        got = [x.cpu().numpy() for x in f(on_gpu(X, odd), torch.tensor(T, device="cuda"), on_gpu(D, odd))]
    finally:
        abdtk.config = old
    mollified = 0
    raw = kernel_config(d_hat=DHAT, kappa=1e-3, eps_x=1e-3, psd=0)
    oracle = O.ipc_hess_pt if kind == "pt" else O.ipc_hess_ee
    for i in range(n):
        ref = oracle(cfg, X[i], int(T[i]), D[i])
        moved = 12 * 2 * 2.3e-16 * np.abs(oracle(raw, X[i], int(T[i]), D[i])[0]).max()
        np.testing.assert_allclose(got[0][i], ref[0], rtol=0, atol=1e-9 * np.abs(ref[0]).max())
        np.testing.assert_allclose(got[1][i], ref[1], rtol=0, atol=1e-10 * np.abs(ref[1]).max() + moved)
        if kind == "ee":
            assert got[2][i] == pytest.approx(ref[2], rel=1e-13, abs=1e-15)
            mollified += ref[2] < 1.0
    assert kind == "pt" or n < 60 or mollified > n // 20


def test_hess_inactive_contacts_are_zero():
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    X, T, _ = contacts("ee", 130, 5)
    f = abdtk.ipc_hess_ee_12x12_batched
    d = torch.full((130,), 2.0 * abdtk.config.d_hat, dtype=torch.float64, device="cuda")
    H, g, m = f(torch.tensor(X, device="cuda"), torch.tensor(T, device="cuda"), d)
    assert float(H.abs().max()) == 0.0 and float(g.abs().max()) == 0.0 and float(m.min()) >= 0.0
