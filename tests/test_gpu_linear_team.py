"""LinearEstimation and LinearEstimationWithRot at the sizes where the CG
solver changes its shape: one row per thread and several on one workgroup
(1024 rows), the smallest team (4096 rows), the largest with one row per
thread and the first with two (32768 rows).

Reference: the same system in FP64 on the CPU, solved by scipy's sparse LU
and refined once; bar 1e-10 relative (the solver stops at 1e-13 of the
right-hand side; the box meshes' systems are conditioned below 1e3)."""
import numpy as np
import pytest
import torch

from meshode_amd import cad, synth

pytestmark = pytest.mark.gpu


def _mesh(n):
    """A tessellated box union of n vertices (odd n: one vertex in no face)."""
    V, F, _, _ = synth.box_union_pair(2, n_boxes=6, n_verts=n // 2 * 2)
    if n % 2:
        V = np.concatenate([V, [[0.3, 0.2, 0.1]]])
    return V, F


def _solve(V, F, diag, w, B):
    import scipy.sparse as sp
    import scipy.sparse.linalg as sl
    n = len(V)
    a, b = np.concatenate([F[:, 0], F[:, 1], F[:, 2]]), np.concatenate([F[:, 1], F[:, 2], F[:, 0]])
    we = w(np.linalg.norm(V[a] - V[b], axis=1))
    W = sp.coo_matrix((np.concatenate([we, we]), (np.concatenate([a, b]), np.concatenate([b, a]))), (n, n)).tocsr()
    A = (sp.diags(np.asarray(W.sum(1)).reshape(-1) + diag) - W).tocsc()
    lu = sl.splu(A)
    x = lu.solve(B)
    return x + lu.solve(B - A @ x)


@pytest.mark.parametrize("n", [1022, 1024, 1025, 4094, 4097, 32768, 32771])
def test_linear_estimation_sizes(gpu, n):
    print(f"[linear team] {n}", flush=True)
    V, F = _mesh(n)
    n = len(V)
    rng = np.random.default_rng(n)
    GV = V + 0.05 * rng.normal(size=V.shape)
    # one graph vertex per vertex: every cluster has one member
    w = lambda d: (2.0 * 2e-2 / (d + 1e-8)) ** 2                       # noqa: E731
    a, b = np.concatenate([F[:, 0], F[:, 1], F[:, 2]]), np.concatenate([F[:, 1], F[:, 2], F[:, 0]])
    r = w(np.linalg.norm(V[a] - V[b], axis=1))[:, None] * (V[a] - V[b])
    B = (1.0 + 1e-6) * GV
    np.add.at(B, a, r)
    np.add.at(B, b, -r)
    want = _solve(V, F, 1.0 + 1e-6, w, B)
    x = torch.from_numpy(V.copy()).to(gpu)
    it = cad.linear_estimation(x, torch.from_numpy(F).to(gpu), torch.zeros(0, 2, dtype=torch.int32, device=gpu),
                               torch.arange(n, dtype=torch.int32, device=gpu), torch.from_numpy(GV).to(gpu), 2.0)
    err = np.linalg.norm(x.cpu().numpy() - want) / np.linalg.norm(want)
    print(f"[linear team]   {it} iterations, {err:.1e}", flush=True)
    assert err <= 1e-10


@pytest.mark.parametrize("n", [1024, 1025, 4097, 32771])
def test_linear_estimation_rot_rigid_motion(gpu, n):
    """A rotated and translated copy is its own solution (the frames are the
    rotation, up to the 1e-8 in the scale's denominator)."""
    print(f"[linear rot team] {n}", flush=True)
    V, F = _mesh(n)
    c, s = np.cos(0.4), np.sin(0.4)
    TV = V @ np.array([[c, -s, 0], [s, c, 0], [0, 0, 1]]).T + [0.1, -0.2, 0.3]
    x = torch.from_numpy(V.copy()).to(gpu)
    cad.linear_estimation_rot(x, torch.from_numpy(F).to(gpu), torch.from_numpy(TV).to(gpu), 1.0)
    # scale = s / (s + 1e-8) with s > 1e-2, the sum of a vertex's edge lengths
    assert np.abs(x.cpu().numpy() - TV).max() <= 1e-5


@pytest.mark.parametrize("spokes", [31, 32, 33, 100])
def test_linear_estimation_merged_edges(gpu, spokes):
    """A fan around vertex 0 (its edges past a short insertion sort), in both
    orders of the faces' corners, some faces repeated: the parallel edges'
    weights add up, and vertices in no face stay alone."""
    print(f"[linear merge] {spokes}", flush=True)
    rng = np.random.default_rng(spokes)
    n = spokes + 3
    V = rng.random((n, 3))
    order = rng.permutation(spokes) + 1
    F = np.array([[0, order[i], order[(i + 1) % spokes]] for i in range(spokes)])
    F[::2] = F[::2, ::-1]
    F = np.concatenate([F, F[3:9, [1, 2, 0]], F[5:6]]).astype(np.int32)
    w = lambda d: (2.0 * 2e-2 / (d + 1e-8)) ** 2                       # noqa: E731
    GV = V + 0.05 * rng.normal(size=V.shape)
    a, b = np.concatenate([F[:, 0], F[:, 1], F[:, 2]]), np.concatenate([F[:, 1], F[:, 2], F[:, 0]])
    r = w(np.linalg.norm(V[a] - V[b], axis=1))[:, None] * (V[a] - V[b])
    B = (1.0 + 1e-6) * GV
    np.add.at(B, a, r)
    np.add.at(B, b, -r)
    W = np.zeros((n, n))
    np.add.at(W, (a, b), w(np.linalg.norm(V[a] - V[b], axis=1)))
    W += W.T
    want = np.linalg.solve(np.diag(W.sum(1) + 1.0 + 1e-6) - W, B)
    x = torch.from_numpy(V.copy()).to(gpu)
    cad.linear_estimation(x, torch.from_numpy(F).to(gpu), torch.zeros(0, 2, dtype=torch.int32, device=gpu),
                          torch.arange(n, dtype=torch.int32, device=gpu), torch.from_numpy(GV).to(gpu), 2.0)
    assert np.linalg.norm(x.cpu().numpy() - want) <= 1e-10 * np.linalg.norm(want)
