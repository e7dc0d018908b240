"""Large pairs on teams of register/LDS workgroups (k_lm_solve_lds_halo:
spatial order, neighbours' copies in LDS).  The result must not depend on
the mesh's numbering (up to the rounding of sums), agrees with the
one-workgroup kernel on global memory, and a mesh whose halo does not fit
the LDS is still solved.  Sizes: just above one workgroup's 8192 vertices
(3 chunks), chunks with one vertex more and less than their neighbours, and
border edges (multiplicity 1 beside 2).  The oracle's exact-step LM checks
the same kernel in test_gpu_lm (12000 vertices).

Small pairs: a launch has as many waves as its largest pair needs, so a
pair's result must not depend on which pairs share the launch.
"""
import numpy as np
import pytest
import torch

from meshode_amd import deform, synth

pytestmark = pytest.mark.gpu

ENERGY_RTOL = 1e-3   # energies of the same steps on different kernels


def _pair(n, open_faces=0, seed=3):
    V, F, tV, tF = synth.box_union_pair(seed, n_boxes=5, n_verts=n // 2 * 2)
    if n % 2:                       # one vertex in no face
        V = np.concatenate([V, [[0.31, 0.2, 0.1]]])
    if open_faces:                  # border edges: multiplicity 1 beside 2
        F = F[open_faces:]
    return V, F, tV, tF


@pytest.mark.parametrize("mesh", ["ico5", "boxes8194", "boxes12289"])
def test_halo_team_any_numbering(gpu, mesh):
    print(f"[lm halo] {mesh}", flush=True)
    V, F, tV, tF = (synth.displaced_sphere_pair(4, src_level=5, tgt_level=4) if mesh == "ico5"
                    else _pair(int(mesh[5:]), open_faces=3))
    perm = np.random.default_rng(1).permutation(len(V))
    inv = np.argsort(perm)
    # few steps: later ones of a box pair's non-smooth problem part ways over
    # the last bits of the FP32 neighbour sums, whichever kernel runs
    opt = deform.default_options(max_num_iterations=3)
    out, st = deform.rigid_deform_batch([(V, F, tV, tF), (V[perm], inv[F].astype(np.int32), tV, tF)],
                                        grid_resolution=32, options=opt)
    assert all(s["solver_path_name"] == "lds_team" for s in st)
    assert abs(st[0]["initial_cost"] - st[1]["initial_cost"]) <= 1e-9 * st[0]["initial_cost"]
    assert abs(st[0]["final_cost"] - st[1]["final_cost"]) <= ENERGY_RTOL * st[0]["final_cost"]
    # one workgroup on global memory solves the same problem
    _, one = deform.rigid_deform_batch([(V, F, tV, tF)], grid_resolution=32,
                                       options=deform.default_options(max_num_iterations=3, kernel_variant=1))
    assert abs(st[0]["final_cost"] - one[0]["final_cost"]) <= ENERGY_RTOL * one[0]["final_cost"]


@pytest.mark.parametrize("side,workgroups", [(443, 64), (444, 49), (512, 64)])
def test_halo_team_largest(gpu, side, workgroups):
    """Sheets of side^2 vertices on either side of 64 workgroups of 3072
    (196608), where the chunks grow to 4096, and the largest that 64 of those
    hold (262144), against the one-workgroup kernel."""
    print(f"[lm halo] {side} x {side}", flush=True)
    i, j = np.meshgrid(np.arange(side), np.arange(side), indexing="ij")
    V = np.stack([i / side, j / side, 0.1 * np.sin(9.0 * i / side + 5.0 * j / side)], -1).reshape(-1, 3)
    k = (i * side + j)[:-1, :-1].reshape(-1)
    F = np.concatenate([np.stack([k, k + side, k + 1], 1), np.stack([k + 1, k + side, k + side + 1], 1)]).astype(np.int32)
    _, _, tV, tF = _pair(1000)
    lo, hi = tV.min(0), tV.max(0)
    pair = (lo + (hi - lo) * V * [1.0, 1.0, 0.5] + (hi - lo) * [0.0, 0.0, 0.4], F, tV, tF)
    opt = dict(max_num_iterations=1, pcg_max_iterations=30)
    _, st = deform.rigid_deform_batch([pair], grid_resolution=32, options=deform.default_options(**opt))
    _, one = deform.rigid_deform_batch([pair], grid_resolution=32, options=deform.default_options(kernel_variant=1, **opt))
    assert st[0]["solver_path_name"] == "lds_team" and st[0]["workgroups"] == workgroups
    assert one[0]["solver_path_name"] == "one_workgroup"
    print(f"[lm halo]   {st[0]['final_cost']:.9e} / {one[0]['final_cost']:.9e}", flush=True)
    # the same FP32 positions and residuals, summed in FP64
    assert abs(st[0]["initial_cost"] - one[0]["initial_cost"]) <= 1e-6 * one[0]["initial_cost"]
    # one step cut off after 30 PCG iterations: 4e-6 apart on every size (the
    # register/LDS kernels take hardware reciprocals in the LM diagonal, 1e-7
    # each, which an unconverged step carries on)
    assert abs(st[0]["final_cost"] - one[0]["final_cost"]) <= 1e-4 * one[0]["final_cost"]


def test_halo_too_long_for_the_lds(gpu):
    """Random triangles: nearly every neighbour is in another chunk, so the
    pair stays on the kernel that reads such neighbours where they are."""
    print("[lm halo] random triangles", flush=True)
    rng = np.random.default_rng(5)
    n = 30000
    V, _, tV, tF = _pair(1000)
    V = rng.random((n, 3)) * (V.max(0) - V.min(0)) + V.min(0)
    F = rng.permutation(np.repeat(np.arange(n, dtype=np.int32), 2)).reshape(-1, 3)
    F = F[(F[:, 0] != F[:, 1]) & (F[:, 1] != F[:, 2]) & (F[:, 2] != F[:, 0])]
    opt = dict(max_num_iterations=3)
    _, st = deform.rigid_deform_batch([(V, F, tV, tF)], grid_resolution=32, options=deform.default_options(**opt))
    _, one = deform.rigid_deform_batch([(V, F, tV, tF)], grid_resolution=32,
                                       options=deform.default_options(kernel_variant=1, **opt))
    assert st[0]["solver_path_name"] == "lds_team"
    assert abs(st[0]["final_cost"] - one[0]["final_cost"]) <= ENERGY_RTOL * one[0]["final_cost"]


def test_planned_pairs_do_not_depend_on_the_batch(gpu):
    """Which pairs get a spatial order is decided by their own counts: pairs
    around what one workgroup's LDS holds (5700 vertices of a closed mesh),
    and one of unshared edges whose adjacency is twice what its counts
    suggest, alone and beside pairs that are planned."""
    print("[lm halo] batches", flush=True)
    rng = np.random.default_rng(8)
    V, F, tV, tF = _pair(5000)
    soup = rng.permutation(np.arange(5000 * 5, dtype=np.int32) % 5000)[:24000].reshape(-1, 3)
    soup = soup[(soup[:, 0] != soup[:, 1]) & (soup[:, 1] != soup[:, 2]) & (soup[:, 2] != soup[:, 0])]
    pairs = [_pair(n, seed=n) for n in (3072, 5600, 5800, 8190, 8194)] + [(V, soup, tV, tF)]
    opt = deform.default_options(max_num_iterations=3)
    out, st = deform.rigid_deform_batch(pairs, grid_resolution=32, options=opt)
    assert [s["solver_path_name"] for s in st] == ["lds", "lds", "lds_team", "lds_team", "lds_team", "lds_team"]
    for k, p in enumerate(pairs):
        alone, sa = deform.rigid_deform_batch([p], grid_resolution=32, options=opt)
        assert torch.equal(alone[0], out[k]) and sa[0]["solver_path_name"] == st[k]["solver_path_name"], k
    # the soup against the one-workgroup kernel
    _, one = deform.rigid_deform_batch([pairs[-1]], grid_resolution=32,
                                       options=deform.default_options(kernel_variant=1, max_num_iterations=3))
    assert abs(st[-1]["final_cost"] - one[0]["final_cost"]) <= ENERGY_RTOL * one[0]["final_cost"]


@pytest.mark.parametrize("n", [200, 258, 514, 602, 770])
def test_more_small_pairs_than_workgroups(gpu, n):
    """600 pairs of 4, 5, 9, 10 and 13 waves: more than the chip holds of the
    wider ones, so workgroups take further pairs; each pair as alone."""
    print(f"[lm small] 600 pairs of {n}", flush=True)
    pairs = [_pair(n, seed=3 + k) for k in range(4)]
    opt = deform.default_options(max_num_iterations=3)
    out, st = deform.rigid_deform_batch([pairs[k % 4] for k in range(600)], grid_resolution=16, options=opt)
    for k in range(4):
        alone, _ = deform.rigid_deform_batch([pairs[k]], grid_resolution=16, options=opt)
        assert all(torch.equal(alone[0], out[j]) for j in range(k, 600, 4))


def test_small_pairs_any_launch_width(gpu):
    """1 to 16 waves per workgroup and both sides of a wave's 64 vertices;
    an open mesh (mixed multiplicities, odd lists) among them."""
    print("[lm small] launch widths", flush=True)
    pairs = [_pair(n, k % 2 * 5, seed=3 + k) for k, n in enumerate((126, 128, 130, 640, 642, 1022, 1024, 2048))]
    opt = deform.default_options(max_num_iterations=10)
    out, st = deform.rigid_deform_batch(pairs, grid_resolution=32, options=opt)
    for k, p in enumerate(pairs):
        alone, sa = deform.rigid_deform_batch([p], grid_resolution=32, options=opt)
        assert torch.equal(alone[0], out[k]), k
        assert sa[0]["final_cost"] == st[k]["final_cost"] and sa[0]["pcg_iterations"] == st[k]["pcg_iterations"]
