"""The on-chip DeformWithRot solver (k_lm_rot_chip) at the edges of its
chunks: one vertex below, at and above a 256-vertex chunk, a last chunk that
is short, a last chunk of one vertex, merged parallel half-edges beyond an
entry's multiplicity, vertices in no face, and a hub whose adjacency does not
fit the LDS (which takes the one-workgroup kernel).  The bar is the one of
the other DeformWithRot tests: the final energy, evaluated by the oracle's
cost at the GPU's result, within 1e-3 of the oracle's exact-step solve."""
import numpy as np
import pytest
import torch

from meshode_amd import deform, pyDeform, synth

pytestmark = pytest.mark.gpu


def _fan(n):
    """A hub joined to a rim of n vertices."""
    a = 2 * np.pi * np.arange(n) / n
    V = np.concatenate([[[0.0, 0.0, 0.3]], np.stack([np.cos(a), np.sin(a), 0 * a], 1)])
    k = np.arange(n)
    return V, np.stack([0 * k, 1 + k, 1 + (k + 1) % n], 1).astype(np.int32)


def _case(name):
    if name.startswith("boxes"):
        sV, sF, tV, tF = synth.box_union_pair(3, n_boxes=3, n_verts=int(name[5:]) // 2 * 2)
        if int(name[5:]) % 2:        # a vertex in no face
            sV = np.concatenate([sV, sV.mean(0, keepdims=True)])
        return sV, sF, tV, tF
    _, _, tV, tF = synth.displaced_sphere_pair(5, src_level=1, tgt_level=2)
    if name == "repeated":           # 70 copies of every half-edge: two entries per neighbour
        sV, sF = synth.icosphere(1)
        return sV * 0.9, np.tile(sF, (70, 1)), tV, tF
    sV, sF = _fan(int(name[3:]))
    return sV, sF, tV, tF


@pytest.mark.parametrize("name,workgroups", [("boxes254", 1), ("boxes256", 1), ("boxes257", 2), ("boxes512", 2),
                                             ("boxes600", 3), ("repeated", 1), ("fan300", 2)])
def test_chip_energy_parity(gpu, oracle, name, workgroups):
    print(f"[rot chip] {name}", flush=True)
    sV, sF, tV, tF = _case(name)
    pid = deform.template_f64(tV, tF, 16)
    _, scale, trans = pyDeform.TemplateInfo(pid)
    grid = pyDeform.TemplateGrid(pid)[0].cpu().numpy().reshape(-1)
    sn = (sV - trans) / scale
    V = torch.from_numpy(sn).to(gpu).contiguous()
    st, W = deform.deform_rot(pid, V, sF, 1.0)
    assert st["workgroups"] == workgroups
    _, _, so = oracle.lm_rot_solve(grid, 16, sn, sF, 1.0)
    eg = oracle.lm_rot_cost(grid, 16, V.cpu().numpy(), W.cpu().numpy(), sn, sF, 1.0)[0]
    print(f"[rot chip]   gpu {eg:.6e} oracle {so['final_cost']:.6e} ({st['iterations']}/{so['iterations']} it)",
          flush=True)
    assert st["initial_cost"] == pytest.approx(so["initial_cost"], rel=1e-4)
    assert abs(eg - so["final_cost"]) <= 1e-3 * so["final_cost"]


@pytest.mark.parametrize("n,team_vertices,workgroups", [(65, 1, 33), (130, 2, 44), (1000, 15, 63), (1000, 16, 63),
                                                        (64, 1, 64), (128, 2, 64), (129, 2, 43)])
def test_no_empty_chunk(gpu, oracle, n, team_vertices, workgroups):
    """team_vertices asking for more chunks than a team has workgroups: chunks
    of ceil(n / 64) vertices, and as many as the vertices fill."""
    print(f"[rot chip] {n} vertices, team_vertices {team_vertices}", flush=True)
    sV, sF = _fan(n - 1)
    _, _, tV, tF = synth.displaced_sphere_pair(5, src_level=1, tgt_level=2)
    pid = deform.template_f64(tV, tF, 16)
    _, scale, trans = pyDeform.TemplateInfo(pid)
    grid = pyDeform.TemplateGrid(pid)[0].cpu().numpy().reshape(-1)
    sn = (sV - trans) / scale
    V = torch.from_numpy(sn).to(gpu).contiguous()
    opt = deform.default_options(pcg_relative_tolerance=1e-6, team_vertices=team_vertices)
    st, W = deform.deform_rot(pid, V, sF, 1.0, options=opt)
    assert st["workgroups"] == workgroups
    eg = oracle.lm_rot_cost(grid, 16, V.cpu().numpy(), W.cpu().numpy(), sn, sF, 1.0)[0]
    assert st["final_cost"] == pytest.approx(eg, rel=1e-3)
    one = torch.from_numpy(sn).to(gpu).contiguous()
    s1, _ = deform.deform_rot(pid, one, sF, 1.0)
    assert st["final_cost"] == pytest.approx(s1["final_cost"], rel=1e-3)


def test_hub_beyond_lds(gpu):
    """A hub of 6000 neighbours does not fit a chunk's LDS: one workgroup."""
    print("[rot chip] fan6000", flush=True)
    sV, sF, tV, tF = _case("fan6000")
    pid = deform.template_f64(tV, tF, 16)
    _, scale, trans = pyDeform.TemplateInfo(pid)
    V = torch.from_numpy((sV - trans) / scale).to(gpu).contiguous()
    opt = deform.default_options(max_num_iterations=2, pcg_max_iterations=20)
    st, _ = deform.deform_rot(pid, V, sF, 1.0, options=opt)
    assert st["workgroups"] == 1 and st["final_cost"] <= st["initial_cost"]


def test_refused_after_the_first_launch(gpu, monkeypatch):
    """A batch that fills the chip twice over takes several cooperative
    launches.  When the runtime refuses a later one, its problems go to one
    workgroup each and the earlier ones keep their results.  Each launch is
    as many problems as are co-resident, so the refused ones are the last of
    the order of sizes; 1100 problems of 2 workgroups are more than fit on
    256 CUs at 4 workgroups each."""
    print("[rot chip] second launch refused", flush=True)
    sV, sF, tV, tF = _case("boxes258")
    pid = deform.template_f64(tV, tF, 16)
    _, scale, trans = pyDeform.TemplateInfo(pid)
    sn = torch.from_numpy((sV - trans) / scale).to(gpu).contiguous()
    Fd = torch.from_numpy(sF).to(gpu)
    opt = deform.default_options(max_num_iterations=2, pcg_max_iterations=10, pcg_relative_tolerance=1e-6)
    n = 1100

    def solve():
        Vs = [sn.clone() for _ in range(n)]
        st, W = deform.deform_rot_batch([pid] * n, Vs, [Fd] * n, [1.0] * n, options=opt)
        return st, Vs

    want_st, want = solve()
    assert all(s["solver_path_name"] == "team" for s in want_st)
    monkeypatch.setenv("MO_LM_COOP_REFUSE", "2")
    st, got = solve()
    monkeypatch.delenv("MO_LM_COOP_REFUSE")
    ran = [s["solver_path_name"] == "team" for s in st]
    k = sum(ran)
    assert 0 < k < n and all(ran[:k])
    assert all(s["solver_path_name"] == "one_workgroup_coop_refused" and s["workgroups"] == 1 for s in st[k:])
    assert all(torch.equal(a, b) for a, b in zip(got[:k], want[:k]))
    for s in st[k:]:
        assert s["final_cost"] == pytest.approx(want_st[0]["final_cost"], rel=1e-6)


TEAM = dict(pcg_relative_tolerance=1e-6, team_vertices=16, block_threads=64)


@pytest.mark.parametrize("name", ["boxes254", "boxes600", "repeated", "fan300"])
def test_one_workgroup_energy_parity(gpu, oracle, monkeypatch, name):
    """The kernel a refused cooperative launch leaves its problems to."""
    print(f"[rot one workgroup] {name}", flush=True)
    sV, sF, tV, tF = _case(name)
    pid = deform.template_f64(tV, tF, 16)
    _, scale, trans = pyDeform.TemplateInfo(pid)
    grid = pyDeform.TemplateGrid(pid)[0].cpu().numpy().reshape(-1)
    sn = (sV - trans) / scale
    V = torch.from_numpy(sn).to(gpu).contiguous()
    monkeypatch.setenv("MO_LM_COOP_REFUSE", "1")
    st, W = deform.deform_rot(pid, V, sF, 1.0, options=deform.default_options(**TEAM))
    monkeypatch.delenv("MO_LM_COOP_REFUSE")
    assert st["solver_path_name"] == "one_workgroup_coop_refused" and st["workgroups"] == 1
    _, _, so = oracle.lm_rot_solve(grid, 16, sn, sF, 1.0)
    eg = oracle.lm_rot_cost(grid, 16, V.cpu().numpy(), W.cpu().numpy(), sn, sF, 1.0)[0]
    assert st["initial_cost"] == pytest.approx(so["initial_cost"], rel=1e-4)
    assert abs(eg - so["final_cost"]) <= 1e-3 * so["final_cost"]


def _sheet(a, b, shuffle=False):
    """A wavy sheet of a x b vertices, numbered by rows or at random."""
    i, j = np.meshgrid(np.arange(a), np.arange(b), indexing="ij")
    V = np.stack([0.1 + 0.8 * i / a, 0.1 + 0.8 * j / b, 0.5 + 0.1 * np.sin(9.0 * i / a + 5.0 * j / b)], -1).reshape(-1, 3)
    k = (i * b + j)[:-1, :-1].reshape(-1)
    F = np.concatenate([np.stack([k, k + b, k + 1], 1), np.stack([k + 1, k + b, k + b + 1], 1)]).astype(np.int32)
    if shuffle:
        perm = np.random.default_rng(2).permutation(len(V))
        V, F = V[perm], np.argsort(perm)[F].astype(np.int32)
    return V, F


@pytest.mark.parametrize("name,team_vertices,workgroups,solver", [
    ("rows16500", 0, 33, "team"),                 # 512 vertices per workgroup, on chip
    ("rows33024", 0, 1, "one_workgroup"),         # more than 64 workgroups of 512
    ("rows33024", 2048, 17, "team"),              # the same on a team in global memory
    ("random16900", 0, 1, "one_workgroup"),       # neighbours everywhere: no chunk fits
    ("random16900", 512, 32, "team"),             # (34 workgroups asked for, 32 given)
    ("fan6000", 512, 12, "team"),
])
def test_large_problems(gpu, monkeypatch, name, team_vertices, workgroups, solver):
    """A few steps on every kernel a large problem can take, against the same
    steps on one workgroup in global memory."""
    print(f"[rot large] {name} team_vertices={team_vertices}", flush=True)
    sV, sF = {"rows16500": lambda: _sheet(165, 100), "rows33024": lambda: _sheet(258, 128),
              "random16900": lambda: _sheet(130, 130, True), "fan6000": lambda: _fan(6000)}[name]()
    _, _, tV, tF = synth.displaced_sphere_pair(5, src_level=1, tgt_level=2)
    pid = deform.template_f64(tV, tF, 16)
    _, scale, trans = pyDeform.TemplateInfo(pid)
    lo, hi = tV.min(0), tV.max(0)
    sn = torch.from_numpy((lo + (hi - lo) * sV - trans) / scale).to(gpu).contiguous()
    steps = dict(max_num_iterations=2, pcg_max_iterations=15, pcg_relative_tolerance=1e-6, block_threads=256)
    V = sn.clone()
    st, _ = deform.deform_rot(pid, V, sF, 1.0, options=deform.default_options(team_vertices=team_vertices, **steps))
    assert st["workgroups"] == workgroups and st["solver_path_name"] == solver
    one = sn.clone()
    monkeypatch.setenv("MO_LM_COOP_REFUSE", "1")
    ref, _ = deform.deform_rot(pid, one, sF, 1.0, options=deform.default_options(team_vertices=256, **steps))
    monkeypatch.delenv("MO_LM_COOP_REFUSE")
    assert ref["solver_path_name"] == "one_workgroup_coop_refused"
    print(f"[rot large]   {st['final_cost']:.9e} / {ref['final_cost']:.9e} ({st['pcg_iterations']} pcg)", flush=True)
    assert st["initial_cost"] == pytest.approx(ref["initial_cost"], rel=1e-6)
    assert st["final_cost"] == pytest.approx(ref["final_cost"], rel=1e-6)
    assert st["final_cost"] < st["initial_cost"]
    assert st["iterations"] == ref["iterations"] and st["pcg_iterations"] == ref["pcg_iterations"]
