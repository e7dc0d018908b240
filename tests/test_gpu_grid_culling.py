"""The grid build's FP32 culling and its second kernel (bricks that walk many
tiles go to k_grid_heavy) against the oracle, bit for bit: points near the
centre of a sphere, where every tile has to be walked (with whole and partial
bricks), random soups, slivers whose plane bound is unsound in FP32, needles,
coordinates far outside the unit box and far larger than FP32 resolves, and
planes through the box spanned by vertices so far away that FP64 places them
to 1e-4."""
import ctypes as C

import numpy as np
import pytest
import torch

from meshode_amd import _lib, pyDeform, synth

pytestmark = pytest.mark.gpu


def _case(name):
    r = np.random.default_rng(7)
    if name.startswith("sphere"):
        V, F = synth.icosphere(4)
        return 0.5 + 0.45 * V, F, int(name[6:])
    if name == "planes":
        c, u, w = r.uniform(0.2, 0.8, (400, 3)), r.normal(size=(400, 3)), r.normal(size=(400, 3))
        u /= np.linalg.norm(u, axis=1, keepdims=True)
        w -= (w * u).sum(1, keepdims=True) * u
        V = np.stack([c + 1e12 * u, c - 5e11 * u + 8e11 * w, c - 5e11 * u - 8e11 * w], 1).reshape(-1, 3)
        return V, np.arange(1200, dtype=np.int32).reshape(-1, 3), 11
    V, F = r.uniform(0, 1, (60, 3)), r.integers(0, 60, (500, 3)).astype(np.int32)
    if name == "slivers":
        V[::2] = V[0] + 1e-9 * r.uniform(0, 1, (30, 3))
    elif name == "needles":
        V *= [1.0, 1e-7, 1e-5]
    elif name == "far":
        V = V * 100 + 50
    elif name == "huge":
        V = V * 1e9 - 4e8
    return V, F, 11


@pytest.mark.parametrize("name", ["sphere16", "sphere13", "soup", "slivers", "needles", "far", "huge", "planes"])
def test_culling_is_exact(gpu, oracle, name):
    print(f"[grid culling] {name}", flush=True)
    V, F, N = _case(name)
    Vd = torch.from_numpy(np.ascontiguousarray(V)).to(gpu)
    Fd = torch.from_numpy(np.ascontiguousarray(F, np.int32)).to(gpu)
    d = torch.empty(N ** 3, dtype=torch.float64, device=gpu)
    t = torch.empty(N ** 3, dtype=torch.int32, device=gpu)
    _lib.call("mo_grid_build", C.c_void_p(Vd.data_ptr()), len(V), C.c_void_p(Fd.data_ptr()), len(F), N,
              C.c_void_p(d.data_ptr()), C.c_void_p(0), C.c_void_p(t.data_ptr()), pyDeform._stream())
    od, _, ot = oracle.build_grid(V, F, N)
    assert np.array_equal(d.cpu().numpy(), od.reshape(-1))
    assert np.array_equal(t.cpu().numpy(), ot.reshape(-1))
