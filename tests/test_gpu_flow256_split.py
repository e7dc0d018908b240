"""The split-bf16 kernels of the 256-wide field (mo_flow256_step_stages,
mo_flow256_adjoint_step / _grads) at the edges of their tiles: 32-point
blocks, 64-point chunks, chunks that are not full, one workgroup and many,
and the FP32-MFMA adjoint (mo_flow256_step_save / _backward / _dw_grads /
_small_grads) on the same problem.

Bar: 2e-6 relative in norm against FP64.  A sum of 256 FP32 products has a
relative rounding error of about 256^(1/2) 2^-24 = 1e-6 against its terms'
norm; four layers forward and four back multiply a handful of such errors,
which add up as independent ones."""
import ctypes as C

import pytest
import torch

from meshode_amd import _lib
from meshode_amd import neuralode as NO
from meshode_amd import pyDeform

pytestmark = pytest.mark.gpu

STEPS = 3


def _problem(n, gpu):
    torch.manual_seed(n)
    m = NO.VelocityMLP(hidden=256, seed=11).to(gpu)
    with torch.no_grad():
        for b in m.biases:
            b.normal_(0, 0.2)
    y0 = (torch.rand(n, 3) * 1.4 - 0.2).to(gpu)
    return m, y0, torch.randn(n, 3).to(gpu)


def _reference(m, y0, w):
    m64 = NO.VelocityMLP(hidden=256, seed=11, dtype=torch.float64).to(y0.device)
    m64.load_state_dict({k: v.double() for k, v in m.state_dict().items()})
    y64 = y0.double().requires_grad_(True)
    y = y64
    for _ in range(STEPS):
        y = NO.rk4_step(m64, y, 1.0 / STEPS)
    return y.detach(), torch.autograd.grad(y, [y64, *m64.parameters()], w.double())


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 65, 257, 8193, 16500])
def test_split_flow_and_adjoint(gpu, n):
    print(f"[flow256 split] n={n}", flush=True)
    m, y0, w = _problem(n, gpu)
    y0.requires_grad_(True)
    y = NO.odeint_rk4(m, y0, steps=STEPS)
    got = torch.autograd.grad(y, [y0, *m.parameters()], w)
    want_y, want = _reference(m, y0.detach(), w)
    errs = [_rel(y.detach(), want_y)] + [_rel(a, b) for a, b in zip(got, want)]
    print("[flow256 split]  ", " ".join(f"{e:.1e}" for e in errs), flush=True)
    assert max(errs) <= 2e-6


@pytest.mark.parametrize("e", [-100, -60, 60, 90])
def test_gradient_magnitudes(gpu, e):
    """The adjoint is linear in dL/dy1: the same bar for gradients scaled by
    powers of two, as long as the three bf16 parts of what it multiplies are
    normal (2^-100 leaves ten powers for the factors that make them smaller)
    and its sums finite."""
    print(f"[flow256 split] gradients 2^{e}", flush=True)
    m, y0, w = _problem(300, gpu)
    y0.requires_grad_(True)
    got = torch.autograd.grad(NO.odeint_rk4(m, y0, steps=STEPS), [y0, *m.parameters()], w * 2.0 ** e)
    _, want = _reference(m, y0.detach(), w)
    assert max(_rel(a.double() * 2.0 ** -e, b) for a, b in zip(got, want)) <= 2e-6


@pytest.mark.parametrize("n", [33, 1000])
def test_fp32_mfma_adjoint_step(gpu, n):
    print(f"[flow256 fp32] n={n}", flush=True)
    m, y0, w = _problem(n, gpu)
    lib, P, s = _lib.load(), NO.flow256_pack(m), pyDeform._stream()
    f = lambda *shape: torch.empty(*shape, device=gpu)      # noqa: E731
    p = lambda t: C.c_void_p(t.data_ptr())                  # noqa: E731
    Hs, Xs, y1, g0, dAs, Gs = f(3, 4, n, 256), f(4, n, 3), f(n, 3), f(n, 3), f(3, 4, n, 256), f(4, n, 3)
    h = 1.0 / STEPS
    _lib.call("mo_flow256_step_save", p(y0), n, p(P), h, p(y1), p(Hs), p(Xs), s)
    _lib.call("mo_flow256_step_backward", n, p(P), h, p(Hs), p(w), p(g0), p(dAs), p(Gs), s)
    dw, work = f(2, 256, 256), f(int(lib.mo_flow256_dw_work_floats()))
    _lib.call("mo_flow256_dw_grads", n, p(dAs), p(Hs), p(dw), p(work), s)
    ns = int(lib.mo_flow256_small_grad_floats())
    small, swork = f(ns), f(256 * ns)
    _lib.call("mo_flow256_small_grads", n, p(dAs), p(Hs), p(Xs), p(Gs), p(small), p(swork), s)
    m64 = NO.VelocityMLP(hidden=256, seed=11, dtype=torch.float64).to(gpu)
    m64.load_state_dict({k: v.double() for k, v in m.state_dict().items()})
    y64 = y0.double().requires_grad_(True)
    out = NO.rk4_step(m64, y64, h)
    want = torch.autograd.grad(out, [y64, *m64.parameters()], w.double())
    got = [g0, small[:768].view(256, 3), dw[0], dw[1], small[1536:2304].view(3, 256), small[768:1024],
           small[1024:1280], small[1280:1536], small[2304:2307]]
    errs = [_rel(y1, out.detach())] + [_rel(a, b) for a, b in zip(got, want)]
    print("[flow256 fp32]  ", " ".join(f"{e:.1e}" for e in errs), flush=True)
    assert max(errs) <= 2e-6


def test_step_beyond_2_30_floats(gpu):
    """As many points as mo_flow256_step takes are taken with the stage
    inputs too: beyond 2^30 floats of them (here by one point), where every
    index into them needs 64 bits."""
    n, k = (1 << 30) // 12 + 1, 4096
    print(f"[flow256 split] n={n}", flush=True)
    m, y0, _ = _problem(k, gpu)
    y = y0.repeat(n // k + 1, 1)[:n].contiguous()
    P = NO.flow256_pack(m)
    want_z = torch.empty(4, k, 3, device=gpu)
    want = NO.flow256_step(P, y0, 1.0 / STEPS, want_z)
    got = NO.flow256_step(P, y, 1.0 / STEPS)
    z = torch.empty(4, n, 3, device=gpu)
    again = NO.flow256_step(P, y, 1.0 / STEPS, z)
    assert torch.equal(got, again)
    # a point's place in its block moves its last bits: the bar of the file
    for lo in (0, k * (n // k // 2), k * (n // k - 1)):
        assert _rel(got[lo:lo + k], want.double()) <= 2e-6
        assert _rel(z[:, lo:lo + k], want_z.double()) <= 2e-6
    tail = n - k * (n // k)
    assert _rel(got[-tail:], want[:tail].double()) <= 2e-6
    assert _rel(z[:, -tail:], want_z[:, :tail].double()) <= 2e-6
