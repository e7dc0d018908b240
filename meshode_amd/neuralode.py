"""NeuralODE deformation (the reference's neuralode_fast.py:7-64 and
cad_neural_deform2.py:40-108, in the configuration of the config-3 workload).

* ``VelocityMLP``: autonomous velocity field v(y) = MLP(y - 0.5),
  3 -> 256 -> 256 -> 256 -> 3 with softplus, Xavier-uniform weights from a
  seed, zero biases.  The reference centres its input the same way
  (neuralode_fast.py:28-32; it also feeds t, which this field does not use).
  As a module its 256x256 layers are FP32 GEMMs (hipBLASLt, on the MFMA
  units).
* ``odeint_rk4``: fixed-grid RK4 over t in [0, 1] with ``steps`` equal steps
  using the 3/8-rule step that torchdiffeq's ``method="rk4"`` applies
  (the reference calls ``odeint(..., method="rk4")``, neuralode_fast.py:55-60):
      k1 = f(y); k2 = f(y + h k1/3); k3 = f(y + h (k2 - k1/3));
      k4 = f(y + h (k1 - k2 + k3)); y' = y + h (k1 + 3 k2 + 3 k3 + k4) / 8.
* On the GPU, with a 256-wide field in FP32, each forward step of
  ``odeint_rk4`` is one fused HIP kernel (``mo_flow256_step_stages``: the
  four stages, the 256 x 256 products on bf16 MFMA with FP32 operands split
  in three, softplus in their epilogue); the parameters are packed once per
  call (``mo_flow256_pack``).  Where a gradient may be asked for, a step also
  writes its four stage inputs; the adjoint (``mo_flow256_adjoint_step``)
  recomputes a step's activations from them on chip while it goes back
  through its stages, and adds the parameter gradients to partial sums that
  ``mo_flow256_adjoint_grads`` adds up once.
* ``RK4Adjoint``: the gradient of the discretized flow (discrete adjoint).
  The forward keeps the state at each step boundary (the fused one the four
  stage inputs, 48 B a point and step); the backward recomputes one step at a
  time from them and back-propagates through its four stages, so memory is
  one step's activations instead of all ``4 * steps`` evaluations.
* ``DistanceRigidityLoss``: 1/2 sum d(y)^2 over all pushed points (the
  pyDeform distance kernels) + 1/2 rho^2 sum ||(y_b - y_a) - (y0_b - y0_a)||^2
  over the source mesh edges (the graph-edge kernels).
"""
from __future__ import annotations

import math

import torch
from torch import nn
from torch.autograd import Function

from . import pyDeform


class VelocityMLP(nn.Module):
    def __init__(self, hidden=256, seed=0, dtype=torch.float32):
        super().__init__()
        g = torch.Generator().manual_seed(seed)
        dims = [3, hidden, hidden, hidden, 3]
        self.weights = nn.ParameterList()
        self.biases = nn.ParameterList()
        for a, b in zip(dims[:-1], dims[1:]):
            bound = math.sqrt(6.0 / (a + b))
            self.weights.append(nn.Parameter((torch.rand(b, a, generator=g, dtype=torch.float64) * 2 - 1)
                                             .mul_(bound).to(dtype)))
            self.biases.append(nn.Parameter(torch.zeros(b, dtype=dtype)))

    def forward(self, y):
        h = y - 0.5
        n = len(self.weights)
        for i, (W, b) in enumerate(zip(self.weights, self.biases)):
            h = torch.addmm(b, h, W.t())
            if i < n - 1:
                h = nn.functional.softplus(h)
        return h


def rk4_step(f, y, h):
    """One 3/8-rule RK4 step (torchdiffeq's ``rk4`` fixed-grid step)."""
    k1 = f(y)
    k2 = f(y + h * k1 / 3.0)
    k3 = f(y + h * (k2 - k1 / 3.0))
    k4 = f(y + h * (k1 - k2 + k3))
    return y + h * (k1 + 3.0 * (k2 + k3) + k4) * 0.125


def _fused_field(func, y):
    """True when the fused MFMA step applies: a 256-wide FP32 VelocityMLP on
    the GPU."""
    return (y.is_cuda and y.dtype == torch.float32 and isinstance(func, VelocityMLP) and len(func.weights) == 4
            and tuple(func.weights[1].shape) == (256, 256) and func.weights[0].shape[1] == 3)


def flow256_pack(func):
    """The field's parameters in the fused step's packed layout (device)."""
    import ctypes as C
    from . import _lib
    ts = [t.detach().contiguous() for pair in zip(func.weights, func.biases) for t in pair]
    out = torch.empty(int(_lib.load().mo_flow256_packed_floats()), dtype=torch.float32, device=ts[0].device)
    _lib.call("mo_flow256_pack", *[C.c_void_p(t.data_ptr()) for t in ts], C.c_void_p(out.data_ptr()),
              pyDeform._stream())
    return out


def flow256_step(packed, y, h, stages=None):
    """One fused RK4 step (FP32, GPU) of the packed 256-wide field; stages:
    a [4, n, 3] tensor that receives the stage inputs."""
    import ctypes as C
    from . import _lib
    y = y.contiguous()
    y1 = torch.empty_like(y)
    _lib.call("mo_flow256_step_stages", C.c_void_p(y.data_ptr()), y.shape[0], C.c_void_p(packed.data_ptr()), float(h),
              C.c_void_p(y1.data_ptr()), C.c_void_p(stages.data_ptr() if stages is not None else 0),
              pyDeform._stream())
    return y1


class RK4Adjoint(Function):
    """y1 = Phi(y0; theta) for ``steps`` RK4 steps; backward by recomputation
    from what each step keeps."""

    @staticmethod
    def forward(ctx, y0, steps, func, *params):
        return RK4Adjoint._integrate(ctx, y0, steps, func, any(ctx.needs_input_grad))

    @staticmethod
    def _integrate(ctx, y0, steps, func, keep):
        """y1; keep: what backward needs stays in ctx."""
        h = 1.0 / steps
        y = y0.detach()
        saved = []
        with torch.no_grad():
            packed = flow256_pack(func) if _fused_field(func, y) else None
            if packed is not None:
                # the fused adjoint starts from the stage inputs: 48 B a point and step
                if keep:
                    saved = [torch.empty((steps, 4) + tuple(y.shape), dtype=torch.float32, device=y.device)]
                for k in range(steps):
                    y = flow256_step(packed, y, h, saved[0][k] if keep else None)
            else:
                for _ in range(steps):
                    if keep:
                        saved.append(y)
                    y = rk4_step(func, y, h)
        ctx.func, ctx.steps, ctx.h, ctx.packed = func, steps, h, packed
        ctx.save_for_backward(*saved)
        return y

    @staticmethod
    def _fused_backward(ctx, gy):
        """Per step, last first, mo_flow256_adjoint_step: back through its
        four stages from their inputs (dL/dy), with the weight-gradient
        products over its 4 n stage points added to the integration's partial
        sums; mo_flow256_adjoint_grads turns those into the gradients."""
        import ctypes as C
        from . import _lib
        zs = ctx.saved_tensors[0].contiguous()
        n, dev = zs.shape[2], zs.device
        gp = [torch.zeros(p.shape, dtype=torch.float32, device=dev) for p in ctx.func.parameters()]
        g = gy.contiguous().to(torch.float32)
        if n == 0:
            return (g, None, None, *gp)
        work = torch.empty(int(_lib.load().mo_flow256_adjoint_work_floats(n)), dtype=torch.float32, device=dev)
        ptr = lambda t: C.c_void_p(t.data_ptr())      # noqa: E731
        for k in reversed(range(ctx.steps)):
            gnew = torch.empty(n, 3, dtype=torch.float32, device=dev)
            _lib.call("mo_flow256_adjoint_step", n, ptr(ctx.packed), float(ctx.h), ptr(zs[k]), ptr(g), ptr(gnew),
                      ptr(work), int(k == ctx.steps - 1), pyDeform._stream())
            g = gnew
        if ctx.steps > 0:
            # weights[0..3], biases[0..3]
            order = [gp[i] for pair in zip(range(4), range(4, 8)) for i in pair]
            _lib.call("mo_flow256_adjoint_grads", n, ptr(work), *[ptr(t) for t in order], pyDeform._stream())
        return (g, None, None, *gp)

    @staticmethod
    def backward(ctx, gy):
        if ctx.packed is not None:
            return RK4Adjoint._fused_backward(ctx, gy)
        ys = ctx.saved_tensors
        params = [p for p in ctx.func.parameters()]
        gp = [torch.zeros_like(p) for p in params]
        for n in reversed(range(ctx.steps)):
            with torch.enable_grad():
                y = ys[n].detach().requires_grad_(True)
                y1 = rk4_step(ctx.func, y, ctx.h)
                grads = torch.autograd.grad(y1, [y] + params, gy, allow_unused=True)
            gy = grads[0]
            for i, g in enumerate(grads[1:]):
                if g is not None:
                    gp[i] += g
        return (gy, None, None, *gp)


class _RK4Inference(RK4Adjoint):
    """RK4Adjoint where no gradient can be asked for.  (needs_input_grad says
    which inputs require one whatever the grad mode, and inside a Function's
    forward the mode is always off.)"""

    @staticmethod
    def forward(ctx, y0, steps, func, *params):
        return RK4Adjoint._integrate(ctx, y0, steps, func, False)


def odeint_rk4(func: nn.Module, y0, steps=16):
    """Integrate dy/dt = func(y) over [0, 1] with ``steps`` RK4 steps."""
    f = RK4Adjoint if torch.is_grad_enabled() else _RK4Inference
    return f.apply(y0, steps, func, *func.parameters())


class _DistanceLoss(Function):
    @staticmethod
    def forward(ctx, y, pid):
        ctx.save_for_backward(y)
        ctx.pid = pid
        return (pyDeform.DistanceFieldLoss_forward(y.contiguous(), pid) * 0.5).sum()

    @staticmethod
    def backward(ctx, g):
        (y,) = ctx.saved_tensors
        return g * pyDeform.DistanceFieldLoss_backward(y.contiguous(), ctx.pid), None


class _GraphLoss(Function):
    @staticmethod
    def forward(ctx, y, E, pid):
        ctx.save_for_backward(y, E)
        ctx.pid = pid
        return (pyDeform.GraphEdgeLoss_forward(y.contiguous(), E, pid) * 0.5).sum()

    @staticmethod
    def backward(ctx, g):
        y, E = ctx.saved_tensors
        return g * pyDeform.GraphEdgeLoss_backward(y.contiguous(), E, ctx.pid), None, None


class NeuralODEDeformer(nn.Module):
    """Pushes ``points`` (the first ``n_mesh`` are the source mesh vertices,
    with edges ``E``) through the flow; loss = distance to the target grid
    (all points) + rho^2 * rigidity (mesh edges)."""

    def __init__(self, points, E, pid, n_mesh, rho=0.1, steps=16, hidden=256, seed=0):
        super().__init__()
        self.field = VelocityMLP(hidden, seed).to(points.device)
        self.register_buffer("y0", points.detach().contiguous())
        self.E = E.contiguous()
        self.pid = pid
        self.n_mesh = n_mesh
        self.rho2 = rho * rho
        self.steps = steps
        pyDeform.StoreGraphInformation(self.y0[:n_mesh].contiguous(), self.E, pid)

    def forward(self):
        y1 = odeint_rk4(self.field, self.y0, self.steps)
        lossD = _DistanceLoss.apply(y1, self.pid)
        lossR = _GraphLoss.apply(y1[: self.n_mesh], self.E, self.pid)
        return lossD + self.rho2 * lossR, y1
