"""D-LinOSS layer whose forward is one fused MI355X kernel.

``DampedLinOSSLayer`` has the reference module's interface (dlinoss.py:48-278):
the same constructor arguments, parameter names and shapes (``A_diag``,
``G_diag``, ``steps`` [P]; ``B`` [P, H, 2]; ``C`` [H, P, 2]; ``D`` [H]), the
same stable-region projection and the same forward contract, so a reference
``state_dict`` loads unchanged.

Forward on a GPU float32 (or bf16 / fp16, computed in float32 as the
reference does) input is ``ossm_dlinoss_layer_forward``: the in-projection
``bu = u B^T``, the D-LinOSS scan and ``y = Re(x C^T) + D u`` in one launch,
with bu and the states kept on chip; for training it also saves the state
entering each 32-step chunk.  The backward is ``ossm_dlinoss_layer_backward``
(the projections of the upstream gradient and of u on the matrix cores, the
states re-run from those carries, the scan adjoint, grad_u), followed by the
two weight-gradient products over the grad_bu and x it returns.  Shapes whose
backward does not fit one workgroup's LDS recompute through the unfused
composition (``unfused_layer_forward``) and differentiate that.

No CPU path computes here: CPU tensors go through the same composition, whose
scan delegates to the reference's CPU module when it is installed (as the
rest of the drop-in does) and raises otherwise.  float64 raises: the device
kernels compute in float32 / complex64.
"""

from __future__ import annotations

import math
from typing import Optional, Tuple

import torch
from torch import Tensor, nn

from . import _lib
from .bridge import run_dlinoss
from .linear import BLOCK_ROWS, rows_product

__all__ = ["DampedLinOSSLayer", "dlinoss_layer_forward", "dlinoss_layer_backward", "DlinossLayerFn",
           "project_parameters", "unfused_layer_forward", "LayerParamsFn", "fused_layer_supported"]

_VARIANTS = {"imex1": 0, "imex2": 1, "im": 2, "ex": 3}
_LAYER_MAX = 256  # largest hidden_dim / ssm_size of the fused kernel
_CHUNK = 32       # steps per workgroup chunk (the carries' second dimension)
_LDS = 160 * 1024


def _bwd_fits(hidden: int, ssm: int) -> bool:
    """The fused backward's LDS (u or gy rows with bu over them, grad_bu tiles)
    fits one workgroup (mirrors layer_bwd_lds_bytes in dlinoss_layer.hip; true
    for every size up to 256)."""
    hp, pp = -(-hidden // 32) * 32, -(-ssm // 32) * 32
    return (_CHUNK * max(hp + 4, 2 * pp + 4) + _CHUNK * (2 * pp + 4) + 4 * ssm) * 4 <= _LDS


def project_parameters(A_diag: Tensor, G_diag: Tensor, steps: Tensor) -> Tuple[Tensor, Tensor, Tensor]:
    """(a, g, dt) inside the stability region (reference _project_parameters,
    dlinoss.py:249-264): dt = sigmoid(steps), g = relu(G), a clamped to
    [(2 + dt g - 2 sqrt(1 + dt g)) / dt^2, (2 + dt g + 2 sqrt(1 + dt g)) / dt^2]
    with the clamp written as relu differences (the same values and gradients)."""
    dt = torch.sigmoid(steps)
    g = torch.relu(G_diag)
    dt2 = torch.clamp(dt * dt, min=1e-6)
    dg = dt * g
    root = torch.sqrt(torch.clamp(1.0 + dg, min=1e-6))
    lo = (2.0 + dg - 2.0 * root) / dt2
    hi = (2.0 + dg + 2.0 * root) / dt2
    a = lo + torch.relu(A_diag - lo) - torch.relu(A_diag - hi)
    return a, g, dt


class LayerParamsFn(torch.autograd.Function):
    """(a, g, dt, lo) of a layer from its stored float32 GPU parameters, one launch
    each way: ``project_parameters`` when ``damped`` (the same float operations;
    ``lo`` is None), else the LinOSS layer's ``(relu(A), 0, sigmoid(steps))``, with
    G_diag None and ``lo`` [3, P] what rounding each to float32 left."""

    @staticmethod
    def forward(ctx, damped: bool, A_diag: Tensor, G_diag: Optional[Tensor],
                steps: Tensor):  # type: ignore[override]
        shape, index = A_diag.shape, A_diag.get_device()
        rest = (G_diag, steps) if damped else (steps,)
        for t in rest:
            if t is None or len(shape) != 1 or t.shape != shape:
                raise RuntimeError("oscillator parameters must be vectors of one length, got "
                                   f"{[x if x is None else tuple(x.shape) for x in (A_diag, *rest)]}")
        for t in (A_diag, *rest):
            if t.dtype is not torch.float32 or index < 0 or t.get_device() != index:
                raise RuntimeError("oscillator parameters must be float32 GPU tensors, on one device")
        A, G, s = (None if t is None else t.contiguous() for t in (A_diag, G_diag, steps))
        out = torch.empty((6, A.numel()), dtype=torch.float32, device=A.device)
        _lib.run(_lib.load().ossm_layer_params_forward, A, int(damped), A.data_ptr(), _lib.ptr(G),
                 s.data_ptr(), out.data_ptr(), A.numel())
        ctx.damped = damped
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(A_diag, G_diag, steps)
        lo = None
        if not damped:
            lo = out[3:]
            ctx.mark_non_differentiable(lo)
        return out[0], out[1], out[2], lo

    @staticmethod
    def backward(ctx, *grads: Optional[Tensor]):  # type: ignore[override]
        params, grads = ctx.saved_tensors, grads[:3]
        if torch.is_grad_enabled():
            # create_graph: differentiable again, as torch operations
            A, G, s = params
            outs = project_parameters(A, G, s) if ctx.damped else \
                (torch.relu(A), None, torch.sigmoid(s))
            pairs = [(o, g) for o, g in zip(outs, grads) if o is not None and g is not None]
            wanted = [t for t, n in zip(params, ctx.needs_input_grad[1:]) if n]
            got = iter(torch.autograd.grad([o for o, _ in pairs], wanted, [g for _, g in pairs],
                                           create_graph=True, allow_unused=True) if pairs else
                       [None] * len(wanted))
            return (None, *[next(got) if n else None for n in ctx.needs_input_grad[1:]])
        A, G, s = (None if t is None else t.contiguous() for t in params)
        up = [None if g is None else g.contiguous() for g in grads]
        out = torch.empty((3, A.numel()), dtype=torch.float32, device=A.device)
        _lib.run(_lib.load().ossm_layer_params_backward, A, int(ctx.damped), A.data_ptr(), _lib.ptr(G),
                 s.data_ptr(), *[_lib.ptr(g) for g in up], out.data_ptr(), A.numel())
        return (None, *[out[i] if n else None for i, n in enumerate(ctx.needs_input_grad[1:])])


def _layer_sizes_fit(batch: int, length: int, hidden: int, ssm: int) -> bool:
    """The fused layer kernels' size limits (those ossm_dlinoss_layer_* refuse above)."""
    return (hidden <= _LAYER_MAX and ssm <= _LAYER_MAX and batch * ssm <= (2 ** 31 - 1) // 8
            and batch * -(-length // _CHUNK) < 2 ** 31)


def fused_layer_supported(inputs: Tensor, params, hidden: int, ssm: int) -> bool:
    """Whether a LinOSS layer with ``params`` (A_diag, B, C, D, steps) runs as the fused
    kernel on ``inputs`` as it is: float32 throughout on one GPU, no autocast, nothing
    empty, nothing that broadcasts."""
    return (inputs.is_cuda and inputs.dtype == torch.float32 and inputs.numel() > 0 and ssm > 0
            and _layer_sizes_fit(inputs.size(0), inputs.size(1), hidden, ssm)
            and all(t.dtype is torch.float32 and t.device == inputs.device for t in params)
            and params[0].shape == params[4].shape == (ssm,) and params[3].shape == (hidden,)
            and params[1].shape == (ssm, hidden, 2) and params[2].shape == (hidden, ssm, 2)
            and not torch.is_autocast_enabled("cuda"))


def _check_layer_args(inputs: Tensor, B: Tensor, C: Tensor, D: Tensor, a: Tensor, g: Tensor,
                      step: Tensor) -> Tuple[int, int, int, int]:
    if inputs.dim() != 3:
        raise ValueError("DampedLinOSSLayer expects input of shape (batch, length, hidden_dim).")
    batch, length, hidden = inputs.shape
    if B.dim() != 3 or B.size(1) != hidden or B.size(2) != 2:
        raise RuntimeError(f"B must have shape (ssm_size, {hidden}, 2), got {tuple(B.shape)}")
    ssm = B.size(0)
    if C.shape != (hidden, ssm, 2):
        raise RuntimeError(f"C must have shape ({hidden}, {ssm}, 2), got {tuple(C.shape)}")
    if D.shape != (hidden,):
        raise RuntimeError(f"D must have shape ({hidden},), got {tuple(D.shape)}")
    for name, t in (("a_diag", a), ("g_diag", g), ("step", step)):
        if t.shape != (ssm,):
            raise RuntimeError(f"{name} must have shape ({ssm},), got {tuple(t.shape)}")
    return batch, length, hidden, ssm


def _check_on_gpu(tensors, hidden: int, ssm: int) -> None:
    index = tensors[0].get_device()
    one = index >= 0
    for t in tensors:
        if t.dtype is not torch.float32:
            raise RuntimeError("the fused D-LinOSS layer computes in float32; got "
                               + ", ".join(str(x.dtype) for x in tensors))
        if t.get_device() != index:
            one = False
    if not one:
        raise RuntimeError("the fused D-LinOSS layer needs every tensor on one GPU")
    if hidden > _LAYER_MAX or ssm > _LAYER_MAX:
        raise RuntimeError(f"the fused D-LinOSS layer supports hidden_dim and ssm_size up to "
                           f"{_LAYER_MAX}, got {hidden} and {ssm}")


def _check_carries(carries: Tensor, batch: int, length: int, ssm: int, device) -> None:
    want = (batch, -(-length // _CHUNK), ssm, 4)
    if tuple(carries.shape) != want or carries.dtype != torch.float32 or \
            not carries.is_contiguous() or carries.device != device:
        raise RuntimeError(f"carries must be a contiguous float32 {want} tensor on {device}")


def _check_lo(lo: Optional[Tensor], a: Tensor) -> Optional[Tensor]:
    if lo is not None and (tuple(lo.shape) != (3, a.numel()) or lo.dtype != torch.float32
                           or not lo.is_contiguous() or lo.device != a.device):
        raise RuntimeError(f"lo must be a contiguous float32 (3, {a.numel()}) tensor on {a.device}")
    return lo


def dlinoss_layer_forward(variant: str, inputs: Tensor, B: Tensor, C: Tensor, D: Tensor,
                          a_diag: Tensor, g_diag: Tensor, step: Tensor,
                          carries: Optional[Tensor] = None, lo: Optional[Tensor] = None) -> Tensor:
    """y = Re(x C^T) + D u with x the D-LinOSS states driven by bu = u B^T, in
    one kernel launch.  Every tensor float32 on one GPU; a, g, step projected.
    ``carries`` (float32 [batch, ceil(length / 32), ssm, 4]) receives the state
    entering each chunk, for ``dlinoss_layer_backward``.  ``lo`` ([3, ssm], from
    ``LayerParamsFn``): what a, g, step leave of their double values; the
    coefficients are formed in double from the sums."""
    variant = variant.lower()
    if variant not in _VARIANTS:
        raise ValueError(f"Unknown D-LinOSS variant '{variant}'.")
    batch, length, hidden, ssm = _check_layer_args(inputs, B, C, D, a_diag, g_diag, step)
    tensors = (inputs, B, C, D, a_diag, g_diag, step)
    _check_on_gpu(tensors, hidden, ssm)
    u, Bc, Cc, Dc, a, g, s = (t.contiguous() for t in tensors)
    out = torch.empty_like(u)
    if out.numel() == 0:
        return out
    if carries is not None:
        _check_carries(carries, batch, length, ssm, u.device)
    _lib.run(_lib.load().ossm_dlinoss_layer_forward_wide, u, _VARIANTS[variant], u.data_ptr(),
             Bc.data_ptr(), Cc.data_ptr(), Dc.data_ptr(), a.data_ptr(), g.data_ptr(), s.data_ptr(),
             _lib.ptr(_check_lo(lo, a)), out.data_ptr(), _lib.ptr(carries), batch, length, hidden, ssm)
    return out


def dlinoss_layer_backward(variant: str, inputs: Tensor, grad_output: Tensor, B: Tensor,
                           C: Tensor, D: Tensor, a_diag: Tensor, g_diag: Tensor, step: Tensor,
                           carries: Tensor, lo: Optional[Tensor] = None):
    """Gradients of the fused layer: ``(grad_inputs, grad_B, grad_C, grad_D, grad_a,
    grad_g, grad_step)`` from the forward's ``carries`` (and
    ``lo``).  One kernel for
    grad_inputs and the scan's parameter gradients; grad_B and grad_C are row
    products over the grad_bu and conj(x) it returns."""
    variant = variant.lower()
    if variant not in _VARIANTS:
        raise ValueError(f"Unknown D-LinOSS variant '{variant}'.")
    batch, length, hidden, ssm = _check_layer_args(inputs, B, C, D, a_diag, g_diag, step)
    if grad_output.shape != inputs.shape:
        raise RuntimeError(f"grad_output must have the inputs' shape {tuple(inputs.shape)}, "
                           f"got {tuple(grad_output.shape)}")
    tensors = (inputs, grad_output, B, C, D, a_diag, g_diag, step)
    _check_on_gpu(tensors, hidden, ssm)
    u, go, Bc, Cc, Dc, a, g, s = (t.contiguous() for t in tensors)
    dev = u.device
    _check_carries(carries, batch, length, ssm, dev)
    gu = torch.empty_like(u)
    gbu = torch.empty((batch, length, ssm, 2), dtype=torch.float32, device=dev)
    xq = torch.empty_like(gbu)
    ga, gg, gs = (torch.empty(ssm, dtype=torch.float32, device=dev) for _ in range(3))
    gD = torch.empty(hidden, dtype=torch.float32, device=dev)
    _lib.run(_lib.load().ossm_dlinoss_layer_backward_wide, u, _VARIANTS[variant], u.data_ptr(),
             go.data_ptr(), Bc.data_ptr(), Cc.data_ptr(), Dc.data_ptr(), a.data_ptr(), g.data_ptr(),
             s.data_ptr(), _lib.ptr(_check_lo(lo, a)), carries.data_ptr(), gu.data_ptr(), gbu.data_ptr(),
             xq.data_ptr(), ga.data_ptr(), gg.data_ptr(), gs.data_ptr(), gD.data_ptr(), batch, length,
             hidden, ssm)
    rows = batch * length
    uf, gof = u.reshape(rows, hidden), go.reshape(rows, hidden)
    # grad_B[p, h, c] = sum_r grad_bu[r, p, c] u[r, h];  grad_C[h, p, c] = sum_r go[r, h] xq[r, p, c]
    gbu2, xq2 = gbu.reshape(rows, 2 * ssm), xq.reshape(rows, 2 * ssm)
    if rows >= BLOCK_ROWS:
        gB, gC = rows_product(gbu2, uf, pairs=True), rows_product(gof, xq2)
    else:
        gB = _sum_rows_product(gbu2, uf).reshape(ssm, 2, hidden).permute(0, 2, 1).contiguous()
        gC = _sum_rows_product(gof, xq2)
    gC = gC.reshape(hidden, ssm, 2)
    return gu, gB, gC, gD, ga, gg, gs


def _sum_rows_product(a: Tensor, b: Tensor, split: int = 32) -> Tensor:
    """a^T b for row-major a [R, M], b [R, N] of fewer rows than ``rows_product``
    takes: the first split * (R // split) rows as ``split`` slices of one batched
    GEMM, the partials added, the remaining rows by one small GEMM."""
    R = a.size(0)
    n = R // split
    if n < 4:
        return a.t() @ b
    head = split * n
    out = torch.bmm(a[:head].view(split, n, -1).transpose(1, 2), b[:head].view(split, n, -1)).sum(0)
    if head < R:
        out += a[head:].t() @ b[head:]
    return out


def unfused_layer_forward(variant: str, inputs: Tensor, B: Tensor, C: Tensor, D: Tensor,
                          a_diag: Tensor, g_diag: Tensor, step: Tensor) -> Tensor:
    """The layer as separate steps (dlinoss.py:210-247): two real GEMMs for bu,
    the scan (``run_dlinoss``, this library's kernels), two GEMMs for Re(x C^T)
    and the D skip.  Differentiable; the fused layer's backward runs through it."""
    batch, length, hidden, ssm = _check_layer_args(inputs, B, C, D, a_diag, g_diag, step)
    flat = inputs.reshape(batch * length, hidden)
    bu = torch.complex(flat @ B[..., 0].t().contiguous(), flat @ B[..., 1].t().contiguous())
    bu_seq = bu.reshape(batch, length, ssm).permute(1, 0, 2).contiguous()
    if length == 0:
        x = bu_seq
    else:
        x = run_dlinoss(variant, a_diag, g_diag, step, bu_seq)
    xf = x.permute(1, 0, 2).reshape(batch * length, ssm)
    proj = xf.real @ C[..., 0].t().contiguous() - xf.imag @ C[..., 1].t().contiguous()
    return proj.reshape(batch, length, hidden) + inputs * D


class DlinossLayerFn(torch.autograd.Function):
    """Fused forward and backward (``dlinoss_layer_backward``); shapes whose
    backward does not fit, and backwards that are differentiated again, go
    through ``unfused(variant, inputs, B, C, D, a_diag, g_diag, step)``, the same
    layer as separate differentiable steps."""

    @staticmethod
    def forward(ctx, variant: str, inputs: Tensor, B: Tensor, C: Tensor, D: Tensor,
                a_diag: Tensor, g_diag: Tensor, step: Tensor, lo: Optional[Tensor] = None,
                unfused=unfused_layer_forward) -> Tensor:  # type: ignore[override]
        ctx.variant = variant
        ctx.unfused = unfused
        batch, length, hidden = inputs.shape
        ssm = B.size(0)
        carries = None
        if any(ctx.needs_input_grad[1:8]) and _bwd_fits(hidden, ssm):
            carries = torch.empty((batch, -(-length // _CHUNK), ssm, 4), dtype=torch.float32,
                                  device=inputs.device)
        ctx.fused_bwd = carries is not None
        ctx.save_for_backward(inputs, B, C, D, a_diag, g_diag, step, carries, lo)
        return dlinoss_layer_forward(variant, inputs, B, C, D, a_diag, g_diag, step, carries, lo)

    @staticmethod
    def backward(ctx, grad_out: Tensor):  # type: ignore[override]
        *saved, carries, lo = ctx.saved_tensors
        needs = ctx.needs_input_grad[1:8]
        tail = (None,) * (len(ctx.needs_input_grad) - 8)  # lo and unfused, where they were passed
        again = torch.is_grad_enabled()  # create_graph
        if ctx.fused_bwd and not again:
            grads = dlinoss_layer_backward(ctx.variant, *saved[:1], grad_out, *saved[1:], carries, lo)
            return (None, *[gr if n else None for gr, n in zip(grads, needs)], *tail)
        with torch.enable_grad():
            args = saved if again else [t.detach().requires_grad_(bool(n)) for t, n in zip(saved, needs)]
            wanted = [t for t, n in zip(args, needs) if n]
            y = ctx.unfused(ctx.variant, *args)
            got = iter(torch.autograd.grad(y, wanted, grad_out, create_graph=again, allow_unused=True)
                       if wanted else ())
        return (None, *[next(got) if n else None for n in needs], *tail)


class DampedLinOSSLayer(nn.Module):
    """Single damped LinOSS layer (reference DampedLinOSSLayer, dlinoss.py:48-278)."""

    def __init__(self, ssm_size: int, hidden_dim: int, *, variant: str = "imex1",
                 initialization: str = "ring", r_min: float = 0.9, r_max: float = 1.0,
                 theta_min: float = 0.0, theta_max: float = math.pi, A_min: float = 0.0,
                 A_max: float = 1.0, G_min: float = 0.0, G_max: float = 1.0,
                 dt_std: float = 0.5) -> None:
        super().__init__()
        variant = variant.lower()
        if variant not in _VARIANTS:
            raise ValueError("DampedLinOSSLayer received unsupported variant "
                             f"'{variant}'. Expected one of {', '.join(_VARIANTS)}.")
        self.variant = variant
        self.ssm_size = ssm_size
        self.hidden_dim = hidden_dim
        self.init_config = dict(initialization=initialization.lower(), r_min=float(r_min),
                                r_max=float(r_max), theta_min=float(theta_min),
                                theta_max=float(theta_max), A_min=float(A_min), A_max=float(A_max),
                                G_min=float(G_min), G_max=float(G_max), dt_std=float(dt_std))
        self.A_diag = nn.Parameter(torch.empty(ssm_size))
        self.G_diag = nn.Parameter(torch.empty(ssm_size))
        self.steps = nn.Parameter(torch.empty(ssm_size))
        self.B = nn.Parameter(torch.empty(ssm_size, hidden_dim, 2))
        self.C = nn.Parameter(torch.empty(hidden_dim, ssm_size, 2))
        self.D = nn.Parameter(torch.empty(hidden_dim))
        self.reset_parameters()

    # -- initialisation (dlinoss.py:100-174) ---------------------------------
    def reset_parameters(self) -> None:
        nn.init.uniform_(self.B, -1.0 / math.sqrt(self.hidden_dim), 1.0 / math.sqrt(self.hidden_dim))
        nn.init.uniform_(self.C, -1.0 / math.sqrt(self.ssm_size), 1.0 / math.sqrt(self.ssm_size))
        nn.init.normal_(self.D, mean=0.0, std=1.0)
        kind = self.init_config["initialization"]
        if kind == "ring":
            a, g, steps = self._ring_values()
        elif kind == "uniform":
            a, g, steps = self._uniform_values()
        else:
            raise ValueError(f"Unknown initialization '{kind}'.")
        with torch.no_grad():
            self.A_diag.copy_(a)
            self.G_diag.copy_(g)
            self.steps.copy_(steps)

    def _ring_values(self) -> Tuple[Tensor, Tensor, Tensor]:
        """Eigenvalue pairs r e^{+-i theta} with r^2 uniform on [r_min^2, r_max^2]
        and theta uniform, mapped to (a, g) for dt = sigmoid(N(0, dt_std^2)): the
        pair's product fixes 1 / (1 + dt g), its sum then fixes a."""
        cfg, n = self.init_config, self.ssm_size
        dtype, device = self.A_diag.dtype, self.A_diag.device
        steps = torch.randn(n, dtype=dtype, device=device) * cfg["dt_std"]
        dt = torch.sigmoid(steps)
        r2 = torch.rand(n, dtype=dtype, device=device) * (cfg["r_max"] ** 2 - cfg["r_min"] ** 2) \
            + cfg["r_min"] ** 2
        theta = torch.rand(n, dtype=dtype, device=device) * (cfg["theta_max"] - cfg["theta_min"]) \
            + cfg["theta_min"]
        pair_sum = 2.0 * torch.sqrt(r2) * torch.cos(theta)
        pair_prod = r2
        g = (1.0 / torch.clamp(pair_prod, min=1e-6) - 1.0) / torch.clamp(dt, min=1e-6)
        g = torch.clamp(g, min=cfg["G_min"])
        a = (2.0 + dt * g - pair_sum * (1.0 + dt * g)) / torch.clamp(dt * dt, min=1e-6)
        return a, g, steps

    def _uniform_values(self) -> Tuple[Tensor, Tensor, Tensor]:
        """(A, G) uniform on their boxes and steps ~ N(0, dt_std^2), kept where the
        discrete oscillator is underdamped (G >= 0 and (G - dt A)^2 < 4 A,
        dlinoss.py:177-179), drawn until ssm_size samples are kept."""
        cfg, n = self.init_config, self.ssm_size
        dtype, device = self.A_diag.dtype, self.A_diag.device
        draw = max(4 * n, 512)
        kept: list[Tuple[Tensor, Tensor, Tensor]] = []
        total = 0
        while total < n:
            A = torch.rand(draw, dtype=dtype, device=device) * (cfg["A_max"] - cfg["A_min"]) + cfg["A_min"]
            G = torch.rand(draw, dtype=dtype, device=device) * (cfg["G_max"] - cfg["G_min"]) + cfg["G_min"]
            s = torch.randn(draw, dtype=dtype, device=device) * cfg["dt_std"]
            dt = torch.sigmoid(s)
            ok = (G >= 0) & ((G - dt * A) ** 2 - 4.0 * A < 0)
            if ok.any():
                kept.append((A[ok], G[ok], s[ok]))
                total += int(ok.sum())
        return tuple(torch.cat([k[i] for k in kept])[:n] for i in range(3))  # type: ignore[return-value]

    # -- forward (dlinoss.py:184-247) ----------------------------------------
    def forward(self, inputs: Tensor) -> Tensor:
        if inputs.dim() != 3:
            raise ValueError("DampedLinOSSLayer expects input of shape (batch, length, hidden_dim).")
        if inputs.size(-1) != self.hidden_dim:
            raise ValueError(f"Expected hidden_dim={self.hidden_dim}, received {inputs.size(-1)}.")
        dtype = inputs.dtype
        if dtype == torch.float64:
            raise RuntimeError("the MI355X D-LinOSS kernels compute in float32/complex64; "
                               "got float64 inputs")
        compute = torch.float32
        u = inputs.to(compute)
        params = [t.to(device=u.device, dtype=compute) for t in
                  (self.A_diag, self.G_diag, self.steps, self.B, self.C, self.D)]
        Bw, Cw, Dw = params[3:]
        if u.is_cuda and self.hidden_dim <= _LAYER_MAX and self.ssm_size <= _LAYER_MAX:
            if params[0].shape == params[1].shape == params[2].shape == (self.ssm_size,):
                a, g, dt, _ = LayerParamsFn.apply(True, *params[:3])
            else:  # replaced parameters may broadcast
                a, g, dt = project_parameters(*params[:3])
            y = DlinossLayerFn.apply(self.variant, u, Bw, Cw, Dw, a, g, dt)
        else:
            a, g, dt = project_parameters(*params[:3])
            y = unfused_layer_forward(self.variant, u, Bw, Cw, Dw, a, g, dt)
        return y if dtype == compute else y.to(dtype)
