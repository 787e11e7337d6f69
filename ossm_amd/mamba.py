"""The Mamba mixer with its pre/post-processing fused around the selective scan.

The reference mixer (``_MambaMixer``, mambarec.py:63-184) runs, between its
projections, a transpose + pad + depthwise Conv1d + SiLU, a softplus pass over
dt, transposes of x_conv, dt and z to ``[B, D, L]`` for the scan (plus
``.contiguous()`` copies) and a transpose of the output.  Here:

* ``ossm_mamba_conv_forward/backward``: the causal depthwise conv + SiLU in the
  mixer's ``[B, L, D]`` layout, reading x straight out of ``in_proj``'s output;
* ``ossm_selective_mamba_forward/backward``: the selective scan reading u, dt
  (before its softplus, with the dt_proj bias) and the gate z in ``[B, L, D]``
  with row strides (z and B, C stay views into the projection outputs) and
  writing ``[B, L, D]`` for ``out_proj``.

``MambaMixer`` has the reference module's constructor arguments and parameter
names (``in_proj``, ``conv1d``, ``x_proj``, ``dt_proj``, ``out_proj``,
``A_log``), so a reference ``state_dict`` loads unchanged.  Device float32
only; there is no CPU path (CPU inputs raise).
"""

from __future__ import annotations

import math
from typing import Optional, Tuple

import torch
import torch.nn.functional as F
from torch import Tensor, nn

from . import _lib
from .linear import is_plain, linear, linear_weight, rows_product

__all__ = ["MambaMixer", "mamba_conv_silu", "selective_scan_mamba", "ConvSiluFn", "MambaScanFn",
           "MixerCoreFn"]


def _rows(t: Tensor, name: str) -> Tuple[Tensor, int]:
    """A ``[B, L, C]`` float32 device tensor as (tensor, row stride): views whose
    last dimension is contiguous and whose batch stride is L row strides pass
    as they are; anything else is made contiguous."""
    if t.dim() != 3:
        raise RuntimeError(f"{name} must be (batch, length, channels), got {tuple(t.shape)}")
    if t.dtype != torch.float32 or not t.is_cuda:
        raise RuntimeError(f"{name} must be a float32 GPU tensor (got {t.dtype} on {t.device})")
    Bz, L, C = t.shape
    ok = t.stride(2) == 1 and t.stride(1) >= C and (Bz <= 1 or t.stride(0) == L * t.stride(1))
    if not ok:
        t = t.contiguous()
    return t, int(t.stride(1)) if L > 0 else C


def _param(t: Optional[Tensor], name: str) -> Optional[Tensor]:
    """A parameter the kernels read as contiguous float32 on the device."""
    if t is None:
        return None
    if t.dtype != torch.float32 or not t.is_cuda:
        raise RuntimeError(f"{name} must be a float32 GPU tensor (got {t.dtype} on {t.device})")
    return t.contiguous()


def _same_device(*ts: Optional[Tensor]) -> None:
    devs = {t.device for t in ts if t is not None}
    if len(devs) > 1:
        raise RuntimeError(f"tensors on different devices: {sorted(map(str, devs))}")


# ------------------------------------------------------------------ conv + SiLU
def _conv_fwd(x: Tensor, weight: Tensor, bias: Optional[Tensor]) -> Tensor:
    x, ld = _rows(x, "x")
    Bz, L, D = x.shape
    w = _param(weight, "conv weight").reshape(D, -1)
    b = _param(bias, "conv bias")
    if b is not None and tuple(b.shape) != (D,):
        raise RuntimeError(f"conv bias must have shape ({D},), got {tuple(b.shape)}")
    _same_device(x, w, b)
    out = torch.empty((Bz, L, D), dtype=torch.float32, device=x.device)
    if out.numel() == 0:
        return out
    with torch.cuda.device(x.device):
        _lib.check(_lib.load().ossm_mamba_conv_forward(
            x.data_ptr(), ld, w.data_ptr(), _lib.ptr(b), out.data_ptr(), Bz, L, D, w.size(1),
            _lib.stream_of(x)))
    return out


class ConvSiluFn(torch.autograd.Function):
    """silu(causal depthwise conv1d(x) + bias) in ``[B, L, D]``."""

    @staticmethod
    def forward(ctx, x: Tensor, weight: Tensor, bias: Optional[Tensor]) -> Tensor:  # type: ignore[override]
        ctx.save_for_backward(x, weight, bias)
        ctx.has_bias = bias is not None
        return _conv_fwd(x, weight, bias)

    @staticmethod
    def backward(ctx, grad_out: Tensor):  # type: ignore[override]
        x, weight, bias = ctx.saved_tensors
        x, ld = _rows(x, "x")
        Bz, L, D = x.shape
        w = _param(weight, "conv weight").reshape(D, -1)
        K = w.size(1)
        go = grad_out.contiguous()
        gx = torch.empty((Bz, L, D), dtype=torch.float32, device=x.device)
        gw = torch.empty((D, K), dtype=torch.float32, device=x.device)
        gb = torch.empty((D,), dtype=torch.float32, device=x.device) if ctx.has_bias else None
        with torch.cuda.device(x.device):
            _lib.check(_lib.load().ossm_mamba_conv_backward(
                x.data_ptr(), ld, w.data_ptr(), _lib.ptr(bias), go.data_ptr(), gx.data_ptr(),
                gw.data_ptr(), _lib.ptr(gb), Bz, L, D, K, _lib.stream_of(x)))
        return gx, gw.reshape(weight.shape), gb


def mamba_conv_silu(x: Tensor, weight: Tensor, bias: Optional[Tensor] = None) -> Tensor:
    """``silu(Conv1d(pad_left(x^T, K-1)))^T`` of mambarec.py:143-150 for x
    ``[B, L, D]`` (a strided view is read in place); weight ``[D, 1, K]`` or
    ``[D, K]``; returns ``[B, L, D]``."""
    return ConvSiluFn.apply(x, weight, bias)


# ------------------------------------------------------------- selective scan
class MambaScanFn(torch.autograd.Function):
    """Selective scan in ``[B, L, D]`` with dt before its softplus."""

    @staticmethod
    def forward(ctx, u: Tensor, dt: Tensor, A: Tensor, Bm: Tensor, Cm: Tensor,
                z: Optional[Tensor], dt_bias: Optional[Tensor]) -> Tensor:  # type: ignore[override]
        lib = _lib.load()
        u, ld_u = _rows(u, "inputs")
        dt, ld_dt = _rows(dt, "dt")
        Bm, ld_b = _rows(Bm, "B")
        Cm, ld_c = _rows(Cm, "C")
        if ld_b != ld_c or (Cm.data_ptr() - Bm.data_ptr()) % 4 != 0:
            Bm, Cm = Bm.contiguous(), Cm.contiguous()
            ld_b = ld_c = Bm.size(2)
        ld_z = 0
        if z is not None:
            z, ld_z = _rows(z, "gate")
        Bz, L, D = u.shape
        N = A.size(1)
        if tuple(dt.shape) != (Bz, L, D) or tuple(A.shape) != (D, N) or \
                tuple(Bm.shape) != (Bz, L, N) or tuple(Cm.shape) != (Bz, L, N) or \
                (z is not None and tuple(z.shape) != (Bz, L, D)) or \
                (dt_bias is not None and tuple(dt_bias.shape) != (D,)):
            raise RuntimeError("selective_scan_mamba: inconsistent shapes "
                               f"u {tuple(u.shape)} dt {tuple(dt.shape)} A {tuple(A.shape)} "
                               f"B {tuple(Bm.shape)} C {tuple(Cm.shape)}")
        Ac = _param(A, "A")
        bias = _param(dt_bias, "dt_bias")
        _same_device(u, dt, Ac, Bm, Cm, z, bias)
        out = torch.empty((Bz, L, D), dtype=torch.float32, device=u.device)
        raw = torch.empty_like(out) if z is not None else None
        n_chunks = int(lib.ossm_selective_num_chunks(L))
        ck = torch.empty((Bz, D, n_chunks, 2 * N), dtype=torch.float32, device=u.device)
        if out.numel() > 0:
            with torch.cuda.device(u.device):
                _lib.check(lib.ossm_selective_mamba_forward(
                    u.data_ptr(), ld_u, dt.data_ptr(), ld_dt, _lib.ptr(bias), Ac.data_ptr(),
                    Bm.data_ptr(), Cm.data_ptr(), ld_b, _lib.ptr(z), ld_z, out.data_ptr(),
                    _lib.ptr(raw), ck.data_ptr(), Bz, D, L, N, _lib.stream_of(u)))
        ctx.has_z = z is not None
        ctx.has_bias = bias is not None
        ctx.lds = (ld_u, ld_dt, ld_b, ld_z)
        ctx.save_for_backward(u, dt, Ac, Bm, Cm, z, bias, ck, raw)
        return out

    @staticmethod
    def backward(ctx, grad_out: Tensor):  # type: ignore[override]
        u, dt, A, Bm, Cm, z, bias, ck, raw = ctx.saved_tensors
        ld_u, ld_dt, ld_b, ld_z = ctx.lds
        Bz, L, D = u.shape
        N = A.size(1)
        go = grad_out.contiguous()
        dev = u.device
        du = torch.empty((Bz, L, D), dtype=torch.float32, device=dev)
        ddt = torch.empty_like(du)
        dz = torch.empty_like(du) if ctx.has_z else None
        dA = torch.empty((D, N), dtype=torch.float32, device=dev)
        dB = torch.empty((Bz, L, N), dtype=torch.float32, device=dev)
        dC = torch.empty_like(dB)
        with torch.cuda.device(dev):
            _lib.check(_lib.load().ossm_selective_mamba_backward(
                go.data_ptr(), u.data_ptr(), ld_u, dt.data_ptr(), ld_dt, _lib.ptr(bias),
                A.data_ptr(), Bm.data_ptr(), Cm.data_ptr(), ld_b, _lib.ptr(z), ld_z, ck.data_ptr(),
                _lib.ptr(raw), du.data_ptr(), ddt.data_ptr(), dA.data_ptr(), dB.data_ptr(),
                dC.data_ptr(), _lib.ptr(dz), Bz, D, L, N, _lib.stream_of(u)))
        dbias = ddt.sum(dim=(0, 1)) if ctx.has_bias else None
        return du, ddt, dA, dB, dC, dz, dbias


def selective_scan_mamba(inputs: Tensor, dt: Tensor, A: Tensor, B: Tensor, C: Tensor,
                         gate: Optional[Tensor] = None, dt_bias: Optional[Tensor] = None) -> Tensor:
    """``y = scan(u, softplus(dt + dt_bias), A, B, C) * silu(gate)`` with every
    ``[B, L, *]`` tensor in the mixer's layout (the reference scan,
    mambarec.py:23-61 and selective_scan_cuda.cu:253-310, on transposes)."""
    return MambaScanFn.apply(inputs, dt, A, B, C, gate, dt_bias)


def _all_float(xz: Tensor, params) -> bool:
    """xz and the parameters as they are: plain float32 tensors on one GPU, no autocast."""
    return (not torch.is_autocast_enabled("cuda") and not torch.compiler.is_compiling()
            and all(t is None or (type(t) in (Tensor, nn.Parameter) and t.dtype == torch.float32
                                  and t.device == xz.device) for t in (xz, *params)))


def _core_shapes(Di: int, R: int, N: int, xz: Tensor, conv_w: Tensor, conv_b: Optional[Tensor],
                 xproj_w: Tensor, dt_w: Tensor, dt_b: Optional[Tensor], A_log: Tensor) -> bool:
    """Whether a mixer of d_inner ``Di``, dt_rank ``R`` and d_state ``N`` has these shapes."""
    return (xz.dim() == 3 and xz.size(2) == 2 * Di
            and conv_w.dim() > 1 and conv_w.size(0) == Di and conv_w.numel() == Di * conv_w.size(-1)
            and (conv_b is None or conv_b.shape == (Di,)) and xproj_w.shape == (R + 2 * N, Di)
            and dt_w.shape == (Di, R) and dt_b is not None and dt_b.shape == (Di,) and A_log.shape == (Di, N))


class _ColumnSplit(torch.autograd.Function):
    """``xz[..., :d], xz[..., d:]`` as views, whose backward writes the gradient
    of ``xz`` in one pass (torch.cat of the two); slicing the tensor directly
    would, in the backward, zero-fill the whole ``[B, L, 2d]`` gradient once per
    slice, copy each slice's gradient in and add the two."""

    @staticmethod
    def forward(ctx, xz: Tensor, d: int):  # type: ignore[override]
        ctx.d = d
        ctx.shape = xz.shape
        return xz[..., :d], xz[..., d:]

    @staticmethod
    def backward(ctx, gx: Optional[Tensor], gz: Optional[Tensor]):  # type: ignore[override]
        d, shape = ctx.d, ctx.shape
        if gx is None and gz is None:
            return None, None
        ref = gx if gx is not None else gz
        if gx is None:
            gx = torch.zeros(*shape[:-1], d, dtype=ref.dtype, device=ref.device)
        if gz is None:
            gz = torch.zeros(*shape[:-1], shape[-1] - d, dtype=ref.dtype, device=ref.device)
        return torch.cat([gx, gz], dim=-1), None


def _mixer_core(xz: Tensor, conv_w: Tensor, conv_b: Optional[Tensor], xproj_w: Tensor, dt_w: Tensor,
                dt_b: Tensor, A_log: Tensor) -> Tensor:
    """``MixerCoreFn`` as separate steps."""
    R, N = dt_w.size(1), A_log.size(1)
    x, z = _ColumnSplit.apply(xz, dt_w.size(0))
    u = mamba_conv_silu(x, conv_w, conv_b)
    proj = linear_weight(u, xproj_w)
    dt = linear_weight(proj[..., :R], dt_w)
    return selective_scan_mamba(u, dt, -torch.exp(A_log), proj[..., R:R + N], proj[..., R + N:], gate=z, dt_bias=dt_b)


class MixerCoreFn(torch.autograd.Function):
    """The mixer between its in and out projections, ``xz`` [B, L, 2 Di] to
    ``y`` [B, L, Di]: conv + SiLU, x_proj, dt_proj, the gated scan.  Its backward
    writes the gradient of ``xz`` and that of x_proj's output in place, part by
    part (the scan the gate's half, B and C; the conv the x half; a product the dt
    part), and adds x_proj's into the scan's du in its own product, where separate
    Functions zero-filled, copied, added and concatenated them: 9 launches and
    about 90 us of a [256, 200, 64] training step's kernels, and as many host
    calls."""

    @staticmethod
    def forward(ctx, xz: Tensor, conv_w: Tensor, conv_b: Optional[Tensor], xproj_w: Tensor,
                dt_w: Tensor, dt_b: Tensor, A_log: Tensor) -> Tensor:  # type: ignore[override]
        params = (conv_w, conv_b, xproj_w, dt_w, dt_b, A_log)
        if dt_w.dim() != 2 or A_log.dim() != 2 or \
                not _core_shapes(*dt_w.shape, A_log.size(1), xz, *params):
            raise RuntimeError("mixer: inconsistent shapes xz, conv weight, conv bias, x_proj, dt_proj, dt bias, "
                               f"A_log: {[t if t is None else tuple(t.shape) for t in (xz, *params)]}")
        index = xz.get_device()
        for t in (xz, *params):
            if t is not None and (t.dtype is not torch.float32 or index < 0 or t.get_device() != index):
                raise RuntimeError("mixer: every tensor must be a float32 GPU tensor, on one device")
        Di, R, N = dt_w.size(0), dt_w.size(1), A_log.size(1)
        lib = _lib.load()
        given, xz = xz, xz.contiguous()
        Bz, L, ld = xz.shape
        w = conv_w.reshape(Di, -1).contiguous()
        dev, st = xz.device, _lib.stream_of(xz)
        bias, dtb = _param(conv_b, "conv bias"), dt_b.contiguous()
        u = torch.empty((Bz, L, Di), dtype=torch.float32, device=dev)
        with torch.cuda.device(dev):
            _lib.check(lib.ossm_mamba_conv_forward(xz.data_ptr(), ld, w.data_ptr(), _lib.ptr(bias),
                                                   u.data_ptr(), Bz, L, Di, w.size(1), st))
            proj = F.linear(u, xproj_w)
            dt = F.linear(proj[..., :R], dt_w)  # its bias goes into the softplus
            A = -torch.exp(A_log.contiguous())
            y, raw = torch.empty_like(u), torch.empty_like(u)
            ck = torch.empty((Bz, Di, int(lib.ossm_selective_num_chunks(L)), 2 * N), dtype=torch.float32,
                             device=dev)
            pp, z = proj.data_ptr() + 4 * R, xz.data_ptr() + 4 * Di
            _lib.check(lib.ossm_selective_mamba_forward(
                u.data_ptr(), Di, dt.data_ptr(), Di, dtb.data_ptr(), A.data_ptr(), pp, pp + 4 * N,
                R + 2 * N, z, ld, y.data_ptr(), raw.data_ptr(), ck.data_ptr(), Bz, Di, L, N, st))
        ctx.save_for_backward(given, u, proj, dt, A, ck, raw, conv_w, conv_b, xproj_w, dt_w, dt_b,
                              A_log)
        return y

    @staticmethod
    def backward(ctx, gy: Tensor):  # type: ignore[override]
        xz, u, proj, dt, A, ck, raw, conv_w, conv_b, xproj_w, dt_w, dt_b, A_log = ctx.saved_tensors
        if torch.is_grad_enabled():
            # create_graph: differentiable again, as separate steps
            inputs = (xz, conv_w, conv_b, xproj_w, dt_w, dt_b, A_log)
            wanted = [t for t, n in zip(inputs, ctx.needs_input_grad) if n]
            got = iter(torch.autograd.grad(_mixer_core(*inputs), wanted, gy, create_graph=True, allow_unused=True))
            return tuple(next(got) if n else None for n in ctx.needs_input_grad)
        xz = xz.contiguous()
        Di, R, N = dt_w.size(0), dt_w.size(1), A.size(1)
        Bz, L, ld = xz.shape
        rows, ldp = Bz * L, R + 2 * N
        dev, st, lib = xz.device, _lib.stream_of(xz), _lib.load()
        gy = gy.contiguous()
        w = conv_w.reshape(Di, -1).contiguous()
        bias, dtb = _param(conv_b, "conv bias"), dt_b.contiguous()
        # of xproj_w, dt_w, dt_b, as the forward's arguments are numbered
        need_xp, need_dtw, need_dtb = ctx.needs_input_grad[3:6]
        with torch.no_grad(), torch.cuda.device(dev):
            new = lambda *s: torch.empty(s, dtype=torch.float32, device=dev)  # noqa: E731
            gxz, gproj, du, ddt = torch.empty_like(xz), torch.empty_like(proj), new(Bz, L, Di), new(Bz, L, Di)
            dA, gw = new(Di, N), new(Di, w.size(1))
            gb = new(Di) if bias is not None else None
            pp, gp = proj.data_ptr() + 4 * R, gproj.data_ptr() + 4 * R
            _lib.check(lib.ossm_selective_mamba_backward_ld(
                gy.data_ptr(), u.data_ptr(), Di, dt.data_ptr(), Di, dtb.data_ptr(), A.data_ptr(), pp,
                pp + 4 * N, ldp, xz.data_ptr() + 4 * Di, ld, ck.data_ptr(), raw.data_ptr(), du.data_ptr(),
                ddt.data_ptr(), dA.data_ptr(), gp, gp + 4 * N, ldp, gxz.data_ptr() + 4 * Di, ld, Bz, Di, L,
                N, st))
            ddt2, gproj2, u2 = ddt.view(rows, Di), gproj.view(rows, ldp), u.view(rows, Di)
            torch.mm(ddt2, dt_w, out=gproj2[:, :R])
            du.view(rows, Di).addmm_(gproj2, xproj_w)
            _lib.check(lib.ossm_mamba_conv_backward_ld(
                xz.data_ptr(), ld, w.data_ptr(), _lib.ptr(bias), du.data_ptr(), gxz.data_ptr(), ld,
                gw.data_ptr(), _lib.ptr(gb), Bz, L, Di, w.size(1), st))
            g_dtw = rows_product(ddt2, proj.view(rows, ldp)[:, :R]) if need_dtw else None
            g_xp = rows_product(gproj2, u2) if need_xp else None
            g_dtb = ddt2.sum(0) if need_dtb else None
            return gxz, gw.view(conv_w.shape), gb, g_xp, g_dtw, g_dtb, dA.mul_(A)


# ------------------------------------------------------------------ the mixer
class MambaMixer(nn.Module):
    """Mamba mixer (reference ``_MambaMixer``, mambarec.py:63-184) whose conv,
    softplus, gate and layout changes run inside this library's kernels."""

    def __init__(self, d_model: int, *, d_state: int, d_conv: int, expand: int,
                 dt_rank: int | str = "auto", dt_min: float = 0.001, dt_max: float = 0.1,
                 dt_init: str = "random", dt_scale: float = 1.0, dt_init_floor: float = 1e-4,
                 conv_bias: bool = True, bias: bool = False) -> None:
        super().__init__()
        if dt_rank == "auto":
            dt_rank = max(1, math.ceil(d_model / 16))
        self.d_model = int(d_model)
        self.d_state = int(d_state)
        self.d_conv = int(d_conv)
        self.expand = int(expand)
        self.d_inner = self.expand * self.d_model
        self.dt_rank = int(dt_rank)
        self.in_proj = nn.Linear(self.d_model, 2 * self.d_inner, bias=bias)
        self.conv1d = nn.Conv1d(self.d_inner, self.d_inner, kernel_size=self.d_conv,
                                groups=self.d_inner, bias=conv_bias, padding=0)
        self.x_proj = nn.Linear(self.d_inner, self.dt_rank + 2 * self.d_state, bias=False)
        self.dt_proj = nn.Linear(self.dt_rank, self.d_inner, bias=True)
        self.out_proj = nn.Linear(self.d_inner, self.d_model, bias=bias)
        # dt_proj: weights uniform or constant at dt_rank^-1/2 * dt_scale; bias =
        # softplus^-1 of dt log-uniform on [dt_min, dt_max] (mambarec.py:111-126)
        std = self.dt_rank ** -0.5 * dt_scale
        if dt_init == "constant":
            nn.init.constant_(self.dt_proj.weight, std)
        elif dt_init == "random":
            nn.init.uniform_(self.dt_proj.weight, -std, std)
        else:
            raise ValueError("dt_init must be 'random' or 'constant'")
        log_lo, log_hi = math.log(dt_min), math.log(dt_max)
        dt = torch.exp(torch.rand(self.d_inner) * (log_hi - log_lo) + log_lo).clamp(min=dt_init_floor)
        with torch.no_grad():
            self.dt_proj.bias.copy_(dt + torch.log(-torch.expm1(-dt)))
        self.dt_proj.bias._no_reinit = True  # type: ignore[attr-defined]
        # A = -(1 .. d_state) per channel, stored as its log (mambarec.py:128-131)
        A = torch.arange(1, self.d_state + 1, dtype=torch.float32).repeat(self.d_inner, 1)
        self.A_log = nn.Parameter(torch.log(A))
        self.A_log._no_weight_decay = True  # type: ignore[attr-defined]
        self.register_parameter("D", None)

    def forward(self, inputs: Tensor) -> Tensor:
        if inputs.ndim != 3:
            raise ValueError("Inputs to Mamba mixer must have shape (batch, length, channels)")
        if inputs.size(1) == 0:
            return torch.zeros_like(inputs)
        if not inputs.is_cuda:
            raise RuntimeError("the fused Mamba mixer runs on the GPU only")
        Di, R, N = self.d_inner, self.dt_rank, self.d_state
        xz = linear(self.in_proj, inputs).float()
        params = (self.conv1d.weight, self.conv1d.bias, self.x_proj.weight, self.dt_proj.weight,
                  self.dt_proj.bias, self.A_log)
        # replaced parameters that do not have the mixer's sizes take the separate steps
        if is_plain(self.x_proj) and self.x_proj.bias is None and xz.numel() > 0 and _all_float(xz, params) \
                and params[3].shape == (Di, R) and params[5].shape == (Di, N) and params[0].size(0) == Di:
            y = MixerCoreFn.apply(xz, *params)
            return linear(self.out_proj, y.to(self.out_proj.weight.dtype))
        x, z = _ColumnSplit.apply(xz, Di)                 # views, row stride 2 * d_inner
        x_conv = mamba_conv_silu(x, self.conv1d.weight.float(),
                                 None if self.conv1d.bias is None else self.conv1d.bias.float())
        proj = linear(self.x_proj, x_conv.to(self.x_proj.weight.dtype)).float()
        dt_raw, B_gen, C_gen = proj[..., :R], proj[..., R:R + N], proj[..., R + N:]
        dt_pre = linear_weight(dt_raw, self.dt_proj.weight.float())  # bias goes into the softplus
        A = -torch.exp(self.A_log.float())
        y = selective_scan_mamba(x_conv, dt_pre, A, B_gen, C_gen, gate=z,
                                 dt_bias=self.dt_proj.bias.float())
        return linear(self.out_proj, y.to(self.out_proj.weight.dtype))
