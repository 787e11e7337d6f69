"""The calls that programs using this library make, as measurable cases.

Eight kinds of call, each through the entry point a program would use: the
LinOSS, D-LinOSS, selective D-LinOSS, diagonal (LRU / S5) and selective scans,
and the three modules built on them (the D-LinOSS layer, the LinOSS layer, the
Mamba mixer).  ``listed()`` names twelve of them, from a 16 MB inference scan
whose time is latency to the Mamba-block selective scan; ``draw(rng)`` gives
others from the same ranges, ragged sizes included.
"""

import math

import torch

VARIANTS = ("imex1", "imex2", "im", "ex")
# the layer's stability projection and initialisations cover these (ex may grow)
LAYER_VARIANTS = ("imex1", "imex2", "im")
# parameter layouts of the selective D-LinOSS scan: per step, per (step, channel),
# per batch row, per channel
SDL_LAYOUTS = ("LBM", "LM", "BM", "M")


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # Inference of one small LinOSS-IM layer: a few microseconds of scan, so
        # launch and look-back latency are what the caller waits for.
        {"name": "linoss_infer_small", "kind": "linoss", "L": 1024, "B": 8, "P": 64, "train": False},
        # Training step of a D-LinOSS scan, the library's headline shape.
        {"name": "dlinoss_train", "kind": "dlinoss", "variant": "imex1", "dtype": "c64",
         "L": 4096, "B": 32, "P": 128, "train": True},
        # Long-sequence D-LinOSS inference: carries cross hundreds of time chunks.
        {"name": "dlinoss_infer_long", "kind": "dlinoss", "variant": "imex1", "dtype": "c64",
         "L": 65536, "B": 4, "P": 256, "train": False},
        # The double-precision D-LinOSS scan (float64 coefficients), forward and
        # backward: models trained or checked in complex128.
        {"name": "dlinoss_train_c128", "kind": "dlinoss", "variant": "imex2", "dtype": "c128",
         "L": 2048, "B": 8, "P": 128, "train": True},
        # Input-dependent (selective) D-LinOSS parameters, odd sizes.
        {"name": "sdlinoss_train", "kind": "sdlinoss", "variant": "im", "layout": "LBM",
         "L": 1000, "B": 16, "P": 100, "train": True},
        # Training step of an S5 / LRU diagonal scan.
        {"name": "s5_train", "kind": "diag", "dtype": "c64", "L": 2048, "B": 16, "P": 128, "train": True},
        # Sequential recommendation: many short sequences through the gated
        # selective scan, training.
        {"name": "selective_train_short", "kind": "selective", "dtype": "f32", "skip": False,
         "B": 256, "D": 128, "L": 200, "N": 16, "train": True},
        # Mamba-block scale, bf16 storage, skip and gate: the largest case.
        {"name": "selective_train_block_bf16", "kind": "selective", "dtype": "bf16", "skip": True,
         "B": 16, "D": 1536, "L": 2048, "N": 16, "train": True},
        # Training step of one D-LinOSS layer (projections included).
        {"name": "dlinoss_layer_train", "kind": "dlinoss_layer", "variant": "imex1",
         "L": 4096, "B": 32, "H": 128, "P": 128, "train": True},
        # Serving one D-LinOSS layer on a few sequences, odd sizes.
        {"name": "dlinoss_layer_infer", "kind": "dlinoss_layer", "variant": "imex2",
         "L": 1030, "B": 8, "H": 100, "P": 64, "train": False},
        # Training step of one LinOSS-IM layer.
        {"name": "linoss_layer_train", "kind": "linoss_layer", "variant": "IM",
         "L": 1024, "B": 8, "H": 64, "P": 64, "train": True},
        # Training step of one Mamba mixer at the recommendation shape.
        {"name": "mamba_mixer_train", "kind": "mamba", "L": 200, "B": 256, "H": 64, "N": 16, "train": True},
    ]


def _size(rng, lo, hi):
    """A whole number between lo and hi, uniform in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_once(rng):
    kind = rng.choice(("linoss", "dlinoss", "sdlinoss", "diag", "selective", "dlinoss_layer",
                       "linoss_layer", "mamba"))
    train = rng.random() < 0.6
    if kind in ("linoss", "sdlinoss", "diag"):
        case = {"kind": kind, "L": _size(rng, 64, 8192), "B": _size(rng, 1, 64), "P": _size(rng, 16, 256),
                "train": train}
        if kind == "diag":
            case["dtype"] = rng.choice(("c64", "c64", "c128"))
        if kind == "sdlinoss":
            case["variant"] = rng.choice(VARIANTS)
            case["layout"] = rng.choice(SDL_LAYOUTS)
    elif kind == "dlinoss":
        dtype = rng.choice(("c64", "c64", "c128"))
        case = {"kind": kind, "variant": rng.choice(VARIANTS), "dtype": dtype,
                "L": _size(rng, 64, 65536 if dtype == "c64" else 2048), "B": _size(rng, 1, 64),
                "P": _size(rng, 16, 256), "train": train}
    elif kind == "selective":
        dtype = rng.choice(("f32", "f32", "bf16"))
        case = {"kind": kind, "dtype": dtype, "skip": dtype == "bf16" or rng.random() < 0.5,
                "B": _size(rng, 1, 256), "D": _size(rng, 32, 1536), "L": _size(rng, 20, 4096),
                "N": rng.choice((8, 16, 16, 32)), "train": train}
    elif kind == "mamba":
        case = {"kind": kind, "L": _size(rng, 20, 2048), "B": _size(rng, 1, 256),
                "H": 4 * _size(rng, 8, 64), "N": rng.choice((8, 16, 16)), "train": train}
    else:
        case = {"kind": kind, "L": _size(rng, 32, 4096), "B": _size(rng, 1, 32), "H": _size(rng, 16, 256),
                "P": _size(rng, 16, 256), "train": train,
                "variant": rng.choice(LAYER_VARIANTS) if kind == "dlinoss_layer" else rng.choice(("IM", "IMEX"))}
    return case


def _cost(case):
    """About what a pass takes, in steps of one channel: cheap enough to bound a draw."""
    n = case["L"] * case["B"]
    if case["kind"] == "selective":
        return n * case["D"] * case["N"] / 48
    if case["kind"] == "mamba":
        return n * case["H"] * (case["H"] + 64) / 16
    if case["kind"].endswith("_layer"):
        return n * max(case["H"], case["P"]) * (3 if case["kind"] == "linoss_layer" else 1)
    return n * case["P"] * (4 if case.get("dtype") == "c128" else 1)


def draw(rng):
    while True:
        case = _draw_once(rng)
        if 2e4 <= _cost(case) <= (1.2e7 if case["kind"] in ("mamba", "linoss_layer") else 1.6e7):
            return case


# --------------------------------------------------------------------- inputs
class _Draws:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def randn(self, *shape, dtype=torch.float32):
        return torch.randn(*shape, device="cuda", generator=self.g, dtype=dtype)

    def rand(self, *shape, dtype=torch.float32):
        return torch.rand(*shape, device="cuda", generator=self.g, dtype=dtype)

    def crandn(self, *shape, dtype=torch.float32):
        return torch.complex(self.randn(*shape, dtype=dtype), self.randn(*shape, dtype=dtype))


def _stable(a, g, dt):
    """a inside the band in which the damped oscillator is stable for (g, dt)."""
    s = dt * g
    root = torch.sqrt(1.0 + s)
    return torch.clamp(a, (2.0 + s - 2.0 * root) / (dt * dt), (2.0 + s + 2.0 * root) / (dt * dt))


def prepare(case, seed):
    make = _Draws(seed)
    kind, train = case["kind"], case["train"]
    L, B = case["L"], case["B"]
    state = {"case": case}
    if kind in ("dlinoss_layer", "linoss_layer", "mamba"):
        # initialised on the CPU from the seed, as a program that seeds torch does
        torch.manual_seed(seed)
        H = case["H"]
        if kind == "dlinoss_layer":
            from ossm_amd.layers import DampedLinOSSLayer
            # the uniform initialisation: the ring one reaches |lambda| = 1, where the
            # parameter gradients are ill-conditioned in 32 bits
            layer = DampedLinOSSLayer(case["P"], H, variant=case["variant"], initialization="uniform")
        elif kind == "linoss_layer":
            from ossm_amd.linoss import LinOSSLayer
            layer = LinOSSLayer(case["P"], H, case["variant"])
        else:
            from ossm_amd.mamba import MambaMixer
            layer = MambaMixer(H, d_state=case["N"], d_conv=4, expand=2)
        state["layer"] = layer.cuda()
        state["x"] = make.randn(B, L, H).requires_grad_(train)
        state["inputs"] = [state["x"], *state["layer"].parameters()]
        state["go"] = make.randn(B, L, H)
        return state
    if kind == "selective":
        D, N = case["D"], case["N"]
        dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
        u = make.randn(B, D, L).to(dt)
        step = torch.nn.functional.softplus(make.randn(B, D, L) - 4.0).to(dt)
        A = -torch.arange(1, N + 1, device="cuda", dtype=torch.float32).repeat(D, 1)
        state["inputs"] = [u, step, A, make.randn(B, L, N).to(dt), make.randn(B, L, N).to(dt),
                           make.randn(B, D, L).to(dt)]
        state["D"] = make.randn(D) if case["skip"] else None
        state["go"] = make.randn(B, D, L).to(dt)
        if not case["skip"]:
            state["inputs"] = [t.requires_grad_(train) for t in state["inputs"]]
        return state
    P = case["P"]
    real = torch.float64 if case.get("dtype") == "c128" else torch.float32
    if kind == "diag":
        # S5 / LRU: |lambda| in [0.9, 0.999], any phase
        r, th = 0.9 + 0.099 * make.rand(P, dtype=real), 2 * math.pi * make.rand(P, dtype=real)
        lam = torch.polar(r, th)
        b = make.crandn(L, B, P, dtype=real)
        state["inputs"] = [lam.requires_grad_(train), b.requires_grad_(train)]
        state["go"] = make.crandn(L, B, P, dtype=real)
        return state
    if kind == "linoss":
        a = torch.relu(make.randn(P)) + 0.1
        dt = torch.sigmoid(make.randn(P))
        schur = 1.0 / (1.0 + dt * dt * a)
        m = [1.0 - dt * dt * a * schur, -dt * a * schur, dt * schur, schur]
        bu = make.crandn(L, B, P)
        b = torch.stack((bu * (m[0] * dt), bu * (m[2] * dt)), -1).contiguous()
        state["inputs"] = [t.to(torch.complex64).requires_grad_(train) for t in m] + [b.requires_grad_(train)]
        state["go"] = make.crandn(L, B, P, 2)
        return state
    shape = (P,)
    if kind == "sdlinoss":
        shape = {"LBM": (L, B, P), "LM": (L, 1, P), "BM": (1, B, P), "M": (P,)}[case["layout"]]
    g, dt = make.rand(*shape, dtype=real), torch.sigmoid(make.randn(*shape, dtype=real))
    a = 0.1 + 0.9 * make.rand(*shape, dtype=real)
    if case["variant"] in ("imex1", "im"):
        a = _stable(a, g, dt)
    else:
        # discretisations with an explicit part: dt a <= 0.3 <= g keeps |lambda| below one
        dt = 0.3 * dt
        g = 0.3 + 0.3 * g
    state["inputs"] = [t.contiguous().requires_grad_(train)
                       for t in (a, g, dt, make.crandn(L, B, P, dtype=real))]
    state["go"] = make.crandn(L, B, P, dtype=real)
    return state


# ------------------------------------------------------------------- the call
def run(state):
    from ossm_amd import _kernels, bridge
    case, ins = state["case"], state["inputs"]
    kind = case["kind"]
    if kind == "selective" and case["skip"]:
        # the scan with the skip D has no autograd wrapper: a program calls both directions
        u, dt, A, B, C, z = ins
        out, chunks, raw = _kernels.selective_scan_cuda_skip(u, dt, A, B, C, state["D"], z)
        if not case["train"]:
            return out
        return [out, *_kernels.selective_scan_cuda_skip_backward(state["go"], u, dt, A, B, C, state["D"],
                                                                 z, chunks, raw)]
    with torch.set_grad_enabled(case["train"]):
        if kind == "linoss":
            y = bridge.try_run_scan(*ins)
        elif kind == "dlinoss":
            y = bridge.run_dlinoss(case["variant"], *ins)
        elif kind == "sdlinoss":
            y = bridge.run_sdlinoss(case["variant"], *ins)
        elif kind == "diag":
            y = bridge.try_run_s5_scan(*ins)
        elif kind == "selective":
            y = bridge.try_selective_scan(*ins)
        else:
            y = state["layer"](state["x"])
        if not case["train"]:
            return y
        return [y, *torch.autograd.grad(y, ins, state["go"])]


# ----------------------------------------------------------------------- work
def work(case):
    """Every input read once and every output written once (training: the upstream
    gradient read and the gradients written too, and no intermediate); the
    operations of the recurrence and of the projections."""
    L, B, train = case["L"], case["B"], case["train"]
    n, kind = L * B, case["kind"]
    both = 3 if train else 1  # the backward does about twice the forward's operations
    if kind == "selective":
        e = 2 if case["dtype"] == "bf16" else 4
        D, N = case["D"], case["N"]
        rows, states = n * D, n * N
        return {"bytes": e * ((4 + (4 if train else 0)) * rows + (4 if train else 2) * states)
                + 8 * D * N, "flops": both * 7 * rows * N}
    if kind == "mamba":
        H, N = case["H"], case["N"]
        D, R = 2 * H, max(1, math.ceil(H / 16))
        weights = 2 * D * H + D * (R + 2 * N) + R * D + H * D + D * (N + 6)
        return {"bytes": 4 * (n * H * (4 if train else 2) + weights * (2 if train else 1)),
                "flops": both * (2 * n * (3 * D * H + D * (2 * R + 2 * N) + 4 * D) + 7 * n * D * N)}
    if kind.endswith("_layer"):
        H, P = case["H"], case["P"]
        return {"bytes": 4 * (n * H * (4 if train else 2) + (4 * H * P + H + 3 * P) * (2 if train else 1)),
                "flops": both * n * (8 * H * P + 14 * P)}
    P = case["P"]
    e = 16 if case.get("dtype") == "c128" else 8
    ch = n * P
    if kind == "linoss":
        return {"bytes": 16 * ch * (4 if train else 2), "flops": both * 32 * ch}
    if kind == "diag":
        return {"bytes": e * ch * (4 if train else 2), "flops": both * 8 * ch}
    par = {"LBM": ch, "LM": L * P, "BM": B * P, "M": P}[case["layout"]] if kind == "sdlinoss" else P
    return {"bytes": e * ch * (4 if train else 2) + 3 * (e // 2) * par * (2 if train else 1),
            "flops": both * (30 if kind == "sdlinoss" else 14) * ch}


# ------------------------------------------------------------------ tolerances
# About four times the distance from the 64-bit result seen on seeded inputs: the
# parameter gradients of the oscillators, sums over every step, set the larger ones.
def tolerance(case):
    kind = case["kind"]
    if case.get("dtype") == "c128":
        return {"rel": 2e-13}
    if kind == "selective":
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 5e-6}
    return {"rel": {"linoss": 2e-5, "diag": 1e-5, "sdlinoss": 1e-5, "mamba": 2e-5, "dlinoss": 1e-4,
                    "dlinoss_layer": 2e-4, "linoss_layer": 2e-4}[kind]}


# ----------------------------------------------------- the same in 64 bits
def _scan2(m, b0, b1):
    """s_t = M s_{t-1} + b_t, M = [[m0, m1], [m2, m3]] per channel (or per step:
    callables of t); both components stacked over time."""
    s0 = s1 = torch.zeros_like(b0[0])
    out0, out1 = [], []
    at = m if callable(m) else (lambda t: m)
    for t, (x0, x1) in enumerate(zip(b0, b1)):
        m0, m1, m2, m3 = at(t)
        s0, s1 = m0 * s0 + m1 * s1 + x0, m2 * s0 + m3 * s1 + x1
        out0.append(s0)
        out1.append(s1)
    return out0, out1


def _dlinoss(variant, a, g, dt, bu):
    """x of the D-LinOSS recurrence; a, g, dt broadcast against bu [L, B, P]."""
    if variant == "imex1":
        s = 1.0 + dt * g
        k = (1 / s, -dt * a / s * dt, 1 / s, 1 - dt * dt * a / s, dt * dt / s, dt * dt / s)
    elif variant == "imex2":
        k = (1 - dt * g, -dt * a, dt - dt * dt * g, 1 - dt * dt * a, dt, dt * dt)
    elif variant == "im":
        s = 1.0 + dt * g + dt * dt * a
        k = (1 / s, -dt * a / s, dt / s, (1 + dt * g) / s, dt / s, dt * dt / s)
    else:
        one = torch.ones_like(a)
        k = (1 - dt * g, -dt * a, dt, one, dt, 0 * one)
    return torch.stack(_scan2(k[:4], (bu * k[4]).unbind(0), (bu * k[5]).unbind(0))[1])


def _sdlinoss(variant, a, g, step, bu):
    """Selective D-LinOSS: w' = (alpha w + dt^2 (bu - a x)) / S, x' = x + w'."""
    full = bu.shape
    dt = torch.clamp(step, 1e-6, 1.0)
    alpha = 1 - dt * g if variant in ("imex2", "ex") else torch.ones_like(dt)
    s = {"imex1": 1 + dt * g, "imex2": 1 + dt * dt * a, "im": 1 + dt * g + dt * dt * a,
         "ex": torch.ones_like(dt * g * a)}[variant].clamp(min=1e-6)
    c0, c1, f = alpha / s, -dt * dt * a / s, dt * dt / s
    fb = (f * bu).unbind(0)
    c0, c1 = (t.expand(full).unbind(0) for t in (c0, c1))
    w = x = torch.zeros_like(fb[0])
    out = []
    for t in range(full[0]):
        w = c0[t] * w + c1[t] * x + fb[t]
        x = x + w
        out.append(x)
    return torch.stack(out)


def _selective(u, dt, A, B, C, z, D=None):
    """u, dt, z [B, D, L]; A [D, N]; B, C [B, L, N]."""
    us, ds, bs, cs = u.unbind(2), dt.unbind(2), B.unbind(1), C.unbind(1)
    h = torch.zeros(u.size(0), u.size(1), A.size(1), dtype=u.dtype, device=u.device)
    ys = []
    for ut, dtt, bt, ct in zip(us, ds, bs, cs):
        h = torch.exp(dtt.unsqueeze(-1) * A) * h + (dtt * ut).unsqueeze(-1) * bt.unsqueeze(1)
        ys.append((h * ct.unsqueeze(1)).sum(-1))
    y = torch.stack(ys, 2)
    if D is not None:
        y = y + D[:, None] * u
    return y * torch.nn.functional.silu(z)


def _cproj(u, w):
    """u [..., H] with complex weights w [P, H, 2]."""
    return torch.complex(u @ w[..., 0].t().contiguous(), u @ w[..., 1].t().contiguous())


def _out(x, c, d, u):
    """Re(x C^T) + D u from x [L, B, P]."""
    x = x.permute(1, 0, 2)
    return x.real @ c[..., 0].t().contiguous() - x.imag @ c[..., 1].t().contiguous() + u * d


def _dlinoss_layer(variant, u, a_p, g_p, s_p, b, c, d):
    dt, g = torch.sigmoid(s_p), torch.relu(g_p)
    dt2, dg = dt * dt, dt * g
    root = torch.sqrt(1 + dg)
    lo, hi = (2 + dg - 2 * root) / dt2, (2 + dg + 2 * root) / dt2
    a = lo + torch.relu(a_p - lo) - torch.relu(a_p - hi)
    bu = _cproj(u, b).permute(1, 0, 2)
    return _out(_dlinoss(variant, a, g, dt, bu), c, d, u)


def _linoss_layer(variant, u, a_p, b, c, d, s_p):
    a, dt = torch.relu(a_p), torch.sigmoid(s_p)
    bu = _cproj(u, b).permute(1, 0, 2)
    if variant == "IM":
        s = 1 / (1 + dt * dt * a)
        m = (1 - dt * dt * a * s, -dt * a * s, dt * s, s)
        f = (m[0] * dt, m[2] * dt)
    else:
        m = (torch.ones_like(a), -dt * a, dt, 1 - dt * dt * a)
        f = (dt, dt * dt)
    return _out(torch.stack(_scan2(m, (bu * f[0]).unbind(0), (bu * f[1]).unbind(0))[1]), c, d, u)


def _mamba(u, p):
    """The mixer from its named parameters."""
    xz = u @ p["in_proj.weight"].t()
    di = xz.size(-1) // 2
    x, z = xz[..., :di], xz[..., di:]
    w = p["conv1d.weight"][:, 0]  # [D, K]
    K = w.size(1)
    xp = torch.nn.functional.pad(x, (0, 0, K - 1, 0))
    x = sum(xp[:, k:k + u.size(1)] * w[:, k] for k in range(K)) + p["conv1d.bias"]
    x = torch.nn.functional.silu(x)
    proj = x @ p["x_proj.weight"].t()
    A = -torch.exp(p["A_log"])
    N, R = A.size(1), p["dt_proj.weight"].size(1)
    dt = torch.nn.functional.softplus(proj[..., :R] @ p["dt_proj.weight"].t() + p["dt_proj.bias"])
    y = _selective(x.transpose(1, 2), dt.transpose(1, 2), A, proj[..., R:R + N], proj[..., R + N:],
                   z.transpose(1, 2))
    return y.transpose(1, 2) @ p["out_proj.weight"].t()


def _wide(t):
    wide = t.detach().to(torch.complex128 if t.is_complex() else torch.float64)
    return wide.requires_grad_(True)


def exact(case, seed):
    state = prepare(case, seed)
    kind, train = case["kind"], case["train"]
    ins = [_wide(t) for t in state["inputs"]]
    with torch.set_grad_enabled(train):
        if kind == "linoss":
            b = ins[4]
            y = torch.stack(tuple(torch.stack(s) for s in
                                  _scan2(ins[:4], b[..., 0].unbind(0), b[..., 1].unbind(0))), -1)
        elif kind == "dlinoss":
            y = _dlinoss(case["variant"], *ins)
        elif kind == "sdlinoss":
            y = _sdlinoss(case["variant"], *ins)
        elif kind == "diag":
            x, xs = torch.zeros_like(ins[1][0]), []
            for bt in ins[1].unbind(0):
                x = ins[0] * x + bt
                xs.append(x)
            y = torch.stack(xs)
        elif kind == "selective":
            if case["skip"]:
                ins.append(_wide(state["D"]))
            y = _selective(*ins)
        elif kind == "mamba":
            names = [k for k, _ in state["layer"].named_parameters()]
            y = _mamba(ins[0], dict(zip(names, ins[1:])))
        else:
            names = [k for k, _ in state["layer"].named_parameters()]
            p = dict(zip(names, ins[1:]))
            if kind == "dlinoss_layer":
                y = _dlinoss_layer(case["variant"], ins[0], p["A_diag"], p["G_diag"], p["steps"],
                                   p["B"], p["C"], p["D"])
            else:
                y = _linoss_layer(case["variant"], ins[0], p["A_diag"], p["B"], p["C"], p["D"], p["steps"])
        if not train:
            return y
        go = state["go"].to(y.dtype)
        grads = list(torch.autograd.grad(y, ins, go))
    if kind == "selective" and case["skip"]:
        # the backward's order: du, ddt, dA, dB, dC, dD, dgate
        grads = grads[:5] + [grads[6], grads[5]]
    return [y.detach(), *grads]
