"""The work that programs built on this package ask of it, as measurable cases.

Each case is one call (or one layer's worth of calls) through the public entry points, at sizes of
this repository's own configurations: the decode step of a Mamba layer, the decode-time and prefill
calls of the selective scan with and without the low-rank P/Q coupling, their training steps, and
the fused block. Activations lie in memory as the Motif block hands them over ("module": delta
channel-major from its GEMM, z the second half of the input projection), or dense.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "motif-mamba_amd"))

import motif_mamba_amd as mm  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # One token of one sequence through a 2.8B-width layer: conv update and state update. What
        # a chat at batch 1 runs per layer and token; latency and launches.
        dict(name="decode_b1", kind="decode", batch=1, dim=5120, dstate=16, dtype="bf16"),
        # The same step for a full serving batch: the states' memory traffic.
        dict(name="decode_b256", kind="decode", batch=256, dim=5120, dstate=16, dtype="bf16"),
        # One token of 64 sequences through a Motif 1.4B-width layer: its step calls the coupled
        # scan with one time step.
        dict(name="pq_step_b64", kind="pq_prefill", batch=64, dim=4096, L=1, dstate=16, rank=2, shared=False,
             groups=1, dtype="fp16", layout="dense"),
        # Two prompts of an odd length through a 130M-width layer.
        dict(name="prefill_130m_odd", kind="prefill", batch=2, dim=1536, L=1777, dstate=16, groups=1,
             dtype="bf16", layout="module"),
        # The prompt pass of a 2.8B-width layer, the headline workload of bench.py.
        dict(name="prefill_2p8b", kind="prefill", batch=4, dim=5120, L=4096, dstate=16, groups=1, dtype="bf16",
             layout="module"),
        # A very long document in float32 with grouped B and C (length extrapolation).
        dict(name="prefill_long_fp32", kind="prefill", batch=1, dim=2560, L=65536, dstate=16, groups=4,
             dtype="fp32", layout="dense"),
        # The prompt pass of a Motif 1.4B-width layer with its rank-2 coupling.
        dict(name="pq_prefill_1p4b", kind="pq_prefill", batch=4, dim=4096, L=2048, dstate=16, rank=2,
             shared=False, groups=1, dtype="fp16", layout="module"),
        # A training step of the 130M-width scan (forward and backward).
        dict(name="train_130m", kind="train", batch=8, dim=1536, L=2048, dstate=16, groups=1, dtype="bf16",
             layout="module"),
        # A training step at the Motif "base" preset's d_state 64, without coupling.
        dict(name="train_base_n64", kind="train", batch=8, dim=1536, L=1024, dstate=64, groups=1, dtype="bf16",
             layout="module"),
        # A training step of the Motif 1.4B-width layer with its coupling (d_state 16).
        dict(name="pq_train_1p4b", kind="pq_train", batch=4, dim=4096, L=2048, dstate=16, rank=2, shared=False,
             groups=1, dtype="fp16", layout="module"),
        # A training step at the Motif "small" preset's d_state 32, with coupling.
        dict(name="pq_train_small_n32", kind="pq_train", batch=8, dim=1024, L=1024, dstate=32, rank=2,
             shared=False, groups=1, dtype="bf16", layout="module"),
        # A whole 2.8B-width block between its projections, forward and backward.
        dict(name="block_train_2p8b", kind="block", batch=4, d_model=2560, L=4096, dstate=16, train=True,
             dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """Mostly whatever a prompt or document has, sometimes a multiple of 64 (packed training rows)."""
    L = _log_int(rng, lo, hi)
    return max(64, L // 64 * 64) if rng.random() < 0.35 and L >= 64 else L


def draw(rng):
    kind = rng.choice(["decode", "pq_prefill", "prefill", "prefill", "pq_prefill", "train", "pq_train", "block"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if kind == "decode":
        return dict(kind=kind, batch=_log_int(rng, 1, 256), dim=64 * _log_int(rng, 8, 80),
                    dstate=rng.choice([16, 16, 16, 32, 64]), dtype=dtype)
    if kind == "block":
        c = dict(kind=kind, batch=rng.randint(1, 4), d_model=64 * _log_int(rng, 4, 40), L=_length(rng, 64, 4096),
                 dstate=rng.choice([16, 16, 32]), train=rng.random() < 0.6, dtype=rng.choice(["bf16", "bf16", "fp16"]))
        if c["dstate"] == 32:
            c["d_model"] = min(c["d_model"], 1024)
        return c
    c = dict(kind=kind, batch=_log_int(rng, 1, 16), dim=32 * _log_int(rng, 8, 160), L=_length(rng, 24, 8192),
             dstate=rng.choice([16, 16, 16, 8, 32, 64]))
    if kind == "prefill" and rng.random() < 0.15:
        c["batch"], c["L"] = 1, _length(rng, 8192, 65536)
    if kind == "pq_prefill" and rng.random() < 0.25:
        c["batch"], c["L"] = _log_int(rng, 1, 256), 1
    if kind in ("pq_prefill", "pq_train"):
        c.update(rank=rng.choice([1, 2, 2, 2, 4, 8]), shared=rng.random() < 0.25)
    groups = rng.choice([1, 1, 1, 2, 4])
    c.update(groups=groups if c["dim"] % (16 * groups) == 0 else 1, dtype=dtype,
             layout="dense" if c["L"] == 1 else rng.choice(["module", "dense"]))
    # No dearer than the listed ones of the kind.
    most = {"prefill": 4 * 5120 * 4096 * 16, "pq_prefill": 4 * 4096 * 2048 * 16, "train": 8 * 1536 * 2048 * 16,
            "pq_train": 8 * 1024 * 1024 * 32}[kind]
    while c["batch"] * c["dim"] * c["L"] * c["dstate"] > most:
        if c["batch"] > 1:
            c["batch"] = (c["batch"] + 1) // 2
        elif c["L"] > 64:
            c["L"] = (c["L"] * 2) // 3
        else:
            c["dim"] = max(32, c["dim"] // 64 * 32)
            c["groups"] = 1
    return c


# ---- inputs --------------------------------------------------------------------------------------


class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def n(self, *shape, scale=1.0):
        return torch.randn(*shape, device="cuda", generator=self.g) * scale

    def u(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, device="cuda", generator=self.g) * (hi - lo) + lo


def _delta_bias(r, dim):
    # softplus(delta_bias) between 1e-3 and 1e-1, as the module initialises its dt projection.
    dt = torch.exp(r.u(dim, lo=math.log(1e-3), hi=math.log(1e-1)))
    return (dt + torch.log(-torch.expm1(-dt))).float()


def _A(r, dim, n):
    # The S4D-real start -1 .. -n, moved a little by training.
    a = torch.arange(1, n + 1, device="cuda", dtype=torch.float32)
    return -(a * torch.exp(r.n(dim, n, scale=0.1))).contiguous()


def _scan_inputs(c, r):
    b, d, L, n, G = c["batch"], c["dim"], c["L"], c["dstate"], c["groups"]
    dt = DTYPES[c["dtype"]]
    t = {"u": r.n(b, d, L).to(dt)}
    if c["layout"] == "module":
        t["delta"] = r.n(d, b, L).to(dt).transpose(0, 1)
        t["z"] = r.n(b, 2 * d, L).to(dt)[:, d:]
    else:
        t["delta"] = r.n(b, d, L).to(dt)
        t["z"] = r.n(b, d, L).to(dt)
    t["A"] = _A(r, d, n)
    t["B"] = r.n(b, n, L).to(dt) if G == 1 else r.n(b, G, n, L).to(dt)
    t["C"] = r.n(b, n, L).to(dt) if G == 1 else r.n(b, G, n, L).to(dt)
    t["D"] = 1.0 + r.n(d, scale=0.1)
    t["delta_bias"] = _delta_bias(r, d)
    if c["kind"].startswith("pq"):
        R = c["rank"]
        t["P"] = r.n(n, R, scale=0.1) if c["shared"] else r.n(d, n, R, scale=0.1)
        t["Q"] = r.n(R, n, scale=0.1) if c["shared"] else r.n(d, R, n, scale=0.1)
    return t


def _decode_inputs(c, r):
    b, d, n = c["batch"], c["dim"], c["dstate"]
    dt = DTYPES[c["dtype"]]
    return dict(conv_state=r.n(b, d, 4).to(dt), state=r.n(b, d, n, scale=0.1), x=r.n(b, d).to(dt),
                dt=r.n(b, d).to(dt), z=r.n(b, d).to(dt), B=r.n(b, n).to(dt), C=r.n(b, n).to(dt),
                w=r.n(d, 4, scale=0.5).to(dt), wb=r.n(d, scale=0.1).to(dt), A=_A(r, d, n), D=1.0 + r.n(d, scale=0.1),
                dt_bias=_delta_bias(r, d))


def _block_inputs(c, r):
    b, m, L, n = c["batch"], c["d_model"], c["L"], c["dstate"]
    d, R = 2 * m, -(-m // 16)
    dt = DTYPES[c["dtype"]]
    return dict(xz=r.n(b, 2 * d, L).to(dt), conv_w=r.n(d, 1, 4, scale=0.5).to(dt), conv_b=r.n(d, scale=0.1).to(dt),
                x_proj=r.n(R + 2 * n, d, scale=d ** -0.5).to(dt), dt_proj=r.n(d, R, scale=R ** -0.5).to(dt),
                out_proj=r.n(m, d, scale=d ** -0.5).to(dt), A=_A(r, d, n), D=1.0 + r.n(d, scale=0.1),
                delta_bias=_delta_bias(r, d))


def _inputs(case, seed):
    r = _Rand(seed)
    kind = case["kind"]
    t = _decode_inputs(case, r) if kind == "decode" else _block_inputs(case, r) if kind == "block" else _scan_inputs(case, r)
    if kind in ("train", "pq_train"):
        t["dout"] = r.n(case["batch"], case["dim"], case["L"]).to(DTYPES[case["dtype"]])
    elif kind == "block" and case["train"]:
        t["dout"] = r.n(case["batch"], case["L"], case["d_model"]).to(DTYPES[case["dtype"]])
    return t


def _trains(case):
    return case["kind"] in ("train", "pq_train") or (case["kind"] == "block" and case["train"])


def prepare(case, seed):
    t = _inputs(case, seed)
    if _trains(case):
        for k, v in t.items():
            if k != "dout":
                v.requires_grad_(True)
    return {"case": case, "t": t}


# ---- one pass ------------------------------------------------------------------------------------

_SCAN_GRADS = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "P", "Q")
_BLOCK_GRADS = ("xz", "conv_w", "conv_b", "x_proj", "dt_proj", "out_proj", "A", "D", "delta_bias")


def _block(t):
    return mm.mamba_inner_fn(t["xz"], t["conv_w"], t["conv_b"], t["x_proj"], t["dt_proj"], t["out_proj"], None,
                             t["A"], None, None, t["D"], t["delta_bias"], delta_softplus=True)


def run(state):
    case, t = state["case"], state["t"]
    kind = case["kind"]
    if kind == "decode":
        x = mm.causal_conv1d_update(t["x"], t["conv_state"], t["w"], t["wb"], activation="silu")
        y = mm.selective_state_update(t["state"], x, t["dt"], t["A"], t["B"], t["C"], t["D"], z=t["z"],
                                      dt_bias=t["dt_bias"], dt_softplus=True)
        return {"conv_state": t["conv_state"], "state": t["state"], "x": x, "y": y}
    if kind == "block":
        if not case["train"]:
            with torch.no_grad():
                return {"y": _block(t)}
        y = _block(t)
        g = torch.autograd.grad(y, [t[k] for k in _BLOCK_GRADS], t["dout"])
        return {"y": y.detach(), **{"d" + k: v for k, v in zip(_BLOCK_GRADS, g)}}
    args = {k: t[k] for k in ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "P", "Q") if k in t}
    if kind in ("prefill", "pq_prefill"):
        with torch.no_grad():
            out, last = mm.selective_scan_fn(**args, delta_softplus=True, return_last_state=True)
        return {"out": out, "last_state": last}
    out = mm.selective_scan_fn(**args, delta_softplus=True)
    names = [k for k in _SCAN_GRADS if k in args]
    g = torch.autograd.grad(out, [args[k] for k in names], t["dout"])
    return {"out": out.detach(), **{"d" + k: v for k, v in zip(names, g)}}


# ---- what a pass cannot do without ---------------------------------------------------------------


def work(case):
    kind, s = case["kind"], SIZES[case["dtype"]]
    if kind == "decode":
        b, d, n = case["batch"], case["dim"], case["dstate"]
        # conv state and ssm state read and written; x, dt, z read, conv x and y written; B, C; weights.
        return {"bytes": b * (2 * 4 * d * s + 2 * d * n * 4 + 5 * d * s + 2 * n * s) + d * (5 * s + 4 * n + 8),
                "flops": b * d * (8 + 7 * n)}
    if kind == "block":
        b, m, L, n = case["batch"], case["d_model"], case["L"], case["dstate"]
        d, R = 2 * m, -(-m // 16)
        gemm = 2 * b * L * (d * (R + 2 * n) + R * d + d * m)
        weights = s * (d * 5 + d * (R + 2 * n) + R * d + d * m) + 4 * (d * n + 2 * d)
        fwd = {"bytes": s * b * L * (2 * d + m) + weights, "flops": gemm + b * L * d * (8 + 7 * n)}
        if not case["train"]:
            return fwd
        return {"bytes": s * b * L * (4 * d + 2 * m) + 2 * weights, "flops": 3 * gemm + b * L * d * (24 + 21 * n)}
    b, d, L, n, G = case["batch"], case["dim"], case["L"], case["dstate"], case["groups"]
    R = case.get("rank", 0)
    pq = 2 * 4 * n * R * (1 if case.get("shared") else d) if R else 0
    per_ch = 4 * (d * n + 2 * d) + pq
    rows, bc = s * b * d * L, s * b * 2 * G * n * L
    if kind in ("prefill", "pq_prefill"):
        return {"bytes": 4 * rows + bc + per_ch + 4 * b * d * n, "flops": b * d * L * (n * (7 + 4 * R) + 8)}
    return {"bytes": 8 * rows + 2 * bc + 2 * per_ch, "flops": b * d * L * (n * (24 + 14 * R) + 24)}


# Four times the distance from float64 that these paths show. 16-bit results round to half an ulp
# (2-norm 1.7e-3 in bf16, 2.1e-4 in fp16), and dz, which reads the rounded pre-gate output, to
# 2.4e-3 / 3e-4; float32 results stay near 1e-6, at cancelling elements 1e-5. In the block the
# roundings of the layer's own 16-bit activations and GEMM results travel on: 5.7e-3 / 7e-4, up to
# 0.1 / 8e-3 of the root mean square for single elements.
_SCAN_TOL = {"bf16": {"rel": 1e-2, "max": 3.2e-2}, "fp16": {"rel": 1.2e-3, "max": 4e-3},
             "fp32": {"rel": 1e-5, "max": 1e-4}}
_BLOCK_TOL = {"bf16": {"rel": 2.4e-2, "max": 0.4}, "fp16": {"rel": 3e-3, "max": 5e-2}}


def tolerance(case):
    return dict((_BLOCK_TOL if case["kind"] == "block" else _SCAN_TOL)[case["dtype"]])


# ---- the same in 64 bits -------------------------------------------------------------------------


def _exact_scan(t, dout=None):
    """selective_scan_fn(delta_softplus=True) in float64, one time step after another, and, with
    dout, the gradients of its inputs by the reverse recurrence."""
    f = {k: v.detach().double() for k, v in t.items()}
    u, z, A, D = f["u"], f["z"], f["A"], f["D"]
    b, d, L = u.shape
    raw = f["delta"] + f["delta_bias"][None, :, None]
    dt = torch.nn.functional.softplus(raw)
    four = f["B"].dim() == 4
    B4, C4 = (f[k] if four else f[k][:, None] for k in ("B", "C"))
    G, n = B4.shape[1], B4.shape[2]

    def bc(v, i):      # (b, G, n, L) -> (b, d, n) of step i
        return v[..., i].repeat_interleave(d // G, dim=1) if G > 1 else v[..., i]

    P = Q = None
    if "P" in f:
        P = f["P"] if f["P"].dim() == 3 else f["P"].expand(d, -1, -1)
        Q = (f["Q"] if f["Q"].dim() == 3 else f["Q"].expand(d, -1, -1)).transpose(1, 2)
        ranks = range(P.shape[2])
    dts, us = dt.permute(2, 0, 1).contiguous(), u.permute(2, 0, 1).contiguous()
    h = torch.zeros(b, d, n, dtype=torch.float64, device=u.device)
    hs = torch.empty(L + 1, b, d, n, dtype=torch.float64, device=u.device) if dout is not None else None
    y = torch.empty(L, b, d, dtype=torch.float64, device=u.device)
    if hs is not None:
        hs[0] = 0
    for i in range(L):
        dti = dts[i][..., None]
        new = torch.exp(dti * A) * h
        new.addcmul_((dts[i] * us[i])[..., None], bc(B4, i))
        if P is not None:
            for k in ranks:
                q = (Q[..., k] * h).sum(-1, keepdim=True)
                new.addcmul_(dti * q, P[..., k])
        h = new
        if hs is not None:
            hs[i + 1] = h
        torch.sum(h * bc(C4, i), -1, out=y[i])
    pre = y.permute(1, 2, 0) + D[None, :, None] * u
    sg = torch.sigmoid(z)
    out = pre * z * sg
    if dout is None:
        return {"out": out, "last_state": h}
    go = dout.double()
    g = go * z * sg
    gs = g.permute(2, 0, 1).contiguous()
    lam = torch.zeros_like(h)
    dA = torch.zeros_like(A)
    dBg, dCg = torch.empty(L, b, G, n, dtype=torch.float64, device=u.device), torch.empty(
        L, b, G, n, dtype=torch.float64, device=u.device)
    du = torch.empty_like(y)
    ddt = torch.empty_like(y)
    if P is not None:
        dP, dQ = torch.zeros_like(P), torch.zeros_like(Q)
    for i in range(L - 1, -1, -1):
        dti, ui, gi = dts[i][..., None], us[i][..., None], gs[i][..., None]
        hp, Bi = hs[i], bc(B4, i)
        lam = lam + bc(C4, i) * gi
        ah = torch.exp(dti * A)
        nxt = ah * lam
        ah = ah * hp
        dCg[i] = (gi * hs[i + 1]).view(b, G, d // G, n).sum(2)
        ld = lam * dti
        dBg[i] = (ld * ui).view(b, G, d // G, n).sum(2)
        lb = (lam * Bi).sum(-1)
        du[i] = dts[i] * lb
        dA += (ld * ah).sum(0)
        acc = us[i] * lb + (lam * A * ah).sum(-1)
        if P is not None:
            for k in ranks:
                q = (Q[..., k] * hp).sum(-1, keepdim=True)
                pl = (P[..., k] * lam).sum(-1, keepdim=True)
                acc += (pl * q)[..., 0]
                dP[..., k] += (ld * q).sum(0)
                dQ[..., k] += (dti * pl * hp).sum(0)
                nxt.addcmul_(dti * pl, Q[..., k])
        ddt[i] = acc
        lam = nxt
    du = du.permute(1, 2, 0) + D[None, :, None] * g
    ddelta = ddt.permute(1, 2, 0) * torch.sigmoid(raw)
    dB, dC = dBg.permute(1, 2, 3, 0), dCg.permute(1, 2, 3, 0)
    res = {"out": out, "du": du, "ddelta": ddelta, "dA": dA, "dB": dB if four else dB[:, 0],
           "dC": dC if four else dC[:, 0], "dD": (g * u).sum((0, 2)),
           "dz": go * pre * sg * (1 + z * (1 - sg)), "ddelta_bias": ddelta.sum((0, 2))}
    if P is not None:
        dQ = dQ.transpose(1, 2)
        res["dP"] = dP.sum(0) if f["P"].dim() == 2 else dP
        res["dQ"] = dQ.sum(0) if f["Q"].dim() == 2 else dQ
    return res


def _exact_decode(t):
    f = {k: v.double() for k, v in t.items()}
    cs = torch.cat([f["conv_state"][..., 1:], f["x"][..., None]], -1)
    xc = torch.nn.functional.silu((cs * f["w"]).sum(-1) + f["wb"])
    x = xc.to(t["x"].dtype).double()                 # the layer's own activation type
    dt = torch.nn.functional.softplus(f["dt"] + f["dt_bias"])
    st = torch.exp(dt[..., None] * f["A"]) * f["state"] + (dt * x)[..., None] * f["B"][:, None]
    y = (st * f["C"][:, None]).sum(-1) + f["D"] * x
    return {"conv_state": cs, "state": st, "x": xc, "y": y * torch.nn.functional.silu(f["z"])}


def _exact_block(t, train):
    f = {k: v.detach().double() for k, v in t.items()}
    b, dd, L = f["xz"].shape
    d, n, R = dd // 2, f["A"].shape[1], f["dt_proj"].shape[1]
    x, z = f["xz"][:, :d], f["xz"][:, d:]
    w, xp = f["conv_w"][:, 0], torch.nn.functional.pad(x, (3, 0))
    pre = sum(w[:, k, None] * xp[..., k:k + L] for k in range(4)) + f["conv_b"][:, None]
    sp = torch.sigmoid(pre)
    xc = pre * sp
    flat = xc.transpose(0, 1).reshape(d, b * L)
    xdbl = f["x_proj"] @ flat
    view = lambda m: m.reshape(m.shape[0], b, L).transpose(0, 1)  # noqa: E731
    s = dict(u=xc, delta=view(f["dt_proj"] @ xdbl[:R]), A=f["A"], B=view(xdbl[R:R + n]), C=view(xdbl[R + n:]),
             D=f["D"], z=z, delta_bias=f["delta_bias"])
    if not train:
        return {"y": _exact_scan(s)["out"].transpose(1, 2) @ f["out_proj"].t()}
    dout = f["dout"]
    dyz = (dout @ f["out_proj"]).transpose(1, 2)
    g = _exact_scan(s, dyz)
    oz = g["out"].transpose(1, 2)
    mat = lambda v: v.transpose(0, 1).reshape(v.shape[1], b * L)  # noqa: E731
    ddel = mat(g["ddelta"])
    dxdbl = torch.cat([f["dt_proj"].t() @ ddel, mat(g["dB"]), mat(g["dC"])])
    dxc = g["du"] + view(f["x_proj"].t() @ dxdbl)
    dpre = dxc * sp * (1 + pre * (1 - sp))
    dpp = torch.nn.functional.pad(dpre, (0, 3))
    dx = sum(w[:, k, None] * dpp[..., 3 - k:3 - k + L] for k in range(4))
    dw = torch.stack([(dpre * xp[..., k:k + L]).sum((0, 2)) for k in range(4)], -1)
    return {"y": oz @ f["out_proj"].t(), "dxz": torch.cat([dx, g["dz"]], 1), "dconv_w": dw[:, None],
            "dconv_b": dpre.sum((0, 2)), "dx_proj": dxdbl @ flat.t(), "ddt_proj": ddel @ xdbl[:R].t(),
            "dout_proj": dout.reshape(b * L, -1).t() @ oz.reshape(b * L, d), "dA": g["dA"], "dD": g["dD"],
            "ddelta_bias": g["ddelta_bias"]}


def exact(case, seed):
    t = _inputs(case, seed)
    with torch.no_grad():
        if case["kind"] == "decode":
            return _exact_decode(t)
        if case["kind"] == "block":
            return _exact_block(t, case["train"])
        return _exact_scan({k: v for k, v in t.items() if k != "dout"}, t.get("dout"))
