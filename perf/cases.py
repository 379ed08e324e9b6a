"""The work that a program has this framework do, as cases that can be timed and compared.

Each kind of case is one call that a model makes through the public Python entry points, at the sizes of the
repository's own workloads (``mamformer_amd/workloads.py``), of the 1b preset (d_inner 2048 with expand 1, 4096 with
expand 2, state size 128, 16 attention heads of 128) and, in ``draw``, of the range around them:

===============  ======================================================================================
``ssd``          prefill of a prompt by the Mamba-2 scan: y and the state that decoding goes on from
``ssd_train``    forward and backward of the gated scan, as a training step of the layer runs it
``ssd_decode``   one token of every sequence in a decode batch, the state updated in place
``kda_gated``    prefill by the decay-gated linear-attention scan
``kda``          prefill of a prompt by the normalised linear-attention scan, with the cache for decoding
``kda_train``    forward and backward of the differential linear-attention scan
``kda_decode``   one token of every sequence from the linear-attention cache
``ref_train``    forward and backward of the scan with the reference's own parameters (a rate per state)
``layer_step``   one token through a whole ``Mamba2Layer`` from its cache
===============  ======================================================================================

``exact`` restates every kind in float64 torch from the equations alone.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import mamformer_amd as mh
from mamformer_amd import layers

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
_DEV = "cuda"


# ------------------------------------------------------------------------------------------------ the cases

def listed():
    return [
        # the 1b-shape prefill of the headline benchmark: two sequences of 4096 tokens, dt ready as fp32
        dict(name="prefill_1b", kind="ssd", dtype="bf16", b=2, L=4096, H=64, N=128, G=1, layer=False, h0=False),
        # one user's prompt of odd length at the 1b preset's width, called as Mamba2Layer calls it (raw dt of the
        # projection's type with bias and softplus, gate fused): latency and idle compute units count here
        dict(name="prefill_prompt", kind="ssd", dtype="bf16", b=1, L=333, H=32, N=128, G=1, layer=True, h0=False),
        # 128K tokens of context from a carried state, eight B / C groups: the largest call
        dict(name="prefill_128k", kind="ssd", dtype="bf16", b=1, L=131072, H=128, N=128, G=8, layer=False, h0=True),
        # the fp32 option, used for reference runs and verification at the 1b preset's width
        dict(name="prefill_fp32", kind="ssd", dtype="fp32", b=1, L=1000, H=32, N=128, G=1, layer=False, h0=False),
        # a training step of the scan at the 1b shape
        dict(name="train_1b", kind="ssd_train", dtype="bf16", b=2, L=4096, H=64, N=128, G=1),
        # a decode batch of 64 sequences: bound by the fp32 state's bytes
        dict(name="decode_b64", kind="ssd_decode", dtype="bf16", b=64, H=64, N=128, G=1),
        # the gated linear-attention benchmark: four sequences of 8192 tokens, 32 heads
        dict(name="kda_gated_8k", kind="kda_gated", dtype="bf16", b=4, L=8192, H=32),
        # one user's prompt through a linear-attention layer of the 1b preset's 16 heads, keeping the cache
        dict(name="kda_prompt", kind="kda", dtype="bf16", b=1, L=1500, H=16, K=128),
        # a training step of that layer
        dict(name="kda_train", kind="kda_train", dtype="bf16", b=2, L=2048, H=16, K=128),
        # a decode batch of 32 sequences through that layer
        dict(name="kda_decode_b32", kind="kda_decode", dtype="bf16", b=32, H=16, K=128),
        # a training step with a reference checkpoint's own parameters
        dict(name="ref_train", kind="ref_train", dtype="bf16", b=1, L=2048, D=2048, N=128),
        # one token of eight sequences through a whole layer of the 1b preset's width: the smallest call
        dict(name="layer_step_b8", kind="layer_step", dtype="bf16", b=8, D=2048, N=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the ranges around the listed ones: sizes log-uniform, most of them odd."""
    kind = rng.choice(["ssd", "ssd", "ssd", "ssd_train", "ssd_train", "ssd_decode", "kda_gated", "kda", "kda_train",
                       "kda_decode", "ref_train", "layer_step"])
    if kind in ("ssd", "ssd_train"):
        H = rng.choice([8, 16, 32, 48, 64, 128])
        c = dict(kind=kind, dtype="bf16", b=rng.choice([1, 1, 2, 3, 4]), H=H, N=rng.choice([64, 128, 128]),
                 G=rng.choice([1, 1, 2, 8]))
        top = 16384 if kind == "ssd" else 4096
        if kind == "ssd":
            c.update(dtype=rng.choice(["bf16", "bf16", "bf16", "fp32"]), layer=rng.random() < 0.5, h0=rng.random() < 0.3)
            top = top if c["dtype"] == "bf16" else 4096
        c["L"] = _log_int(rng, 24, min(top, (1 << 19) // (c["b"] * H)))
        return c
    if kind == "ssd_decode":
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "fp32"]), b=_log_int(rng, 1, 256),
                    H=rng.choice([16, 32, 64]), N=rng.choice([64, 128]), G=rng.choice([1, 1, 4]))
    if kind in ("kda_gated", "kda", "kda_train"):
        b, H = rng.choice([1, 1, 2, 4]), rng.choice([8, 16, 32])
        c = dict(kind=kind, dtype="bf16", b=b, H=H)
        if kind != "kda_gated":
            c["K"] = rng.choice([128, 128, 64])
        c["L"] = _log_int(rng, 50, min(8192, (1 << (20 if kind == "kda_gated" else 18)) // (b * H)))
        return c
    if kind == "kda_decode":
        return dict(kind=kind, dtype="bf16", b=_log_int(rng, 1, 128), H=rng.choice([8, 16, 32]),
                    K=rng.choice([128, 128, 64]))
    if kind == "ref_train":
        D = rng.choice([512, 1024, 2048])
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "fp32"]), b=rng.choice([1, 2]), D=D,
                    N=rng.choice([16, 64, 128]), L=_log_int(rng, 64, min(2048, (1 << 21) // D)))
    return dict(kind=kind, dtype="bf16", b=_log_int(rng, 1, 64), D=rng.choice([512, 1024, 2048]),
                N=rng.choice([64, 128]))


# ------------------------------------------------------------------------------------------------ inputs

class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device=_DEV).manual_seed(seed)

    def randn(self, *shape, scale=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device=_DEV) * scale).to(dtype)

    def rand(self, *shape):
        return torch.rand(*shape, generator=self.g, device=_DEV)


def _ssd_common(c, g, dt_shape):
    """Inputs of the per-head scan: the recipes of ``mamformer_amd.workloads`` (A = -exp(U(0, ln 16)), dt around
    softplus(-4.6))."""
    H = c["H"]
    return dict(A=-torch.exp(g.rand(H) * math.log(16.0)), D=1.0 + 0.1 * g.randn(H),
                dt_bias=torch.full((H,), -4.6, device=_DEV) + 0.1 * g.randn(H), dt=g.randn(*dt_shape))


def _layer_weights(c, g):
    """A ``Mamba2Layer`` with weights of a trained layer's size (every projection keeps its input's scale)."""
    layer = layers.Mamba2Layer(c["D"], d_state=c["N"], device=_DEV, dtype=_DTYPES[c["dtype"]])
    with torch.no_grad():
        for name, p in layer.named_parameters():
            if name == "conv_weight":
                p.copy_(g.randn(*p.shape, scale=0.5))
            elif p.dim() == 2:
                p.copy_(g.randn(*p.shape, scale=1.0 / math.sqrt(p.shape[1])))
            elif name == "A_log":
                p.copy_(g.rand(*p.shape) * math.log(16.0))
            elif name == "dt_bias":
                p.copy_(-4.6 + 0.1 * g.randn(*p.shape))
            elif name == "D":
                p.copy_(1.0 + 0.1 * g.randn(*p.shape))
    return layer


def prepare(case, seed):
    c, g, dt_, kind = case, _Gen(seed), _DTYPES[case["dtype"]], case["kind"]
    s = {"case": c}
    b = c["b"]
    if kind in ("ssd", "ssd_train"):
        L, H, N, G = c["L"], c["H"], c["N"], c["G"]
        s.update(_ssd_common(c, g, (b, L, H)))
        s.update(x=g.randn(b, L, H * 64, dtype=dt_), B=g.randn(b, L, G, N, dtype=dt_), C=g.randn(b, L, G, N, dtype=dt_))
        if kind == "ssd" and not c["layer"]:
            s["dt"] = F.softplus(s["dt"] - 4.6)
            s["h0"] = g.randn(b, H * 64, N, scale=0.1) if c["h0"] else None
        else:
            s["dt"] = s["dt"].to(dt_)
            s["z"] = g.randn(b, L, H * 64, dtype=dt_)
            s["h0"] = g.randn(b, H * 64, N, scale=0.1) if c.get("h0") else None
        if kind == "ssd_train":
            s["leaves"] = {k: s[k].requires_grad_() for k in ("x", "dt", "A", "B", "C", "D", "dt_bias", "z")}
            s["dy"] = g.randn(b, L, H * 64, dtype=dt_)
    elif kind == "ssd_decode":
        H, N, G = c["H"], c["N"], c["G"]
        s.update(_ssd_common(c, g, (b, H)))
        s.update(x=g.randn(b, H, 64, dtype=dt_), B=g.randn(b, G, N, dtype=dt_), C=g.randn(b, G, N, dtype=dt_),
                 state=g.randn(b, H, 64, N, scale=0.1))
    elif kind in ("kda_gated", "kda", "kda_train", "kda_decode"):
        H, L = c["H"], c.get("L", 1)
        r = 1.0 / math.sqrt(128)
        for k in ("q1", "q2", "k", "v"):
            s[k] = g.randn(b, H, L, 128, scale=r, dtype=dt_)
        s["lambda_raw"] = torch.linspace(-2.0, 3.0, H, device=_DEV) + 0.1 * g.randn(H)
        if kind == "kda_gated":
            s["g"] = F.logsigmoid(g.randn(b, H, L, 128)) / 16.0
        elif kind == "kda_train":
            s["leaves"] = {k: s[k].requires_grad_() for k in ("q1", "q2", "k", "v", "lambda_raw")}
            s["do"] = g.randn(b, H, L, 128, scale=r, dtype=dt_)
        elif kind == "kda_decode":
            # a cache after some hundred tokens: z near their count, S their values' sum
            s["cache"] = {"S": g.randn(b, H, c["K"], 128, scale=2.0),
                          "z": 500.0 + 20.0 * g.randn(b, H, c["K"], 1), "attn_type": "linear"}
    elif kind == "ref_train":
        L, D, N = c["L"], c["D"], c["N"]
        s.update(x=g.randn(b, L, D, dtype=dt_), dt=g.randn(b, L, D, dtype=dt_),
                 A=torch.log(torch.linspace(0.5, 8.0, N, device=_DEV)) + 0.05 * g.randn(N),
                 B=g.randn(b, L, N, dtype=dt_), C=g.randn(b, L, N, dtype=dt_), D=1.0 + 0.1 * g.randn(D),
                 dt_bias=torch.full((D,), -3.0, device=_DEV) + 0.1 * g.randn(D))
        s["leaves"] = {k: s[k].requires_grad_() for k in ("x", "dt", "A", "B", "C", "D", "dt_bias")}
        s["dy"] = g.randn(b, L, D, dtype=dt_)
    else:
        s["layer"] = _layer_weights(c, g)
        s["u"] = g.randn(b, 1, c["D"], dtype=dt_)
        s["cache"] = {"conv_state": g.randn(b, 3, c["D"], dtype=dt_), "ssm_state": g.randn(b, c["D"], c["N"], scale=0.1)}
    return s


# ------------------------------------------------------------------------------------------------ one pass

def run(state):
    s, c, kind = state, state["case"], state["case"]["kind"]
    if kind == "ssd":
        if c["layer"]:
            return mh.selective_scan(s["x"], s["dt"], s["A"], s["B"], s["C"], s["D"], return_final_state=True,
                                     dt_bias=s["dt_bias"], dt_softplus=True, z=s["z"], initial_state=s["h0"])
        return mh.selective_scan(s["x"], s["dt"], s["A"], s["B"], s["C"], s["D"], return_final_state=True,
                                 initial_state=s["h0"])
    if kind == "ssd_train":
        v = s["leaves"]
        y = mh.selective_scan(v["x"], v["dt"], v["A"], v["B"], v["C"], v["D"], dt_bias=v["dt_bias"], dt_softplus=True,
                              z=v["z"])
        return y, torch.autograd.grad(y, list(v.values()), s["dy"])
    if kind == "ssd_decode":
        y = mh.selective_state_update(s["state"], s["x"], s["dt"], s["A"], s["B"], s["C"], s["D"],
                                      dt_bias=s["dt_bias"], dt_softplus=True)
        return y, s["state"]
    if kind == "kda_gated":
        return mh.linear_attn_scan(s["q1"], s["q2"], s["k"], s["v"], g=s["g"], lam=0.8, return_final_state=True)
    if kind == "kda":
        out, cache = layers.kda_linear_attention(s["q1"], s["q2"], s["k"], s["v"], s["lambda_raw"], c["K"],
                                                 use_cache=True)
        return out, cache["S"], cache["z"]
    if kind == "kda_train":
        v = s["leaves"]
        y = mh.linear_attention_scan(v["q1"], v["q2"], v["k"], v["v"], c["K"], v["lambda_raw"])
        return y, torch.autograd.grad(y, list(v.values()), s["do"])
    if kind == "kda_decode":
        out, cache = layers.kda_linear_attention(s["q1"], s["q2"], s["k"], s["v"], s["lambda_raw"], c["K"],
                                                 use_cache=True, cache=s["cache"])
        return out, cache["S"], cache["z"]
    if kind == "ref_train":
        v = s["leaves"]
        y = mh.selective_scan_reference(v["x"], v["dt"], v["A"], v["B"], v["C"], v["D"], dt_bias=v["dt_bias"],
                                        dt_softplus=True)
        return y, torch.autograd.grad(y, list(v.values()), s["dy"])
    with torch.no_grad():
        out, cache = s["layer"](s["u"], use_cache=True, cache=s["cache"])
    return out, cache["conv_state"], cache["ssm_state"]


def work(case):
    """Bytes of the inputs and outputs, each once, and operations of the dense chunked form (256-token chunks for the
    scans over heads, 64-token ones for linear attention), or of the recurrence where there is no such form."""
    c, kind, b = case, case["kind"], case["b"]
    es = 2 if c["dtype"] == "bf16" else 4
    if kind in ("ssd", "ssd_train"):
        L, H, N, G, P = c["L"], c["H"], c["N"], c["G"], 64
        Q = min(L, 256)
        layer = kind == "ssd_train" or c["layer"]
        xb, bc, dtb, st = b * L * H * P * es, b * L * G * N * es, b * L * H * (es if layer else 4), b * H * P * N * 4
        fwd_b = xb * (3 if layer else 2) + 2 * bc + dtb
        fwd_f = b * L * (2 * Q * N * G + H * (2 * Q * P + 4 * N * P))
        if kind == "ssd":
            return {"bytes": fwd_b + st * (2 if c["h0"] else 1), "flops": fwd_f}
        q = min(L, 64)
        bwd_f = b * L * (2 * q * N * G + H * (4 * q * P + 4 * q * N + 10 * P * N))
        return {"bytes": fwd_b + xb * 3 + 2 * bc + dtb, "flops": fwd_f + bwd_f}
    if kind == "ssd_decode":
        H, N, G = c["H"], c["N"], c["G"]
        return {"bytes": 2 * b * H * 64 * N * 4 + 2 * b * H * 64 * es + 2 * b * G * N * es + b * H * 4,
                "flops": 6 * b * H * 64 * N}
    if kind in ("kda_gated", "kda", "kda_train"):
        n, q = b * c["H"] * c["L"], min(c["L"], 64)
        K = c.get("K", 128)
        if kind == "kda_gated":
            return {"bytes": n * (5 * 256 + 512) + b * c["H"] * 128 * 128 * 4, "flops": n * 4 * (64 * q + 64 * q + 128 * 128)}
        fwd = n * (2 * (2 * q * K + 2 * q * 128 + 2 * K * 128) + 2 * K * 128)
        if kind == "kda":
            return {"bytes": n * 5 * 256 + b * c["H"] * K * 129 * 4, "flops": fwd}
        return {"bytes": n * 10 * 256, "flops": 3 * fwd}
    if kind == "kda_decode":
        return {"bytes": b * c["H"] * (2 * c["K"] * 129 * 4 + 5 * 256), "flops": 6 * b * c["H"] * c["K"] * 128}
    if kind == "ref_train":
        n = b * c["L"] * c["D"]
        return {"bytes": n * 6 * es + 4 * b * c["L"] * c["N"] * es, "flops": 22 * n * c["N"]}
    D, N, r = c["D"], c["N"], math.ceil(c["D"] / 32)
    weights = 3 * D * D + 2 * D * N + D * r + r * (D // 64)
    return {"bytes": 2 * weights + 2 * b * D * N * 4 + b * D * (2 + 2 + 6 + 6) * 1.0, "flops": 2 * b * weights + 6 * b * D * N}


# about four times the largest error against float64 that the outputs of these calls show at the listed sizes: 3.1e-3
# for the scans with bf16 operands and their gradients, 3.4e-3 gated linear attention, 3.2e-3 its training step,
# 1.8e-3 where only inputs and outputs are bf16, 3.8e-3 through a layer's projections, 1.1e-6 in fp32
_REL = {"ssd": 1.2e-2, "ssd_train": 1.2e-2, "ssd_decode": 7e-3, "kda_gated": 1.4e-2, "kda": 7e-3, "kda_train": 1.3e-2,
        "kda_decode": 7e-3, "ref_train": 7e-3, "layer_step": 1.5e-2}


def tolerance(case):
    return {"rel": _REL[case["kind"]] if case["dtype"] == "bf16" else 5e-6}


# ------------------------------------------------------------------------------------------------ float64

def _f64(t):
    return None if t is None else t.detach().double()


def _ssd_piece(x, a, u, B, C, h):
    """The scan of one piece of whole 64-token blocks: x (b, L, H, P), a = A dt and u = dt (b, L, H), B and C
    (b, L, G, N), h (b, H, P, N) before it.  Returns the read-out of the state and the state after."""
    b, L, H, P = x.shape
    G, N, Q = B.shape[2], B.shape[3], 64
    k = L // Q
    cs = a.view(b, k, Q, H).cumsum(2)
    diff = cs[:, :, :, None] - cs[:, :, None]                                         # (b, k, t, s, H)
    causal = torch.ones(Q, Q, dtype=torch.bool, device=x.device).tril()[:, :, None]
    M = torch.exp(diff.masked_fill(~causal, -math.inf)).permute(0, 1, 4, 2, 3)        # (b, k, H, t, s)
    Bk, Ck = (t.view(b, k, Q, G, N).permute(0, 1, 3, 2, 4) for t in (B, C))           # (b, k, G, Q, N)
    CB = torch.matmul(Ck, Bk.transpose(-1, -2).contiguous())
    xu = (x * u[..., None]).view(b, k, Q, H, P).permute(0, 1, 3, 2, 4)                # (b, k, H, Q, P)
    y = torch.matmul(M * CB.repeat_interleave(H // G, dim=2), xu)
    ends = cs[:, :, -1]                                                               # (b, k, H)
    xw = xu * torch.exp(ends[:, :, None] - cs).permute(0, 1, 3, 2)[..., None]
    Bh, Ch = (t.repeat_interleave(H // G, dim=2) for t in (Bk, Ck))
    S = torch.matmul(xw.transpose(-1, -2).contiguous(), Bh)                           # (b, k, H, P, N)
    e = torch.exp(ends)
    hs = []
    for i in range(k):
        hs.append(h)
        h = h * e[:, i, :, None, None] + S[:, i]
    read = torch.matmul(Ch, torch.stack(hs, 1).transpose(-1, -2).contiguous())
    y = y + read * torch.exp(cs).permute(0, 1, 3, 2)[..., None]
    return y.permute(0, 1, 3, 2, 4).reshape(b, L, H, P), h


def _ssd_exact(x, dt, A, B, C, D, dt_bias=None, z=None, h0=None, piece=4096):
    b, L, H = dt.shape
    xs, dt = x.view(b, L, H, 64), dt if dt_bias is None else F.softplus(dt + dt_bias)
    h = torch.zeros(b, H, 64, B.shape[-1], dtype=x.dtype, device=x.device) if h0 is None else h0.view(b, H, 64, -1)
    ys = []
    for t in range(0, L, piece):
        n = min(piece, L - t)
        pad = -n % 64
        part = [F.pad(v[:, t:t + n], (0, 0) * (v.dim() - 2) + (0, pad)) for v in (xs, dt * A, dt, B, C)]
        y, h = _ssd_piece(*part, h)
        ys.append(y[:, :n])
    y = (torch.cat(ys, 1) + xs * D[:, None]).reshape(b, L, H * 64)
    return (y if z is None else y * F.silu(z)), h


def _phi(t, K):
    return F.elu(t[..., :K]) + 1.0


def _kda_exact(q1, q2, k, v, lam, K):
    """The normalised scan as masked attention, one (batch, head) after the other."""
    L = q1.shape[2]
    mask = torch.ones(L, L, dtype=torch.float64, device=q1.device).tril()
    outs = []
    for i in range(q1.shape[0]):
        for h in range(q1.shape[1]):
            pk = _phi(k[i, h], K).T
            o = []
            for q in (q1, q2):
                w = (_phi(q[i, h], K) @ pk) * mask
                o.append((w @ v[i, h]) / (w.sum(-1, keepdim=True) + 1e-8))
            outs.append((o[0] - lam[h] * o[1]) / (1.0 - lam[h] + 1e-8))
    return torch.stack(outs).view(v.shape)


def _lam(raw):
    return torch.clamp(torch.sigmoid(raw), max=0.99)


def _grads(y, leaves, gy):
    return [t.to(torch.float64) for t in torch.autograd.grad(y, leaves, gy)]


def _layer_exact(s, c):
    p = {k: _f64(v) for k, v in s["layer"].named_parameters()}
    u, conv, st = _f64(s["u"]), _f64(s["cache"]["conv_state"]), _f64(s["cache"]["ssm_state"])
    b, D, N, H = c["b"], c["D"], c["N"], c["D"] // 64
    x, z = (u[:, 0] @ p["in_proj.weight"].T).chunk(2, dim=-1)
    rows = torch.cat([conv, x[:, None]], 1)
    xa = F.silu((rows * p["conv_weight"][:, 0].T).sum(1))
    dt = F.softplus(xa @ p["dt_proj.0.weight"].T @ p["dt_proj.1.weight"].T + p["dt_bias"])
    Bm, Cm = xa @ p["B_proj.weight"].T, xa @ p["C_proj.weight"].T
    xh, h = xa.view(b, H, 64), st.view(b, H, 64, N)
    h = (h * torch.exp(-torch.exp(p["A_log"]) * dt)[:, :, None, None]
         + (xh * dt[..., None])[..., None] * Bm[:, None, None])
    y = (h * Cm[:, None, None]).sum(-1) + xh * p["D"][:, None]
    out = (y.reshape(b, D) * F.silu(z)) @ p["out_proj.weight"].T
    return out[:, None], rows[:, 1:], h.reshape(b, D, N)


def exact(case, seed):
    c, s, kind = case, prepare(case, seed), case["kind"]
    b = c["b"]
    if kind == "ssd":
        with torch.no_grad():
            lay = c["layer"]
            y, h = _ssd_exact(*(_f64(s[k]) for k in ("x", "dt", "A", "B", "C", "D")), _f64(s["dt_bias"]) if lay else None,
                              _f64(s["z"]) if lay else None, _f64(s["h0"]))
        return y, h.reshape(b, c["H"] * 64, c["N"])
    if kind == "ssd_train":
        v = [_f64(t).requires_grad_() for t in s["leaves"].values()]
        y, _ = _ssd_exact(*v)
        return y.detach(), _grads(y, v, _f64(s["dy"]))
    if kind == "ssd_decode":
        x, dt, A, B, C, D, bias, h = (_f64(s[k]) for k in ("x", "dt", "A", "B", "C", "D", "dt_bias", "state"))
        dt = F.softplus(dt + bias)
        r = c["H"] // c["G"]
        h = (h * torch.exp(A * dt)[..., None, None]
             + (x * dt[..., None])[..., None] * B.repeat_interleave(r, 1)[:, :, None])
        return (h * C.repeat_interleave(r, 1)[:, :, None]).sum(-1) + x * D[:, None], h
    if kind == "kda_gated":
        q, k, v, e = _f64(s["q1"]) - 0.8 * _f64(s["q2"]), _f64(s["k"]), _f64(s["v"]), torch.exp(_f64(s["g"]))
        S = torch.zeros(b, c["H"], 128, 128, dtype=torch.float64, device=_DEV)
        o = torch.empty_like(v)
        for t in range(c["L"]):
            S = S * e[:, :, t, :, None] + k[:, :, t, :, None] * v[:, :, t, None]
            o[:, :, t] = (q[:, :, t, :, None] * S).sum(2)
        return o, S
    if kind == "kda":
        q1, q2, k, v, lr = (_f64(s[n]) for n in ("q1", "q2", "k", "v", "lambda_raw"))
        pk = _phi(k, c["K"])
        return (_kda_exact(q1, q2, k, v, _lam(lr), c["K"]), torch.matmul(pk.transpose(-1, -2).contiguous(), v),
                pk.sum(2)[..., None])
    if kind == "kda_train":
        v = [_f64(t).requires_grad_() for t in s["leaves"].values()]
        y = _kda_exact(*v[:4], _lam(v[4]), c["K"])
        return y.detach(), _grads(y, v, _f64(s["do"]))
    if kind == "kda_decode":
        K = c["K"]
        q1, q2, k, v = (_f64(s[n])[:, :, 0] for n in ("q1", "q2", "k", "v"))
        pk, lam = _phi(k, K), _lam(_f64(s["lambda_raw"]))[None, :, None]
        S = _f64(s["cache"]["S"]) + pk[..., None] * v[:, :, None]
        z = _f64(s["cache"]["z"]) + pk[..., None]
        o = [(_phi(q, K)[..., None] * S).sum(2) / ((_phi(q, K) * z[..., 0]).sum(-1, keepdim=True) + 1e-8) for q in (q1, q2)]
        return ((o[0] - lam * o[1]) / (1.0 - lam + 1e-8))[:, :, None], S, z
    if kind == "ref_train":
        x, dt, A, B, C, D, bias = v = [_f64(t).requires_grad_() for t in s["leaves"].values()]
        d, rate = F.softplus(dt + bias), -torch.exp(A.clamp(-5.0, 5.0))
        h, ys = torch.zeros(b, c["D"], c["N"], dtype=torch.float64, device=_DEV), []
        for dt_t, ux, B_t, C_t in zip(d.unbind(1), (d * x).unbind(1), B.unbind(1), C.unbind(1)):
            h = h * torch.exp(dt_t[..., None] * rate) + ux[..., None] * B_t[:, None]
            ys.append((h * C_t[:, None]).sum(-1))
        y = torch.stack(ys, 1) + x * D
        return y.detach(), _grads(y, v, _f64(s["dy"]))
    with torch.no_grad():
        return _layer_exact(s, c)
