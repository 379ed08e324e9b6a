"""Layer-level counterparts of the reference's scan call sites.

``Mamba2Layer`` mirrors ``Mamba2Block`` (R/mamformer/layers/mamba2.py:153-364) around the
SSD scan: in_proj -> causal depthwise conv1d -> SiLU -> dt/B/C projections -> scan (full
prefill, or the one-token recurrent step when a cache holds an SSM state) -> SiLU(z) gate
-> out_proj, with the reference's cache dict ``{"conv_state", "ssm_state"}``.  The conv,
SiLU, scan, z-gate and decode step run the HIP kernels of ``mamformer_amd.ops`` (conv and
SiLU fused; the gate applied by the scan / step kernels as y is stored); the projections are
plain library GEMMs, except that one bf16 token of up to 64 sequences runs the whole layer in its own
kernels (``Mamba2Layer._step``).

Recorded deviation (per-head SSD convention): the reference parameterises dt per channel
(``dt_proj: d_inner -> d_inner``) and A per state (``A_log (d_state,)``), which is a
Mamba-1-style diagonal decay that is not MFMA-factorable.  Here ``dt_proj`` ends in
``nheads`` outputs, ``A_log``, ``D`` and ``dt_bias`` are per head, and B/C have ``ngroups``
groups; dt = softplus(dt_proj(x) + dt_bias) inside the kernel.

``kda_linear_attention`` mirrors the recurrent-state handling of
``LinearDiffAttention.forward`` (R/mamformer/layers/kda_diff.py:286-338) on already
projected, rotated and GQA-expanded q1, q2, k, v (B, H, S, D).
"""

from __future__ import annotations

import math
from typing import Optional

import torch
import torch.nn as nn
from torch.autograd import forward_ad as _forward_ad

from . import ops

__all__ = ["Mamba2Layer", "kda_linear_attention"]


class Mamba2Layer(nn.Module):
    """Head-structured Mamba-2 layer; forward/cache semantics of ``Mamba2Block.forward`` (mamba2.py:249-364)."""

    def __init__(self, d_model: int, d_state: int = 128, d_conv: int = 4, expand: int = 1, headdim: int = 64,
                 ngroups: int = 1, dt_rank: Optional[int] = None, bias: bool = False, device=None, dtype=None):
        super().__init__()
        fk = {"device": device, "dtype": dtype}
        self.d_model = d_model
        self.d_inner = d_model * expand
        if self.d_inner % headdim:
            raise ValueError("Mamba2Layer: d_model * expand must be a multiple of headdim")
        self.headdim = headdim
        self.nheads = self.d_inner // headdim
        if self.nheads % ngroups:
            raise ValueError("Mamba2Layer: nheads must be a multiple of ngroups")
        self.ngroups = ngroups
        self.d_state = d_state
        self.d_conv = d_conv
        self.dt_rank = dt_rank if dt_rank is not None else math.ceil(d_model / 32)       # mamba2.py:191
        self.in_proj = nn.Linear(d_model, 2 * self.d_inner, bias=bias, **fk)
        self.conv_weight = nn.Parameter(torch.empty(self.d_inner, 1, d_conv, **fk))      # nn.Conv1d depthwise layout
        self.conv_bias = nn.Parameter(torch.zeros(self.d_inner, **fk)) if bias else None
        self.dt_proj = nn.Sequential(nn.Linear(self.d_inner, self.dt_rank, bias=bias, **fk),
                                     nn.Linear(self.dt_rank, self.nheads, bias=bias, **fk))
        self.B_proj = nn.Linear(self.d_inner, ngroups * d_state, bias=bias, **fk)
        self.C_proj = nn.Linear(self.d_inner, ngroups * d_state, bias=bias, **fk)
        self.A_log = nn.Parameter(torch.log(torch.linspace(1.0, 16.0, self.nheads, device=device)))
        self.dt_bias = nn.Parameter(torch.zeros(self.nheads, device=device))
        self.D = nn.Parameter(torch.ones(self.nheads, device=device))
        self.out_proj = nn.Linear(self.d_inner, d_model, bias=bias, **fk)
        self._init_weights()

    def _init_weights(self):
        """Initialisation of mamba2.py:229-247 (normal, std 0.02; dt projection std 0.001)."""
        nn.init.normal_(self.in_proj.weight, std=0.02)
        nn.init.normal_(self.out_proj.weight, std=0.02)
        for layer in self.dt_proj:
            nn.init.normal_(layer.weight, std=0.001)
        nn.init.normal_(self.B_proj.weight, std=0.02)
        nn.init.normal_(self.C_proj.weight, std=0.02)
        nn.init.normal_(self.conv_weight, std=0.02)

    def forward(self, u: torch.Tensor, use_cache: bool = False, cache: Optional[dict] = None,
                return_h_states: bool = False):
        """u (b, L, d_model) -> (out, cache) or (out, cache, h_states), as mamba2.py:249-364.

        Path choice of mamba2.py:285-334: an incremental one-token step (only the last token's SSM
        output, :296 / :435-438) when ``use_cache`` and ``cache["ssm_state"]`` is set; otherwise the full
        chunked scan.  The cache is ``{"conv_state": last d_conv-1 raw x rows, "ssm_state": (b, d_inner, N)
        fp32}`` (:343-364).
        """
        if use_cache and cache is not None and not return_h_states:
            step = self._step(u, cache)
            if step is not None:
                return step
        b, L, _ = u.shape
        x, z = self.in_proj(u).chunk(2, dim=-1)                 # mamba2.py:272-273
        raw_x = x
        conv_state = cache.get("conv_state") if (use_cache and cache is not None) else None
        x_act = ops.causal_conv1d(x, self.conv_weight, self.conv_bias, conv_state, silu=True)   # :279-283
        incremental = use_cache and cache is not None and cache.get("ssm_state") is not None    # :289
        dt = self.dt_proj(x_act)                                 # (b, L, H); softplus(+ dt_bias) in the kernel
        Bm = self.B_proj(x_act).view(b, L, self.ngroups, self.d_state)
        Cm = self.C_proj(x_act).view(b, L, self.ngroups, self.d_state)
        # A_log is clamped to [-5, 5] on the prefill path only, as the reference does (clamp in the scan,
        # mamba2.py:87; none in the decode step, :441-443)
        A_log = self.A_log.float()
        A = -torch.exp(A_log if incremental else A_log.clamp(-5.0, 5.0))
        D = self.D.float()
        h_states = None
        # the z-gate y * silu(z) (:337-338) is applied by the kernels as y is stored
        if incremental:
            y, final = ops.recurrent_step(x_act, dt, Bm, Cm, cache["ssm_state"], A, D,
                                          dt_bias=self.dt_bias, dt_softplus=True, z=z)
        else:
            res = ops.selective_scan(x_act, dt, A, Bm, Cm, D, return_h_states=return_h_states,
                                     return_final_state=use_cache, dt_bias=self.dt_bias, dt_softplus=True, z=z)
            res = res if isinstance(res, tuple) else (res,)
            y = res[0]
            h_states = res[1] if return_h_states else None
            final = res[-1] if use_cache else None
        out = self.out_proj(y)
        new_cache = None
        if use_cache:
            k = self.d_conv - 1
            conv_x = raw_x[:, -k:] if raw_x.shape[1] >= self.d_conv else raw_x   # :355
            if cache is not None and "conv_state" in cache:
                conv_x = torch.cat([cache["conv_state"], conv_x], dim=1)[:, -k:]
            new_cache = {"conv_state": conv_x, "ssm_state": final}
        if return_h_states:
            return out, new_cache, h_states
        return out, new_cache

    def _step(self, u, cache):
        """One token from the cache by ``mh_mamba2_layer_step`` (four launches; the composition below takes about
        twenty): (out, new cache), or None where the call is not that kernel's -- more than one token or 64 sequences,
        another dtype or layout, gradients wanted, or projections that are more than plain ``nn.Linear`` calls (hooks,
        parametrisations, autocast, tracing, function or dispatch modes) -- and the general path runs."""
        h0, cs = cache.get("ssm_state"), cache.get("conv_state")
        if not (type(u) is type(h0) is type(cs) is torch.Tensor and u.dtype is cs.dtype is torch.bfloat16
                and h0.dtype is torch.float32 and u.is_cuda and u.dim() == 3 and cs.dim() == 3):
            return None
        b, L, D = u.shape
        di, N, K = self.d_inner, self.d_state, self.d_conv
        if L != 1 or not 1 <= b <= 64 or D != self.d_model or D % 32 or di % 32 or N not in (8, 16, 32, 64, 128, 256) \
                or not 2 <= K <= 8 or not _plain_calls():
            return None
        S = cs.shape[1]
        if not 1 <= S < K or cs.shape[0] != b or cs.shape[2] != di or cs.stride(2) != 1 \
                or h0.numel() != b * di * N or not h0.is_contiguous() or u.stride(2) != 1 or u.stride(0) % 8:
            return None
        par = self._step_parameters()
        if par is None:
            return None
        weights, biases, cb, cw, *f32 = par
        r = weights[1].shape[0]
        G = self.ngroups
        if [t.shape for t in weights] != [(2 * di, D), (r, di), (self.nheads, r), (G * N, di), (G * N, di), (D, di)] \
                or cw.shape != (di, 1, K) or cb is not None and cb.shape != (di,) \
                or any(t.shape != (self.nheads,) for t in f32):
            return None
        w = []
        for t, bias in zip(weights, biases):
            if bias is not None and bias.shape != t.shape[:1]:
                return None
            w += (t, bias)
        bf16, dev = torch.bfloat16, u.device
        track = torch.is_grad_enabled()
        for t in (u, h0, cs, *w, cw, cb, *f32):
            if t is not None and (t.device != dev or not t.is_contiguous() and t is not u and t is not cs
                                  or track and t.requires_grad):
                return None
        if any(t is not None and t.dtype is not bf16 for t in (*w, cw, cb)) or any(t.dtype is not torch.float32
                                                                                   for t in f32):
            return None
        p = [None if t is None else t.data_ptr() for t in (u, h0, *w, cw, cb, *f32, cs)]
        if (p[0] | p[1] | p[2] | p[4] | p[8] | p[10] | p[12]) % 16:
            return None
        out = torch.empty((b, 1, D), device=dev, dtype=bf16)
        conv = torch.empty((b, min(S + 1, K - 1), di), device=dev, dtype=bf16)
        state = torch.empty((b, di, N), device=dev, dtype=torch.float32)
        ops.mamba2_layer_step(
            b, D, self.nheads, self.headdim, N, G, r, K, p[0], u.stride(0), p[2], p[3], p[14], p[15], *p[4:14],
            *p[16:19], p[19], S, cs.stride(0), cs.stride(1), p[1], state.data_ptr(), conv.data_ptr(), out.data_ptr(),
            device=dev)
        return out, {"conv_state": conv, "ssm_state": state}

    def _step_parameters(self):
        """The parameters that ``mh_mamba2_layer_step`` reads -- weights and biases of the six projections, conv_bias,
        conv_weight, A_log, dt_bias, D -- or None where one is not a plain ``nn.Parameter`` in its place (parametrised,
        deleted, a buffer or tensor instead) or a projection is not a plain, unhooked ``nn.Linear``: what reading the
        attribute or calling the module gives is then for the general path to find out."""
        mods, par = self._modules, self._parameters
        dtp = mods.get("dt_proj")
        if type(dtp) is not nn.Sequential or len(dtp._modules) != 2 or not _unhooked(dtp):
            return None
        weights, biases = [], []
        for m in (mods.get("in_proj"), *dtp._modules.values(), mods.get("B_proj"), mods.get("C_proj"),
                  mods.get("out_proj")):
            if type(m) is not nn.Linear or not _unhooked(m) or "bias" not in m._parameters:
                return None
            weights.append(m._parameters.get("weight"))
            biases.append(m._parameters["bias"])
        own = [par.get("conv_weight"), par.get("A_log"), par.get("dt_bias"), par.get("D")]
        cb = self.conv_bias
        for t in (*weights, *own):
            if type(t) is not nn.Parameter:
                return None
        for t in (*biases, cb):
            if t is not None and type(t) is not nn.Parameter:
                return None
        return weights, biases, cb, *own


def _plain_calls():
    """Whether a call runs eagerly as written: no autocast, tracing, functorch transform, forward-mode level, function
    or dispatch mode, and no hooks on every module."""
    from torch.nn.modules import module as m
    return not (torch.is_autocast_enabled() or torch.jit.is_tracing() or torch.compiler.is_compiling()
                or torch._C._functorch.peek_interpreter_stack() is not None or _forward_ad._current_level >= 0
                or torch._C._len_torch_function_stack() or torch._C._len_torch_dispatch_stack()
                or m._global_forward_hooks or m._global_forward_pre_hooks or m._global_backward_hooks
                or m._global_backward_pre_hooks)


def _unhooked(m):
    return not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                or "forward" in m.__dict__)


def kda_linear_attention(q1, q2, k, v, lambda_raw, kernel_dim, use_cache=False, cache=None):
    """Recurrent-state semantics of ``LinearDiffAttention.forward`` (R/mamformer/layers/kda_diff.py:286-338).

    q1, q2, k, v (B, H, S, D) after projection, RoPE and GQA expansion; lambda_raw (H,); kernel_dim K.
    * seq_len == 1 with ``use_cache``: one recurrent step from the cached (S, z) (:301-308, :564-605).
    * otherwise the normalised chunked scan from a zero state -- a cached state is *not* used for the
      outputs of a multi-token forward (:309-325, reference quirk, kept).
    * with ``use_cache`` the new cache is S = S_prev + phi(K)^T V, z = z_prev + sum_t phi(k_t) (:327-338),
      S (B, H, K, D) and z (B, H, K, 1) in float32.
    Returns (attn_output (B, H, S, D), new_cache or None).
    """
    Bb, H, S, Dh = q1.shape
    K = min(int(kernel_dim), Dh)
    if not use_cache:
        return ops.linear_attention_scan(q1, q2, k, v, K, lambda_raw), None
    S_prev = z_prev = None
    if cache is not None and cache.get("attn_type") == "linear":
        S_prev = cache["S"].to(torch.float32)
        z_prev = cache["z"].to(torch.float32)
    if S == 1:
        if S_prev is None:
            S_prev = torch.zeros((Bb, H, K, Dh), device=q1.device, dtype=torch.float32)
            z_prev = torch.zeros((Bb, H, K, 1), device=q1.device, dtype=torch.float32)
        # one step (dk = K) from the cache into new tensors, as the reference returns: the state has K rows, so
        # only the first K channels of q and k enter
        args = (q1[..., :K], q2[..., :K], k[..., :K], v)
        if _forward_ad._current_level >= 0 or torch.is_grad_enabled() and (S_prev.requires_grad
                                                                           or z_prev.requires_grad):
            # a cache that autograd tracks: its identity gradient goes through the copies that the step updates
            St = S_prev.clone(memory_format=torch.contiguous_format)
            zt = z_prev.clone(memory_format=torch.contiguous_format)
            out = ops.linear_attn_step(St, zt, *args, lam=lambda_raw, kernel_dim=K, apply_phi=True, _lam_raw=True)
        else:
            St = torch.empty(S_prev.shape, device=S_prev.device, dtype=torch.float32)
            zt = torch.empty(z_prev.shape, device=z_prev.device, dtype=torch.float32)
            out = ops.linear_attn_step(ops._step_input(S_prev), ops._step_input(z_prev), *args, lam=lambda_raw,
                                       kernel_dim=K, apply_phi=True, _out=(St, zt), _lam_raw=True)
        out = out.reshape(Bb, H, 1, Dh)
        return out, {"S": St, "z": zt, "attn_type": "linear"}
    out, S_new, z_new = ops.linear_attn_scan(q1, q2, k, v, mode="reference", kernel_dim=K, lam=lambda_raw,
                                             return_final_state=True, _lam_raw=True)
    S_new, z_new = S_new[:, :, :K], z_new[:, :, :K, None]
    if S_prev is not None:
        S_new, z_new = S_prev + S_new, z_prev + z_new
    return out, {"S": S_new.contiguous(), "z": z_new.contiguous(), "attn_type": "linear"}
