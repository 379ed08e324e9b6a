"""One token through ``Mamba2Layer`` by its own kernels, against the layer's general path (the same call with
``return_h_states``, which the step's kernels do not take) at the edges of its tiles, and the calls it leaves alone.

Both round the same intermediates to bf16 (2^-9 each) from fp32 sums in different orders, so a value may land one bf16
step apart anywhere along the chain: outputs agree to 1e-2 (relative L2), the raw rows of the new conv_state and the
fp32 state, one rounding down the chain, to 4e-3.
"""

import pytest
import torch

from mamformer_amd import layers, ops
from mamformer_amd.layers import Mamba2Layer
from tests.gpu_helpers import check, host, say

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def make(D=64, seed=0, **kw):
    torch.manual_seed(seed)
    lay = Mamba2Layer(D, device="cuda", dtype=BF, **kw)
    with torch.no_grad():
        for n, p in lay.named_parameters():
            if p.dim() >= 2:
                p.normal_(std=p.shape[-1] ** -0.5)
            elif n.endswith("bias") and n != "dt_bias":
                p.normal_(std=0.5)
        lay.dt_bias.fill_(-2.0)
    return lay


def cache_of(lay, b, rows):
    return {"conv_state": torch.randn(b, rows, lay.d_inner, device="cuda").to(BF),
            "ssm_state": 0.3 * torch.randn(b, lay.d_inner, lay.d_state, device="cuda")}


def taken(monkeypatch, lay, u, cache):
    calls = []
    orig = ops.mamba2_layer_step
    monkeypatch.setattr(ops, "mamba2_layer_step", lambda *a, **k: (calls.append(1), orig(*a, **k)))
    out = lay(u, use_cache=True, cache=cache)
    monkeypatch.setattr(ops, "mamba2_layer_step", orig)
    return out, bool(calls)


@pytest.mark.parametrize("b,D,rows,kw", [
    (1, 64, 3, {}), (16, 96, 3, {}), (17, 64, 2, {"bias": True}), (33, 64, 1, {"d_state": 64}),
    (64, 544, 3, {"d_state": 16, "dt_rank": 7}), (5, 512, 3, {"expand": 2, "ngroups": 4, "headdim": 32}),
    (3, 64, 1, {"d_conv": 2, "d_state": 256}), (2, 2048, 7, {"d_conv": 8, "bias": True}),
])
def test_step_matches_general_path(monkeypatch, b, D, rows, kw):
    if D % kw.get("headdim", 64):
        kw = dict(kw, headdim=32)
    lay = make(D, **kw)
    u, cache = torch.randn(b, 1, D, device="cuda").to(BF), cache_of(lay, b, rows)
    say(f"layer step b={b} D={D} rows={rows} {kw}")
    with torch.no_grad():
        want, wc, _ = lay(u, use_cache=True, cache=cache, return_h_states=True)
        (out, c), fast = taken(monkeypatch, lay, u, cache)
        assert fast
        # a conv_state that is a strided view, as the prefill leaves it, and a second step from the new cache
        wide = torch.randn(b, rows, 2 * lay.d_inner, device="cuda").to(BF)
        wide[..., :lay.d_inner] = cache["conv_state"]
        (out2, _), fast = taken(monkeypatch, lay, u, dict(cache, conv_state=wide[..., :lay.d_inner]))
        assert fast and torch.equal(out, out2)
        nxt = lay(u, use_cache=True, cache=c)[0]
        wnxt = lay(u, use_cache=True, cache=wc, return_h_states=True)[0]
    torch.cuda.synchronize()
    check("out", out, host(want), 1e-2)
    check("next out", nxt, host(wnxt), 1e-2)
    assert c["conv_state"].shape == wc["conv_state"].shape and c["ssm_state"].shape == wc["ssm_state"].shape
    check("conv_state", c["conv_state"], host(wc["conv_state"]), 4e-3)
    check("ssm_state", c["ssm_state"], host(wc["ssm_state"]), 4e-3)


def test_other_calls_take_the_general_path(monkeypatch):
    lay = make()
    u, cache = torch.randn(2, 1, 64, device="cuda").to(BF), cache_of(lay, 2, 3)
    seen = []
    with torch.no_grad():
        assert taken(monkeypatch, lay, u, cache)[1]
        h = lay.B_proj.register_forward_hook(lambda *a: seen.append(1))
        assert not taken(monkeypatch, lay, u, cache)[1] and seen
        h.remove()
        assert not taken(monkeypatch, lay, torch.cat([u, u], 1), cache)[1]              # two tokens
        assert not taken(monkeypatch, lay, u, dict(cache, ssm_state=cache["ssm_state"].transpose(1, 2)
                                                   .contiguous().transpose(1, 2)))[1]   # a strided state
        big = torch.randn(65, 1, 64, device="cuda").to(BF)
        assert not taken(monkeypatch, lay, big, cache_of(lay, 65, 3))[1]
        with torch.autocast("cuda", dtype=BF):
            assert not taken(monkeypatch, lay, u, cache)[1]
        with torch.autograd.forward_ad.dual_level():
            assert not taken(monkeypatch, lay, u, cache)[1]
    assert not taken(monkeypatch, lay, u, cache)[1]                                     # gradients wanted
    lay32 = Mamba2Layer(64, device="cuda")
    with torch.no_grad():
        assert not taken(monkeypatch, lay32, u.float(), {k: v.float() for k, v in cache.items()})[1]
    assert layers._plain_calls()
