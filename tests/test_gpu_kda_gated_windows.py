"""Gated scan at the edges of its tiles and factorisation windows, against the float64 recurrence.

A tile is one window where G stays within 40 of its midpoint on every channel and is cut otherwise.  The gates here
change sign (growth as well as decay), come near half of that line, and drop in one token of one channel, so that one
tile of several is cut; test_gpu_kda_gated_cut.py has the line itself.  Tolerance: bf16 operands and output, as every bf16 scan (1e-2 of the 2-norm).
"""

import pytest
import torch

import mamformer_amd as mh
from oracle import kda as okda
from tests.gpu_helpers import check, dev, host, say

BF = torch.bfloat16


def gate(kind, B, H, S, g):
    n = torch.randn(B, H, S, 128, generator=g)
    if kind == "mild":
        return -0.05 * n.abs()
    if kind == "near":                       # a full tile's end near -50
        return -0.74 - 0.05 * n.abs()
    if kind == "signs":                      # rises and falls within a tile; the end is near 0, the middle is not
        t = torch.arange(S) % 64
        return torch.where(t < 32, 1.0, -1.0)[None, None, :, None] * 0.7 + 0.02 * n
    lg = -0.02 * n.abs()
    lg[:, :, (2 * S) // 3, 5] = -120.0       # "drop"
    if S > 3:
        lg[:, -1, S // 3, 77] = -60.0
    return lg


@pytest.mark.gpu
@pytest.mark.parametrize("S", [1, 63, 64, 65, 200, 257])
@pytest.mark.parametrize("kind", ["mild", "near", "signs", "drop"])
def test_gated_windows(S, kind):
    B, H = (2, 1) if S == 65 else (1, 3)
    g = torch.Generator().manual_seed(S)
    r = 128 ** -0.5
    q1, q2, k, v = ((torch.randn(B, H, S, 128, generator=g) * r).to(BF) for _ in range(4))
    s0, lg = torch.randn(B, H, 128, 128, generator=g) * 0.1, gate(kind, B, H, S, g)
    q2 = None if S == 63 else q2
    say(f"gated windows S={S} {kind}")
    plan = mh.plan_linear_attn_scan(dev(q1, BF), None if q2 is None else dev(q2, BF), dev(k, BF), dev(v, BF), g=dev(lg),
                                    lam=0.8, initial_state=dev(s0), return_final_state=True)
    plan()
    torch.cuda.synchronize()
    f = lambda t: t.double().numpy()
    o, s = okda.gated_recurrent(f(q1), f(torch.zeros_like(q1) if q2 is None else q2), f(k), f(v), f(lg), 0.8,
                                initial_state=f(s0))
    check("o", plan.o, o, 1e-2)
    check("S", plan.final_state, s, 1e-2)
    first = host(plan.o)
    plan()
    assert (host(plan.o) == first).all()
