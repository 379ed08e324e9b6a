"""Gated scan whose tiles are cut into several factorisation windows, against the float64 recurrence: spreads on both
sides of the line (80 within a tile), windows of many tokens, of a few and of one; cut and whole tiles in turn; one
channel alone; split and unsplit walks.

Tolerance: bf16 operands and output, as every bf16 scan (1e-2 of the 2-norm); between the two walks 4e-3 (two bf16
roundings).
"""

import pytest
import torch

import mamformer_amd as mh
from oracle import kda as okda
from tests.gpu_helpers import check, dev, host, say

BF = torch.bfloat16


def gate(kind, B, H, S, g):
    n = torch.rand(B, H, S, 128, generator=g)
    t = torch.arange(S)
    if kind == "below":                      # a spread of 79 over a tile's 64 tokens
        return -1.25 - 0.01 * n
    if kind == "above":                      # 81: windows of 62 or 63 tokens and of one or two
        return -1.285 - 0.01 * n
    if kind == "two":                        # about 40 tokens a window
        return -2.0 - 0.1 * n
    if kind == "few":                        # two or three
        return -20.0 - n
    if kind == "one":                        # a window a token
        return -60.0 - n
    lg = -0.02 * n
    if kind == "channel":
        lg[..., 101] = -3.0
    elif kind == "turns":                    # every other tile
        lg = torch.where(((t // 64) % 2 == 1)[None, None, :, None], -2.0 * n, lg)
    elif kind == "last":                     # only the last tile, and only its last token's drop
        lg[:, :, -1, 3] = -300.0
    elif kind == "rise":                     # growth and decay of 30 within a tile: whole
        lg = torch.where((t % 64 < 32)[None, None, :, None], 0.95, -0.95) + lg
    elif kind == "peak":                     # growth of 50 and decay within eight tokens: between the midpoint's samples
        lg[..., 9] = torch.where(t % 64 == 4, 50.0, torch.where(t % 64 == 12, -50.0, 0.0))
    elif kind == "first":                    # a drop in each tile's first token: whole
        lg[..., 64] = torch.where(t % 64 == 0, -200.0, -0.1)
    elif kind == "head":                     # one head of several
        lg[:, 0] = -4.0 * n[:, 0]
    return lg


# one tile, ragged ones, three tiles, a split of several segments with a ragged last one
@pytest.mark.gpu
@pytest.mark.parametrize("S", [2, 64, 100, 192, 577])
@pytest.mark.parametrize("kind", ["below", "above", "two", "few", "one", "channel", "turns", "last", "rise", "peak", "first", "head"])
def test_windows_of_cut_tiles(S, kind):
    B, H = 1, 2
    g = torch.Generator().manual_seed(3 * S + len(kind))
    q1, q2, k, v = ((torch.randn(B, H, S, 128, generator=g) * 128 ** -0.5).to(BF) for _ in range(4))
    s0, lg = torch.randn(B, H, 128, 128, generator=g) * 0.1, gate(kind, B, H, S, g)
    q2 = None if S == 100 else q2
    say(f"gated cut tiles S={S} {kind}")
    plan = mh.plan_linear_attn_scan(dev(q1, BF), None if q2 is None else dev(q2, BF), dev(k, BF), dev(v, BF), g=dev(lg),
                                    lam=0.8, initial_state=dev(s0), return_final_state=True)
    f = lambda t: t.double().numpy()
    o, s = okda.gated_recurrent(f(q1), f(torch.zeros_like(q1) if q2 is None else q2), f(k), f(v), f(lg), 0.8,
                                initial_state=f(s0))
    plan()
    torch.cuda.synchronize()
    check("o", plan.o, o, 1e-2)
    check("S", plan.final_state, s, 1e-2)
    if plan._ws is not None:
        split = host(plan.o), host(plan.final_state)
        plan._ws, plan._ws_bytes = None, 0
        plan()
        check("o unsplit", plan.o, o, 1e-2)
        check("S unsplit", plan.final_state, s, 1e-2)
        check("o of both walks", plan.o, split[0], 4e-3)
        check("S of both walks", plan.final_state, split[1], 4e-3)
    first = host(plan.o)
    plan()
    assert (host(plan.o) == first).all()
