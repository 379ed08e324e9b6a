"""Gates that are not finite: the outputs before the first such token keep their values, in its tile too.

A NaN or an infinity makes a channel's cumsum useless from its token on, and the state with it; nothing of that may
reach an earlier token.  Tolerance: bf16 operands and output (1e-2 of the 2-norm).
"""

import pytest
import torch

import mamformer_amd as mh
from oracle import kda as okda
from tests.gpu_helpers import check, dev, host, say

BF = torch.bfloat16


# first, inner and last tokens of a tile, of the first, an inner and a ragged last one
@pytest.mark.gpu
@pytest.mark.parametrize("S,at", [(64, 63), (150, 0), (150, 31), (150, 32), (150, 64), (150, 100), (150, 149), (400, 200)])
@pytest.mark.parametrize("value", ["nan", "inf", "-inf"])
@pytest.mark.parametrize("strong", [False, True])
def test_earlier_tokens_keep_their_outputs(S, at, value, strong):
    B, H = 1, 2
    g = torch.Generator().manual_seed(S + at)
    q1, q2, k, v = ((torch.randn(B, H, S, 128, generator=g) * 128 ** -0.5).to(BF) for _ in range(4))
    lg = -(1.1 if strong else 0.02) * torch.rand(B, H, S, 128, generator=g)
    s0 = 0.1 * torch.randn(B, H, 128, 128, generator=g)
    f = lambda t: t.double().numpy()
    want, _ = okda.gated_recurrent(f(q1[:, :, :at]), f(q2[:, :, :at]), f(k[:, :, :at]), f(v[:, :, :at]), f(lg[:, :, :at]),
                                   0.8, initial_state=f(s0))
    lg[0, 1, at, 37] = float(value)
    say(f"gated scan with {value} at {at} of {S}, strong {strong}")
    plan = mh.plan_linear_attn_scan(dev(q1, BF), dev(q2, BF), dev(k, BF), dev(v, BF), g=dev(lg), lam=0.8,
                                    initial_state=dev(s0), return_final_state=True)
    for split in (True, False):
        if not split:
            plan._ws, plan._ws_bytes = None, 0
        plan()
        torch.cuda.synchronize()
        o = host(plan.o)
        if at:
            check("before", o[:, :, :at], want, 1e-2)
        if value == "nan":
            assert (o[0, 1, at:] != o[0, 1, at:]).all() and (o[0, 0] == o[0, 0]).all()
            s = host(plan.final_state)
            assert (s[0, 1, 37] != s[0, 1, 37]).all() and (s[0, 1, :37] == s[0, 1, :37]).all()
