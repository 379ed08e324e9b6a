"""The SSD backward's heads in sequence within a workgroup: D per head against the same values per channel (both read
from a stage that the head before fetched), and no D at all, over one, an odd number and several heads per workgroup,
whole and ragged last segments.

dx, ddt, dA, dB and dC of the two D forms come from the same operations on the same values: equal bit for bit.  Per
channel, dD's 64 sums of a head add up to its one, in another order: 2^-24 sqrt(64 L) of the sum's scale at most in
practice, 1e-5 of the largest allowed.  Without D, dx lacks D dy: one bf16 rounding of each (2^-8 of their sum).
"""

import pytest
import torch

import mamformer_amd as mh
from mamformer_amd import workloads as W
from tests.gpu_helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,b,L,H,N,G", [
    (torch.bfloat16, 1, 1, 4, 128, 1), (torch.bfloat16, 2, 4096, 24, 128, 1), (torch.bfloat16, 1, 4097, 64, 128, 1),
    (torch.bfloat16, 2, 2050, 64, 64, 2), (torch.bfloat16, 1, 130, 3, 64, 1), (torch.float32, 1, 1000, 32, 64, 1),
], ids=lambda v: str(v).replace("torch.", ""))
def test_d_forms(dtype, b, L, H, N, G):
    say(f"bwd D forms {dtype} b{b} L{L} H{H} N{N} G{G}")
    inp = W.ssd_inputs(W.SSDConfig("p", b, L, H, 64, N, G, 64, dtype, L), device="cuda")
    g = torch.Generator(device="cuda").manual_seed(L)
    dy = torch.randn(b, L, H, 64, device="cuda", generator=g).to(dtype)
    D = inp["D"].reshape(H).contiguous()

    def run(d):
        return mh.selective_scan_bwd(dy, inp["x"], inp["dt"], inp["A"], inp["B"], inp["C"], d)
    head, chan, none = run(D), run(D[:, None].expand(H, 64).contiguous()), run(None)
    torch.cuda.synchronize()
    for n in ("dx", "ddt", "dA", "dB", "dC"):
        assert torch.equal(head[n], chan[n]), n
    for n in ("ddt", "dA", "dB", "dC"):
        assert torch.equal(head[n], none[n]), n
    s = chan["dD"].view(H, 64).double().sum(1)
    assert (s - head["dD"].double()).abs().max() <= 1e-5 * (b * L * 64) ** 0.5 + 1e-5 * s.abs().max()
    want = none["dx"].float() + D[:, None] * dy.float()
    eps = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -21
    assert ((head["dx"].float() - want).abs() <= eps * (none["dx"].float().abs() + want.abs()) + 1e-6).all()
