"""The SSD backward's head blocks: a call over all heads against calls over parts of them, whose workgroups take other
numbers of heads.

Everything per head (dx, ddt, dA, dD, d_dt_bias, d h0) does not depend on the block and is equal bit for bit; dB and dC
are sums over the heads, added in another order and rounded to the I/O type per part: the parts' sum carries one more
rounding each (2^-9 of a part for bf16, 2^-24 for fp32).
"""

import pytest
import torch

import mamformer_amd as mh
from mamformer_amd import workloads as W
from tests.gpu_helpers import check, host, say

pytestmark = pytest.mark.gpu


# blocks of 1 head (few segments), 2 and 4 (more), 32 (enough segments for one round), and heads no block above 1 divides
@pytest.mark.parametrize("dtype,b,L,H,N,parts", [
    (torch.bfloat16, 1, 64, 32, 128, 4), (torch.bfloat16, 1, 1000, 32, 128, 2), (torch.bfloat16, 2, 2000, 64, 64, 8),
    (torch.bfloat16, 2, 4096, 64, 128, 2), (torch.bfloat16, 2, 130, 7, 64, 7), (torch.float32, 1, 65, 16, 128, 2),
    (torch.float32, 1, 1000, 32, 64, 4),
])
def test_backward_by_head_parts(dtype, b, L, H, N, parts):
    say(f"bwd head parts {dtype} b{b} L{L} H{H} N{N} parts={parts}")
    inp = W.ssd_inputs(W.SSDConfig("p", b, L, H, 64, N, 1, 64, dtype, L, init_state=True), device="cuda")
    g = torch.Generator(device="cuda").manual_seed(L)
    dy = torch.randn(b, L, H, 64, device="cuda", generator=g).to(dtype)
    dfin = 0.1 * torch.randn(b, H, 64, N, device="cuda", generator=g)
    bias = 0.1 * torch.randn(H, device="cuda", generator=g)

    def run(a, z):
        return mh.selective_scan_bwd(dy[:, :, a:z].contiguous(), inp["x"][:, :, a:z].contiguous(),
                                     inp["dt"][:, :, a:z].contiguous(), inp["A"][a:z], inp["B"], inp["C"],
                                     inp["D"][a:z], d_final_state=dfin[:, a:z], dt_bias=bias[a:z], dt_softplus=True,
                                     initial_state=inp["initial_state"][:, a:z])
    whole, k = run(0, H), H // parts
    part = [run(i * k, (i + 1) * k) for i in range(parts)]
    torch.cuda.synchronize()
    for n, dim in (("dx", 2), ("ddt", 2), ("dA", 0), ("dD", 0), ("d_dt_bias", 0), ("d_initial_state", 1)):
        assert torch.equal(whole[n], torch.cat([p[n] for p in part], dim)), n
    for n in ("dB", "dC"):
        check(n, whole[n], host(sum(p[n].double() for p in part)), 4e-3 if dtype == torch.bfloat16 else 2e-6)
