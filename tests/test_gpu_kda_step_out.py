"""The KDA step into buffers other than its inputs, and the kernels' own lambda = min(sigmoid(lambda_raw), 0.99).

The step's arithmetic does not depend on where it writes, so its results equal the in-place step's bit for bit;
lambda in the kernel and in torch agree to fp32 rounding, which a differential output amplifies by at most
1 / (1 - 0.99): 1e-2 of it is bf16 rounding already, 1e-5 bounds it in fp32.
"""

import pytest
import torch

import mamformer_amd as mh
from mamformer_amd.layers import kda_linear_attention
from oracle import kda as okda
from tests.gpu_helpers import check_per_head, dev, host, say

pytestmark = pytest.mark.gpu
RAW = torch.tensor([-3.0, 0.0, 2.0, 4.59511985, 30.0])       # the fourth: sigmoid = 0.99


def inputs(B, D, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    H = RAW.numel()
    mk = lambda *s: torch.randn(*s, generator=g)
    q = [(mk(B, H, 1, D) / D ** 0.5).to(dtype) for _ in range(4)]
    return q, 2.0 * mk(B, H, D, D), 50.0 + 5.0 * torch.rand(B, H, D, 1, generator=g)


@pytest.mark.parametrize("B,D,K,dtype", [(1, 128, 128, torch.bfloat16), (3, 128, 64, torch.bfloat16),
                                         (2, 64, 64, torch.float32)])
@pytest.mark.parametrize("layout", ["contiguous", "transposed", "misaligned"])
def test_step_into_new_cache_equals_in_place(B, D, K, dtype, layout):
    (q1, q2, k, v), S, z = inputs(B, D, dtype, 10 * D + K)
    S, z = dev(S[:, :, :K]).contiguous(), dev(z[:, :, :K]).contiguous()
    q1, q2, k, v = (dev(t, dtype) for t in (q1, q2, k, v))
    say(f"kda step out B={B} D={D} K={K} {dtype} {layout}")
    St, zt = S.clone(), z.clone()
    want = mh.linear_attn_step(St, zt, q1[..., :K], q2[..., :K], k[..., :K], v, lam=mh.diff_lambda(dev(RAW)),
                               kernel_dim=K)
    if layout == "transposed":
        S_in = S.transpose(2, 3).contiguous().transpose(2, 3)
    elif layout == "misaligned":
        S_in = torch.cat([S.new_zeros(1), S.reshape(-1)])[1:].view(S.shape)
        assert S_in.data_ptr() % 16
    else:
        S_in = S
    before = S_in.clone()
    out, cache = kda_linear_attention(q1, q2, k, v, dev(RAW), K, use_cache=True,
                                      cache={"S": S_in, "z": z, "attn_type": "linear"})
    torch.cuda.synchronize()
    assert torch.equal(S_in, before)                          # the old cache is not touched
    assert torch.equal(cache["S"], St) and torch.equal(cache["z"], zt)
    tol = 1e-2 if dtype == torch.bfloat16 else 1e-5
    check_per_head("out", out, host(want), tol)
    # the reference's calling form, on features that the caller mapped (here rounded to the I/O type, once for both)
    f = [torch.as_tensor(okda.feature_map(t.double().cpu().numpy(), K)).to("cuda", dtype) for t in (q1, q2, k)]
    r = mh.linear_attention_recurrent(*f, v, S_in, z, dev(RAW))
    want = mh.linear_attn_step(S.clone(), z.clone(), *f, v, lam=mh.diff_lambda(dev(RAW)), apply_phi=False)
    check_per_head("recurrent", r, host(want), tol)
    assert torch.equal(S_in, before)


def test_lambda_raw_keeps_nan_and_rejects_a_float():
    (q1, q2, k, v), _, _ = inputs(1, 128, torch.bfloat16, 3)
    a = [dev(t, torch.bfloat16) for t in (q1, q2, k, v)]
    raw = RAW.clone()
    raw[1] = float("nan")
    o = mh.linear_attention_scan(*a, 128, dev(raw))
    assert torch.isnan(o[:, 1]).all() and torch.isfinite(o[:, [0, 2, 3, 4]]).all()
    with pytest.raises(TypeError):
        mh.linear_attention_scan(*a, 128, 0.5)


@pytest.mark.parametrize("trains", [True, False])
def test_lambda_raw_may_be_written_before_the_backward(trains):
    (q1, q2, k, v), _, _ = inputs(2, 128, torch.bfloat16, 4)
    a = [dev(t, torch.bfloat16).requires_grad_() for t in (q1, q2, k, v)]
    raw = dev(RAW).requires_grad_(trains)
    leaves = a + [raw] * trains
    want = torch.autograd.grad(mh.linear_attention_scan(*a, 128, raw).float().sum(), leaves)
    loss = mh.linear_attention_scan(*a, 128, raw).float().sum()
    with torch.no_grad():
        raw.add_(1.0)                                         # an optimizer's step on this parameter alone
    got = torch.autograd.grad(loss, leaves)
    assert all(torch.equal(x, y) for x, y in zip(got, want))
