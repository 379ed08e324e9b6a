"""GPU parity of the reference-form backward where its pieces of 16 tokens, its blocks of 64 channels and its 8-element
rows end (csrc/ssd_refform.hip: rf_sweep_kernel, rf_grad_kernel), against autograd of the float64 recurrence
(tests/test_gpu_ssd_refform_bwd.py); with the h_states gradient given at an address aligned to its elements only; and
the log-rates' gradient at, inside and outside the clamp and for a NaN, against torch.

Tolerance: relative L2 <= 1e-4 (fp32 I/O) and <= 1e-2 (bf16 I/O: dx, dB and dC are stored with a rounding of at most
2^-8 each), as everywhere for this op.
"""

import pytest
import torch

import mamformer_amd as mh
from tests.gpu_helpers import check, say
from tests.test_gpu_ssd_refform_bwd import BF, F32, TOLS, make, ref_scan

pytestmark = pytest.mark.gpu


def offset_view(t):
    """The same values in a contiguous tensor that starts one element past an aligned address."""
    buf = torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)
    out = buf[1:].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.parametrize("dtype,b,L,di,N", [
    (F32, 1, 1, 16, 16), (F32, 2, 15, 80, 32), (F32, 1, 16, 64, 64), (F32, 1, 17, 144, 16), (F32, 2, 33, 16, 128),
    (F32, 1, 31, 80, 256), (BF, 2, 1, 64, 128), (BF, 1, 17, 80, 64), (BF, 1, 33, 144, 16), (BF, 1, 16, 16, 256),
], ids=lambda v: str(v).replace("torch.", ""))
def test_pieces_and_channel_blocks(dtype, b, L, di, N):
    inp, (wy, wh, wf) = make(3 * L + di + N, b, L, di, N, dtype)
    say(f"ref-form pieces {dtype} b{b} L{L} d_inner{di} N{N}")
    io = {"x": dtype, "B": dtype, "C": dtype}
    lv = {k: v.to(io.get(k, F32)).cuda().requires_grad_() for k, v in inp.items()}
    y, hs, fin = mh.selective_scan_reference(lv["x"], lv["dt"], lv["A_log"], lv["B"], lv["C"], lv["D"], True, True,
                                             initial_state=lv["h0"], dt_bias=lv["bias"], dt_softplus=True)
    wy, wh = wy.to(dtype), wh.to(dtype)                    # the gradients as the kernels get them
    torch.autograd.backward((y, hs, fin), (wy.cuda(), offset_view(wh.cuda()), wf.float().cuda()))
    torch.cuda.synchronize()
    r = {k: v.clone().requires_grad_() for k, v in inp.items()}
    want = ref_scan(r["x"], r["dt"], r["A_log"], r["B"], r["C"], r["D"], r["h0"], r["bias"], True, None)
    torch.autograd.backward(want, (wy.double(), wh.double(), wf.float().double()))
    for k in lv:
        check(f"d{k}", lv[k].grad.double().cpu(), r[k].grad.numpy(), TOLS[dtype])


def test_log_rates_at_the_clamp():
    inp, _ = make(5, 1, 20, 32, 16, F32, h0=False, bias=False, D=True)
    log = inp["A_log"].float()
    log[0], log[1], log[2], log[3] = -5.0, 5.0, -5.0000005, 5.5
    log[4] = float("nan")
    say("ref-form log-rates at the clamp")
    lv = {k: inp[k].float().cuda() for k in ("x", "dt", "B", "C", "D")}
    A = log.cuda().requires_grad_()
    y, fin = mh.selective_scan_reference(lv["x"], lv["dt"], A, lv["B"], lv["C"], lv["D"], False, True, dt_softplus=True)
    assert torch.isnan(y).all() and torch.isnan(fin[..., 4]).all() and torch.isfinite(fin[..., 5:]).all()
    fin[..., :4].sum().backward()
    g = A.grad.cpu()
    assert g[0] != 0 and g[1] != 0 and g[2] == 0 and g[3] == 0 and (g[5:] == 0).all()
    r = log.double().requires_grad_()
    rfin = ref_scan(inp["x"], inp["dt"], r, inp["B"], inp["C"], inp["D"], None, None, True, None)[2]
    rfin[..., :4].sum().backward()
    check("dA_log", g[:2].double(), r.grad[:2].numpy(), 1e-4)


def test_frozen_log_rates_may_be_written_before_the_backward():
    inp, (wy, _, _) = make(6, 1, 33, 64, 32, F32, h0=False, bias=False)
    say("ref-form frozen log-rates")
    grads = []
    for write in (False, True):
        x = inp["x"].float().cuda().requires_grad_()
        A = inp["A_log"].float().cuda()
        y = mh.selective_scan_reference(x, inp["dt"].float().cuda(), A, inp["B"].float().cuda(),
                                        inp["C"].float().cuda(), inp["D"].float().cuda(), dt_softplus=True)
        if write:
            A.zero_()
        y.backward(wy.float().cuda())
        grads.append(x.grad)
    assert torch.equal(*grads)
