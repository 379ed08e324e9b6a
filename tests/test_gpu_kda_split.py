"""KDA scans whose sequence is split into segments that walk side by side (few heads), against the unsplit walk of
the same kernels and the float64 oracle.

Split and unsplit differ in the order of the fp32 state sums and, gated, in one bf16 rounding of each segment's
k e^{G_end - G}: both are held to 4e-3 of each other (two bf16 roundings, 2^-8 each) and to 1e-2 of the oracle.
"""

import ctypes as ct

import pytest
import torch

import mamformer_amd as mh
from mamformer_amd import _lib
from oracle import kda as okda
from oracle import kda_bwd as obwd
from tests.gpu_helpers import check, check_per_head, dev, host, say

BF = torch.bfloat16


def inputs(B, H, S, seed, gate=1.0):
    g = torch.Generator().manual_seed(seed)
    mk = lambda s: (torch.randn(B, H, S, 128, generator=g) * s / 128 ** 0.5).to(BF)
    q1, q2, k, v = mk(4.0), mk(4.0), mk(4.0), mk(1.0)
    lg = torch.nn.functional.logsigmoid(torch.randn(B, H, S, 128, generator=g)) * gate / 16.0
    return q1, q2, k, v, lg, 0.1 * torch.randn(B, H, 128, 128, generator=g), 1.0 + torch.rand(B, H, 128, generator=g)


def both_walks(plan):
    """The plan's outputs with its workspace (split) and without (each sequence walked at once)."""
    assert plan._ws is not None, "these sizes are meant to split"
    names = [n for n in ("o", "o2", "final_state", "final_z") if getattr(plan, n) is not None]
    plan()
    split = {n: getattr(plan, n).clone() for n in names}
    plan._ws, plan._ws_bytes = None, 0
    plan()
    torch.cuda.synchronize()
    return split, {n: getattr(plan, n) for n in names}


# chunks: 4 (smallest split), a ragged last chunk of 1 token, of 63, a short last segment, 16 segments
@pytest.mark.gpu
@pytest.mark.parametrize("B,H,S", [(1, 3, 256), (1, 2, 321), (2, 3, 447), (1, 8, 1000), (1, 1, 2049)])
@pytest.mark.parametrize("kd,pair", [(128, False), (64, True)])
def test_split_reference_scan(B, H, S, kd, pair):
    q1, q2, k, v, _, s0, z0 = inputs(B, H, S, S + H)
    s0[:, :, kd:], z0[:, :, kd:] = 0, 0
    lam = torch.linspace(0.1, 0.9, H)
    say(f"split ref B={B} H={H} S={S} kd={kd} pair={pair}")
    plan = mh.plan_linear_attn_scan(*(dev(t, BF) for t in (q1, q2, k, v)), mode="reference", kernel_dim=kd, pair=pair,
                                    lam=dev(lam), initial_state=dev(s0), initial_z=dev(z0), return_final_state=True)
    split, whole = both_walks(plan)
    for n in split:
        check(f"split vs unsplit {n}", split[n], host(whole[n]), 4e-3)
    f = lambda t: t.double().numpy()
    r1, r2, rs, rz = okda.ref_scan_pair(f(q1), f(q2), f(k), f(v), kd, initial_state=f(s0)[:, :, :kd],
                                        initial_z=f(z0)[:, :, :kd])
    if pair:
        check("o1", split["o"], r1, 1e-2)
        check("o2", split["o2"], r2, 1e-2)
    else:
        lm = f(lam)[None, :, None, None]
        check_per_head("o", split["o"], (r1 - lm * r2) / (1 - lm + 1e-8), 1e-2)
    check("S", split["final_state"][:, :, :kd], rs, 1e-2)
    check("z", split["final_z"][:, :, :kd], rz, 1e-2)


# gate: the benchmark's, none, and one whose in-chunk decay passes e^-50 in many channels (factorisation windows)
@pytest.mark.gpu
@pytest.mark.parametrize("B,H,S,gate", [(1, 3, 256, 1.0), (2, 2, 383, 0.0), (1, 8, 1000, 1.0), (1, 2, 449, 40.0)])
def test_split_gated_scan(B, H, S, gate):
    q1, q2, k, v, lg, s0, _ = inputs(B, H, S, S, gate)
    say(f"split gated B={B} H={H} S={S} gate={gate}")
    plan = mh.plan_linear_attn_scan(*(dev(t, BF) for t in (q1, q2, k, v)), g=None if gate == 0.0 else dev(lg), lam=0.8,
                                    initial_state=dev(s0), return_final_state=True)
    split, whole = both_walks(plan)
    for n in split:
        check(f"split vs unsplit {n}", split[n], host(whole[n]), 4e-3)
    f = lambda t: t.double().numpy()
    o, s = okda.gated_recurrent(f(q1), f(q2), f(k), f(v), f(lg), 0.8, initial_state=f(s0))
    check("o", split["o"], o, 1e-2)
    check("S", split["final_state"], s, 1e-2)


# the query gradient's walk in 2 segments (few chunks), a ragged last chunk, and as many as the workspace takes
@pytest.mark.gpu
@pytest.mark.parametrize("B,H,S,kd", [(1, 2, 320, 128), (1, 3, 833, 100), (2, 1, 1000, 128)])
def test_split_backward(B, H, S, kd):
    q1, q2, k, v, _, s0, z0 = inputs(B, H, S, 3 * S + H)
    s0[:, :, kd:], z0[:, :, kd:] = 0, 0
    g = torch.Generator().manual_seed(S)
    d1, d2 = ((torch.randn(B, H, S, 128, generator=g) / 128 ** 0.5).to(BF) for _ in range(2))
    say(f"split bwd B={B} H={H} S={S} kd={kd}")
    t = lambda x: dev(x, BF)
    run = lambda: mh.linear_attn_scan_bwd(t(q1), t(q2), t(k), t(v), kernel_dim=kd, do1=t(d1), do2=t(d2), pair=True,
                                          initial_state=dev(s0), initial_z=dev(z0))
    r, again = run(), run()
    torch.cuda.synchronize()
    f = lambda x: x.double().numpy()
    ref = obwd.ref_scan_pair_backward(f(q1), f(q2), f(k), f(v), kd, f(d1), f(d2), initial_state=f(s0)[:, :, :kd],
                                      initial_z=f(z0)[:, :, :kd])
    for n in ("dq1", "dq2", "dk", "dv"):
        check(n, r[n], ref[n], 1e-2)
        assert torch.equal(r[n], again[n]), n
    check("dS0", r["d_initial_state"][:, :, :kd], ref["dS0"], 1e-2)
    check("dz0", r["d_initial_z"][:, :, :kd], ref["dz0"], 1e-2)


def _args(B, H, S):
    a = _lib.KdaArgs()
    a.batch, a.nheads, a.seqlen, a.dk, a.dv = B, H, S, 128, 128
    a.dtype, a.lam = _lib.MH_BF16, 0.8
    a.q1 = a.q2 = a.k = a.v = a.o = ct.c_void_p(4096)
    return a


def test_workspace_of_a_split_scan():
    n = ct.c_size_t(7)
    for B, H, S, splits in ((4, 32, 8192, False), (1, 16, 64, False), (1, 16, 1500, True), (1, 16, 0, False)):
        a = _args(B, H, S)
        assert _lib.lib().mh_kda_workspace_bytes(ct.byref(a), ct.byref(n)) == 0
        assert (n.value > 0) == splits and n.value % (B * H * (128 * 128 + 128) * 4) == 0
    a = _args(1, 16, 1500)
    a.dtype = _lib.MH_F32                              # the fp32 kernels walk each sequence at once
    assert _lib.lib().mh_kda_workspace_bytes(ct.byref(a), ct.byref(n)) == 0 and n.value == 0
    a = _args(1, 16, 1500)
    assert _lib.lib().mh_kda_chunk_scan_fwd_ws(ct.byref(a), 0, 8192, 64, None) == -7
    a.v = None
    assert _lib.lib().mh_kda_workspace_bytes(ct.byref(a), ct.byref(n)) == -1
