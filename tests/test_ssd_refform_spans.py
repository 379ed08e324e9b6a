"""The reference-form backward of sequences whose workspace would pass 2 GiB, taken a span of the sequence, or some batch
rows, at a time: what it asks for, and its gradients against those of shorter calls that autograd chains through the
state (or of fewer rows), each of them taken whole.

Both form the same sums of fp32 terms in another order: 1e-4 of the 2-norm in fp32; dx, dB and dC in bf16 (2^-8 a
rounding) to 1e-2, and most of them bit for bit.
"""

import ctypes as ct
import random

import pytest
import torch

import mamformer_amd as mh
from mamformer_amd import _lib
from tests.gpu_helpers import say
from tests.test_abi import _good_ref, _rc

BF, F32 = torch.bfloat16, torch.float32
GIB = 1 << 30


def workspace(b, L, di, N):
    g = _lib.SsdRefBwdArgs()
    f = _good_ref()
    f.batch, f.seqlen, f.nheads, f.headdim, f.dstate = b, L, di // 16, 16, N
    f.x_stride_l = f.y_stride_l = f.dt_stride_l = di
    f.x_stride_b = f.y_stride_b = f.dt_stride_b = L * di
    f.B_stride_l = f.C_stride_l = N
    f.B_stride_b = f.C_stride_b = L * N
    g.fwd = f
    g.dy = g.dx = g.ddt = g.dA = g.dB = g.dC = ct.c_void_p(4096)
    n = ct.c_size_t()
    assert _rc("mh_ssd_ref_scan_bwd_workspace_bytes", ct.byref(g), ct.byref(n)) == 0
    return n.value


def test_workspace_stays_near_the_states():
    rng = random.Random(2)
    sizes = [(2, 4096, 2048, 128), (1, 16384, 4096, 128), (1, 1 << 20, 4096, 128), (4096, 64, 2048, 128), (3, 16, 65536, 256)]
    for _ in range(400):
        b = rng.choice([1, 1, 2, 3, 8, 100])
        sizes.append((b, int(2 ** rng.uniform(9 if b < 3 else 0, 20)), 16 * int(2 ** rng.uniform(0, 9)),
                      rng.choice([16, 32, 64, 128, 256])))
    for b, L, di, N in sizes:
        if b * di * L > 1 << 37:
            continue
        states = 4 * b * -(-L // 16) * di * N
        n = workspace(b, L, di, N)
        # (and what alignment, or a row more than a third of 3 or 4 rows, adds)
        assert n <= max(2 * GIB, states // 8 * 9) + 4096, (b, L, di, N)
        assert n >= (states if b < 3 else states // 4)
    # two rows of the 1b preset: whole, 2.5 times the states
    assert 1.3e9 < workspace(2, 4096, 2048, 128) < 1.5e9


def leaves(seed, b, L, di, N, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    t = {"x": r(b, L, di).to(dtype), "dt": r(b, L, di) - 3.0, "A": torch.log(torch.linspace(0.5, 8.0, N, device="cuda")),
         "B": r(b, L, N).to(dtype), "C": r(b, L, N).to(dtype), "D": 1 + 0.1 * r(di), "h0": 0.1 * r(b, di, N),
         "bias": 0.1 * r(di)}
    w = r(b, L, di).to(dtype), r(b, L, N).to(dtype), r(b, di, N)
    return {k: v.requires_grad_() for k, v in t.items()}, w


def grads(t, outs, ws):
    torch.autograd.backward(outs, ws)
    torch.cuda.synchronize()
    got = {k: v.grad for k, v in t.items()}
    for v in t.values():
        v.grad = None
    return got


def scan(t, rows=slice(None), tok=slice(None), h0=None):
    return mh.selective_scan_reference(t["x"][rows, tok], t["dt"][rows, tok], t["A"], t["B"][rows, tok], t["C"][rows, tok],
                                       t["D"], True, True, initial_state=t["h0"][rows] if h0 is None else h0,
                                       dt_bias=t["bias"], dt_softplus=True)


def compare(got, want, dtype):
    for k in got:
        a, b = got[k].double(), want[k].double()
        e = float((a - b).norm() / b.norm())
        say(f"d{k}: {e:.2e}, {float((a != b).double().mean()):.1e} of the values differ")
        assert torch.isfinite(got[k]).all() and e <= (1e-2 if dtype == BF and k in "xBC" else 1e-4), k


# two spans and a ragged last block; a dozen spans, states of one 16-token block; rows that stay side by side
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,b,L,di,N,parts", [(BF, 1, 16400, 2048, 128, 2), (F32, 1, 33003, 1024, 256, 4),
                                                  (BF, 2, 65999, 2048, 16, 2), (BF, 1, 50001, 3008, 64, 4)])
def test_spans(dtype, b, L, di, N, parts):
    t, ws = leaves(L, b, L, di, N, dtype)
    step = -(-L // parts)
    say(f"ref-form spans {dtype} b{b} L{L} d_inner{di} N{N}: {workspace(b, L, di, N) / GIB:.2f} GiB")
    assert workspace(b, step, di, N) > 1.5 * 4 * b * (step // 16) * di * N, "the parts are meant to be taken whole"
    assert workspace(b, L, di, N) < 2.5 * 4 * b * (L // 16) * di * N, "the call is meant to be taken in spans"
    got = grads(t, scan(t), ws)
    ys, hss, h = [], [], None
    for i in range(0, L, step):
        y, hs, h = scan(t, tok=slice(i, i + step), h0=h)
        ys.append(y)
        hss.append(hs)
    compare(got, grads(t, (torch.cat(ys, 1), torch.cat(hss, 1), h), ws), dtype)


@pytest.mark.gpu
def test_rows():
    b, L, di, N = 2101, 31, 512, 128
    t, ws = leaves(5, b, L, di, N, BF)
    say(f"ref-form rows: {workspace(b, L, di, N) / GIB:.2f} GiB")
    assert workspace(b, L, di, N) < 2.5 * 4 * b * 2 * di * N and workspace(b // 3, L, di, N) > 2.5 * 4 * (b // 3) * 2 * di * N
    got = grads(t, scan(t), ws)
    outs = [scan(t, rows=slice(i, i + b // 3)) for i in range(0, b, b // 3)]
    want = grads(t, [torch.cat(o) for o in zip(*outs)], ws)
    compare(got, want, BF)
    for k in ("x", "dt", "B", "C", "h0"):
        assert torch.equal(got[k], want[k]), k
