"""The chunk the SSD prefill picks: its range, the no-allocation entry point's scratch, and parity at its edges."""

import ctypes as ct
import random

import pytest
import torch

import mamformer_amd as mh
from mamformer_amd import _lib
from mamformer_amd import workloads as W
from oracle import ssd as ref
from tests.gpu_helpers import TOL, check, dev, host, say
from tests.test_abi import _good_ssd


def one_round(b, L, H, N, G, f32):
    """The chunk of one workgroup per CU, at least 256 tokens."""
    hg = 1 if f32 and N > 64 else 4
    while hg > 1 and (H // G) % hg:
        hg //= 2
    want = -(-L * b * (H // hg) // 256)
    return min(max(-(-want // 64) * 64, 256), 16384)


def workspace(b, L, H, N, G, dtype, chunk):
    a = _good_ssd()
    a.batch, a.seqlen, a.nheads, a.ngroups, a.dstate, a.dtype, a.chunk_len = b, L, H, G, N, dtype, chunk
    a.x_stride_l = a.y_stride_l = H * 64
    a.x_stride_b = a.y_stride_b = L * H * 64
    a.B_stride_l = a.C_stride_l = G * N
    a.B_stride_b = a.C_stride_b = L * G * N
    a.dt_stride_l, a.dt_stride_b = H, L * H
    n = ct.c_size_t()
    assert _lib.lib().mh_ssd_workspace_bytes(ct.byref(a), ct.byref(n)) == 0
    return n.value


def test_chunk_rule_range_and_scratch():
    rng = random.Random(1)
    sizes = [(1, 0, 8, 64, 1), (1, 1, 1, 64, 1), (1, 1 << 20, 128, 128, 8), (512, 4096, 64, 128, 1)]
    for _ in range(300):
        H = rng.choice([1, 3, 8, 24, 64, 128])
        sizes.append((rng.choice([1, 2, 7, 32]), int(2 ** rng.uniform(0, 18)), H, rng.choice([64, 128]),
                      rng.choice([g for g in (1, 2, 8) if H % g == 0])))
    for b, L, H, N, G in sizes:
        for code, dtype in ((_lib.MH_BF16, torch.bfloat16), (_lib.MH_F32, torch.float32)):
            c = mh.ssd_chunk_len(b, L, H, 64, N, G, dtype)
            assert c % 64 == 0 and (64 if dtype == torch.float32 else 256) <= c <= 16384
            one = one_round(b, L, H, N, G, dtype == torch.float32)
            if workspace(b, L, H, N, G, code, one) <= _lib.NOALLOC_SCRATCH_BYTES:
                assert workspace(b, L, H, N, G, code, 0) <= _lib.NOALLOC_SCRATCH_BYTES, (b, L, H, N, G, dtype)


# around the shortest chunks: one segment, a chunk and one token, two chunks, and more than 8 chunks (bf16, of 256 tokens:
# the states' pass; fp32: one-segment chunks)
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,b,L,H,N,G", [
    (torch.float32, 1, 63, 8, 128, 1), (torch.float32, 2, 129, 8, 64, 2), (torch.float32, 1, 1025, 32, 128, 1),
    (torch.float32, 3, 705, 64, 64, 8), (torch.bfloat16, 1, 193, 48, 64, 1), (torch.bfloat16, 2, 385, 16, 128, 2),
    (torch.bfloat16, 1, 1729, 8, 128, 1), (torch.bfloat16, 1, 257, 48, 64, 1), (torch.bfloat16, 2, 513, 16, 128, 2),
    (torch.bfloat16, 1, 2305, 8, 128, 1),
])
def test_chosen_chunk_vs_oracle(dtype, b, L, H, N, G):
    cfg = W.SSDConfig("c", b, L, H, 64, N, G, 256, dtype, L, init_state=True)
    inp = W.ssd_inputs(cfg)
    say(f"chunk rule {dtype} b{b} L{L} H{H} N{N} G{G}: {mh.ssd_chunk_len(b, L, H, 64, N, G, dtype)}")
    x, B, C = (dev(inp[k], dtype) for k in ("x", "B", "C"))
    y, fin = mh.selective_scan(x, dev(inp["dt"]), dev(inp["A"]), B, C, dev(inp["D"]), return_final_state=True,
                               initial_state=dev(inp["initial_state"]))
    f = lambda t: t.double().numpy()
    ry, rf = ref.ssd_chunked(host(x), f(inp["dt"]), f(inp["A"]), host(B), host(C), f(inp["D"]),
                             initial_state=f(inp["initial_state"]), chunk_size=64)
    check("y", y, ry, TOL[dtype])
    check("final", fin, rf, TOL[dtype])
