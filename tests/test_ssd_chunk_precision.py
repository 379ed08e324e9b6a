"""What the prefill's choice of chunk may cost in precision.

A bf16 chunk's state is rounded to bf16 (and, beyond 8 chunks, the state entering it once more), so more chunks mean
more roundings: cut from 256 tokens to 192, the error of y grew by 4% and that of the final state by 18% at steps near
1e-3, where states live for hundreds of tokens.  bf16 therefore takes the chunk of one workgroup per CU and no other;
fp32 rounds no state and may take a shorter one, at no larger error.
"""

import random

import pytest
import torch

import mamformer_amd as mh
from oracle import ssd as ref
from tests.gpu_helpers import dev, host, rel_l2, say
from tests.test_ssd_chunk_rule import one_round

BF, F32 = torch.bfloat16, torch.float32


def test_bf16_chunk_is_one_round():
    rng = random.Random(5)
    for _ in range(500):
        H = rng.choice([1, 3, 8, 24, 32, 48, 64, 128])
        b, L, N = rng.choice([1, 1, 2, 3, 7, 32]), int(2 ** rng.uniform(0, 18)), rng.choice([64, 128])
        G = rng.choice([g for g in (1, 2, 8) if H % g == 0])
        assert mh.ssd_chunk_len(b, L, H, 64, N, G, BF) == one_round(b, L, H, N, G, False), (b, L, H, N, G)


# bf16: 8 chunks of 256 (9 to 11 of 192: over the state pass), 6 of 256; fp32: chunks of 64 to 192 tokens
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,b,L,H,N,G", [(BF, 1, 2000, 8, 128, 1), (BF, 1, 1500, 16, 64, 1), (BF, 1, 1000, 8, 128, 2),
                                             (F32, 1, 1000, 32, 128, 1), (F32, 1, 2000, 16, 64, 2)])
@pytest.mark.parametrize("step", [1e-3, 1e-2])
def test_error_against_one_round(dtype, b, L, H, N, G, step):
    g = torch.Generator().manual_seed(L + N)
    x, B, C = (torch.randn(*s, generator=g).to(dtype) for s in ((b, L, H * 64), (b, L, G, N), (b, L, G, N)))
    dt = step * (0.5 + torch.rand(b, L, H, generator=g))
    A = -torch.exp(torch.rand(H, generator=g) * 2.77)
    f = lambda t: t.double().numpy()
    want = ref.ssd_chunked(f(x.view(b, L, H, 64)), f(dt), f(A), f(B), f(C), None, chunk_size=64)
    one = one_round(b, L, H, N, G, dtype == F32)
    say(f"chunk precision {dtype} b{b} L{L} H{H} N{N} G{G} dt {step}: {mh.ssd_chunk_len(b, L, H, 64, N, G, dtype)}, "
        f"one round {one}")
    err = []
    for chunk in (None, one):
        y, h = mh.selective_scan(dev(x, dtype), dev(dt), dev(A), dev(B, dtype), dev(C, dtype), None,
                                 return_final_state=True, chunk_size=chunk)
        err.append([rel_l2(host(y).reshape(want[0].shape), want[0]), rel_l2(host(h).reshape(want[1].shape), want[1])])
    say(f"error of y and h: {err[0]}, one round {err[1]}")
    # bf16: the same chunk, the same bits; fp32 sums in another order scatter by a few percent of 1e-6
    slack = 1.0 if dtype == BF else 1.1
    assert err[0][0] <= slack * err[1][0] and err[0][1] <= slack * err[1][1]
