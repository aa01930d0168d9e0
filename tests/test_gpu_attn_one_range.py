"""Decode attention over caches of up to 256 rows in one range (head_dim 64: one pass of 256 keys, or half of one) against a plain
computation in 64 bits: the result is rounded once from 32-bit sums, so it lies within half an ulp plus the sums' own error."""
import pytest
import torch

from tests.test_gpu_big_tiles import _rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Hk,Dh", [(1, 8, 8, 64), (5, 8, 2, 64), (3, 4, 4, 64), (8, 32, 8, 128)])
@pytest.mark.parametrize("S", [128, 129, 145, 256])
def test_one_range(B, H, Hk, Dh, S, dtype):
    from flashsvd_amd import hip_ops as ops
    assert ops.pick_nsplit(S, B, H, Dh) == 1
    q, k, v = _rand(B, H, Dh, seed=1, dtype=dtype), _rand(B, S, Hk, Dh, seed=2, dtype=dtype), _rand(B, S, Hk, Dh, seed=3, dtype=dtype)
    for n in sorted({0, 1, 31, 32, 127, 128, min(129, S), (128 + S) // 2, S - 1, S}):
        lens = torch.full((B,), n, dtype=torch.int32, device="cuda")
        lens[-1] = max(n - 1, 0)
        got = ops.attn_decode_densekv(q, k, v, lens)
        for b in range(B):
            m = int(lens[b])
            kk, vv = (t[b, :m].double().repeat_interleave(H // Hk, 1) for t in (k, v))
            w = torch.softmax((q[b].double()[None] * kk).sum(-1) / Dh ** 0.5, 0)                     # [m, H]
            want = (w[..., None] * vv).sum(0) if m else torch.zeros(H, Dh, dtype=torch.float64, device="cuda")
            bound = want.abs() * 2.0 ** (-8 if dtype == torch.bfloat16 else -11) + 2e-5 * (1 + vv.abs().amax() if m else 1)
            assert ((got[b].double() - want).abs() <= bound).all(), (b, m, (got[b].double() - want).abs().max())
