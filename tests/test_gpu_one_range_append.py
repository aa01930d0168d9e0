"""Decode attention over caches of 129 to 256 rows with the new row appended by the call, against a plain computation in 64 bits: the result is
rounded once from 32-bit sums, so it lies within half an ulp plus the sums' own error.  Rotations are by powers of two, whose products are exact.
Rows past a sequence's length hold NaN: nothing of them may reach the result."""
import pytest
import torch

from tests.test_gpu_big_tiles import _rand

pytestmark = pytest.mark.gpu


def _rotated(x, c, s):
    """x [B, h, Dh] by rows c, s [B, Dh / 2] in 32 bits, rounded once."""
    a, b = x.float().chunk(2, -1)
    c, s = c.float()[:, None], s.float()[:, None]
    return torch.cat([a * c - b * s, a * s + b * c], -1).to(x.dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Hk,Dh", [(1, 8, 8, 64), (3, 8, 2, 64), (32, 32, 8, 64), (32, 32, 8, 128), (16, 32, 16, 128), (16, 32, 8, 128), (40, 32, 8, 64), (17, 16, 16, 128)])
@pytest.mark.parametrize("S", [129, 145, 256])
def test_appended_row(B, H, Hk, Dh, S, dtype):
    from flashsvd_amd import hip_ops as ops
    gen = torch.Generator().manual_seed(S)
    pick = torch.randint(0, 4, (S, Dh // 2), generator=gen).cuda()
    cos, sin = (torch.tensor(t, device="cuda", dtype=dtype)[pick] for t in ([1.0, 0.5, 0.0, -1.0], [0.0, 0.5, 1.0, -0.25]))
    q, kn, vn = _rand(B, H, Dh, seed=1, dtype=dtype), _rand(B, Hk, Dh, seed=4, dtype=dtype), _rand(B, Hk, Dh, seed=5, dtype=dtype)
    for n in sorted({0, 1, 126, 127, 128, S - 2, S - 1}):
        lens = torch.full((B,), n, dtype=torch.int32, device="cuda")
        if B > 1:
            lens[-1] = n // 2
        k, v = _rand(B, S, Hk, Dh, seed=2, dtype=dtype), _rand(B, S, Hk, Dh, seed=3, dtype=dtype)
        past = torch.arange(S, device="cuda")[None] >= lens[:, None]
        k[past], v[past] = float("nan"), float("nan")
        wk, wv, at = k.clone(), v.clone(), (torch.arange(B, device="cuda"), lens.long())
        wk[at], wv[at] = _rotated(kn, cos[lens.long()], sin[lens.long()]), vn
        got = ops.attn_decode_densekv(q, k, v, lens, k_new=kn, v_new=vn, cos=cos, sin=sin)
        assert torch.equal(k.view(torch.int16), wk.view(torch.int16)) and torch.equal(v.view(torch.int16), wv.view(torch.int16))
        qr = _rotated(q, cos[lens.long()], sin[lens.long()]).double()
        for b in range(B):
            m = int(lens[b]) + 1
            kk, vv = (t[b, :m].double().repeat_interleave(H // Hk, 1) for t in (wk, wv))
            w = torch.softmax((qr[b][None] * kk).sum(-1) / Dh ** 0.5, 0)                              # [m, H]
            want = (w[..., None] * vv).sum(0)
            bound = want.abs() * 2.0 ** (-8 if dtype == torch.bfloat16 else -11) + 2e-5 * (1 + vv.abs().amax())
            assert ((got[b].double() - want).abs() <= bound).all(), (n, b, m, (got[b].double() - want).abs().max())
