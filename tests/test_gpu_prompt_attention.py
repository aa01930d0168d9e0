"""Prompt attention at the edges of its forms (one to three groups of waves, 64 or 128 query rows per workgroup): chunks of any
length behind cached tokens, grouped heads, padding masks that leave whole key tiles unseen, additive masks of the lowest
value, outputs off the 8-byte grid.  Reference in fp64; a result is one rounding of a sum whose weights carry about 16 bits:
half an ulp of the result plus 2^-14 of the largest value."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v, start, causal, pad=None, add=None):
    B, M, H, Dh = q.shape
    n = min(start + M, k.shape[1])
    G = H // k.shape[2]
    kk = k[:, :n].double().repeat_interleave(G, 2).permute(0, 2, 1, 3)
    vv = v[:, :n].double().repeat_interleave(G, 2).permute(0, 2, 1, 3)
    s = torch.matmul(q.double().permute(0, 2, 1, 3), kk.transpose(-1, -2).contiguous()) * Dh ** -0.5
    if add is not None:
        s = s + add[:, None, :, :n].double()
    ok = torch.ones(B, 1, M, n, dtype=torch.bool)
    if causal:
        ok &= torch.arange(n)[None] <= start + torch.arange(M)[:, None]
    if pad is not None:
        ok &= pad[:, None, None, :n].bool()
    s = s.masked_fill(~ok, -float("inf"))
    m = s.amax(-1, keepdim=True)
    e = torch.exp(s - torch.where(m == -float("inf"), torch.zeros_like(m), m))
    e = e / e.sum(-1, keepdim=True).clamp_min(1e-300)
    return torch.matmul(e, vv).permute(0, 2, 1, 3)


def _check(out, ref, vmax, dtype):
    err = (out.double().cpu() - ref).abs()
    bound = ref.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) + vmax * 2.0 ** -14
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,M,H,Hk,start", [(1, 1, 2, 2, 0), (1, 17, 4, 1, 300), (2, 63, 4, 4, 1), (2, 77, 8, 2, 1411), (1, 64, 4, 4, 128),
                                            (1, 65, 3, 3, 0), (1, 127, 2, 1, 191), (1, 128, 2, 2, 0), (2, 700, 16, 4, 0), (1, 1030, 32, 32, 7),
                                            (4, 390, 32, 8, 0)])
def test_chunks(dtype, B, M, H, Hk, start):
    from flashsvd_amd import hip_ops
    gen = torch.Generator().manual_seed(M)
    S = start + M + 3
    q, k, v = (torch.randn(B, *s, 128, generator=gen).to(dtype) for s in ((M, H), (S, Hk), (S, Hk)))
    out = hip_ops.attn_prefill(q.cuda(), k.cuda(), v.cuda(), q_pos0=torch.full((B,), start, dtype=torch.int32, device="cuda"), causal=True)
    rows = slice(0, M) if M < 256 else slice(M - 200, M)        # the CPU reference in parts
    heads = min(H, 4 * (H // Hk))
    ref = _reference(q[:, rows, :heads], k[:, :, :heads * Hk // H], v[:, :, :heads * Hk // H], start + (rows.start or 0), True)
    _check(out[:, rows, :heads], ref, float(v.abs().max()), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,M,H,Hk,start", [(1, 31, 2, 2, 0), (1, 32, 8, 2, 33), (3, 33, 4, 2, 62), (2, 95, 4, 4, 161), (1, 97, 4, 1, 1), (1, 256, 32, 8, 70),
                                            (8, 32, 32, 32, 225), (8, 40, 32, 8, 90), (1, 257, 32, 32, 0), (12, 30, 32, 8, 5), (13, 30, 32, 8, 500)])
def test_chunks_around_the_rules(dtype, B, M, H, Hk, start):
    """32 rows per workgroup up to 256 workgroups, 64 in groups up to 384, then without; fewer key tiles than groups, unequal shares of them."""
    test_chunks(dtype, B, M, H, Hk, start)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("M,H", [(77, 4), (200, 4), (512, 70)])
def test_padding_masks(M, H, causal):
    """Kept keys on the right, on the left, scattered, a single one, none: tiles without a masked key, with some, with only those."""
    from flashsvd_amd import hip_ops
    gen = torch.Generator().manual_seed(M)
    B = 5
    q, k, v = (torch.randn(B, M, H, 128, generator=gen).bfloat16() for _ in range(3))
    pad = torch.zeros(B, M, dtype=torch.uint8)
    pad[0, : M // 2 + 1] = 1
    pad[1, M - 70:] = 1
    pad[2] = (torch.rand(M, generator=gen) < 0.5).to(torch.uint8)
    pad[3, 3] = 1
    out = hip_ops.attn_prefill(q.cuda(), k.cuda(), v.cuda(), causal=causal, pad_mask=pad.cuda())
    n = min(H, 3)
    _check(out[:, :, :n], _reference(q[:, :, :n], k[:, :, :n], v[:, :, :n], 0, causal, pad=pad), float(v.float().abs().max()), torch.bfloat16)
    assert float(out[4].float().abs().max()) == 0.0
    # an output whose rows start off the 8-byte grid
    odd = torch.zeros(B, M, H, 129, dtype=torch.bfloat16, device="cuda")[..., 1:]
    hip_ops.attn_prefill(q.cuda(), k.cuda(), v.cuda(), causal=causal, pad_mask=pad.cuda(), out=odd)
    assert torch.equal(odd, out)


def test_additive_mask_of_the_lowest_value():
    """Rows whose every key carries the lowest finite value weigh their keys alike, rows of -inf give zero."""
    from flashsvd_amd import hip_ops
    gen = torch.Generator().manual_seed(5)
    B, M, H = 1, 90, 2
    q, k, v = (torch.randn(B, M, H, 128, generator=gen).bfloat16() for _ in range(3))
    add = torch.randn(B, M, M, generator=gen)
    add[:, 10] = torch.finfo(torch.float32).min
    add[:, 20] = -float("inf")
    add[:, 30, ::3] = -float("inf")
    out = hip_ops.attn_prefill(q.cuda(), k.cuda(), v.cuda(), causal=False, add_mask=add.cuda())
    ref = _reference(q, k, v, 0, False, add=add)
    ref[:, 10] = v.double().mean(1)
    _check(out, ref, float(v.float().abs().max()), torch.bfloat16)
    assert float(out[:, 20].float().abs().max()) == 0.0
