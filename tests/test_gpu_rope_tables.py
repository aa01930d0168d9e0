"""Rotation tables of given positions in one launch against the tensor operations they replace: the same fp32 angles, cosine and sine
within two fp32 ulps of one another, so the 16-bit roundings agree but for values next to a rounding boundary."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,half", [(1, 1), (3, 64), (2, 129), (8192, 64), (77, 32)])
def test_tables(rows, half, dtype):
    from flashsvd_amd import hip_ops
    pos = torch.randint(0, 131072, (1, rows), generator=torch.Generator().manual_seed(rows)).cuda()
    inv = (1.0 / (10000.0 ** (torch.arange(half, dtype=torch.float32) / half))).cuda()
    cos, sin = hip_ops.rope_tables(pos, inv, dtype)
    ang = (pos.float()[..., None] * inv).view(rows, half)
    for got, fn in ((cos, torch.cos), (sin, torch.sin)):
        want = fn(ang.double())                                            # of the fp32 angle
        half_ulp = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)         # of values below one
        assert got.dtype == dtype and (got.double() - want).abs().max() <= half_ulp * 1.001
        assert (got != fn(ang).to(dtype)).float().mean() <= 1e-3


def test_refusals():
    from flashsvd_amd import hip_ops
    pos, inv = torch.zeros(4, dtype=torch.long, device="cuda"), torch.ones(8, device="cuda")
    for bad in ((pos.int(), inv, torch.bfloat16), (pos, inv.half(), torch.bfloat16), (pos, inv, torch.float32), (pos[::2], inv, torch.bfloat16), (pos, inv[::2], torch.float16)):
        with pytest.raises((ValueError, RuntimeError)):
            hip_ops.rope_tables(*bad)


@pytest.mark.parametrize("rows,half,shape", [(1, 1, (1, 1)), (3, 64, (4, 3)), (77, 32, (3, 255)), (1024, 64, (2, 128)), (5, 64, (1, 257)), (2, 3, (0, 4))])
def test_mask_bytes_beside_the_tables(rows, half, shape):
    from flashsvd_amd import hip_ops
    gen = torch.Generator().manual_seed(rows)
    pos = torch.randint(0, 8192, (1, rows), generator=gen).cuda()
    inv = torch.rand(half, generator=gen).cuda()
    mask = torch.randint(-1, 2, shape, generator=gen).cuda()
    mask[mask == -1] = -2 ** 40                                              # no bit in the low word
    cos, sin, pad = hip_ops.rope_tables_mask(pos, inv, torch.bfloat16, mask)
    want = hip_ops.rope_tables(pos, inv, torch.bfloat16)
    assert torch.equal(cos, want[0]) and torch.equal(sin, want[1])
    assert pad.dtype == torch.uint8 and torch.equal(pad, (mask != 0).view(torch.uint8))
    for bad in (mask.int(), torch.ones(2, 6, dtype=torch.long, device="cuda")[:, ::2]):
        with pytest.raises((ValueError, RuntimeError)):
            hip_ops.rope_tables_mask(pos, inv, torch.bfloat16, bad)
