"""Projections of prompts with about one output tile per compute unit (ring of LDS stages) at the edges of their tilings: rows and
columns that are no multiple of the tile, K shorter than the ring, strided rows, outputs off the 8-byte grid, bias and residual,
both rounding modes of the gate / up pair, head expansions from 16 rows on, against the same product in fp32."""
import pytest
import torch

from tests.test_gpu_big_tiles import _check, _rand
from tests.util import form_taken

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,K", [
    (200, 4096, 256), (128, 2048, 1024),                                              # 64 x 64, K halved between the waves
    (129, 5123, 128), (193, 4099, 384), (333, 3077, 128), (511, 4096, 256), (420, 3072, 640),     # 128 x 64, likewise
    (770, 3079, 64), (1025, 3072, 192), (1000, 4096, 128), (1500, 1540, 320),         # 128 x 128
])
def test_linear(B, N, K, dtype):
    from flashsvd_amd import hip_ops
    x, w = _rand(B, K + 8, seed=1, dtype=dtype)[:, 8:], _rand(N, K + 16, std=K ** -0.5, seed=2, dtype=dtype)[:, :K]
    bias, res = _rand(N, seed=3, dtype=dtype), _rand(B, N + 1, seed=4, dtype=dtype)[:, 1:]
    ref = x.float() @ w.float().t()
    _check(hip_ops.linear(x, w), ref.to(dtype), "plain")
    ref = ((ref + bias.float()).to(dtype).float() + res.float()).to(dtype)
    _check(hip_ops.linear(x, w, bias, residual=res), ref, "bias and residual")
    out = torch.full((B + 1, N + 3), 7.0, device="cuda", dtype=dtype)                 # rows and columns around the output stay as they are
    hip_ops.linear(x, w, bias, residual=res, out=out[:B, 1:N + 1])
    _check(out[:B, 1:N + 1], ref, "odd output")
    assert bool((out[B] == 7).all()) and bool((out[:, 0] == 7).all()) and bool((out[:, N + 1:] == 7).all())


@pytest.mark.parametrize("B,D,R", [(333, 11008, 64), (512, 11001, 128), (640, 5504, 192), (1030, 5507, 256), (1600, 5504, 64),
                                   (154, 11008, 128), (250, 11005, 64), (500, 5504, 320)])
def test_swiglu(B, D, R):
    from flashsvd_amd import hip_ops
    p = _rand(B, 2 * R + 8, seed=1)[:, :2 * R]
    gu, uu = _rand(D, R, std=R ** -0.5, seed=2), _rand(D, R, std=R ** -0.5, seed=3)
    g, u = p[:, :R].float() @ gu.float().t(), p[:, R:].float() @ uu.float().t()
    for mode in (0, 1):
        ref = torch.nn.functional.silu(g.bfloat16()) * u.bfloat16() if mode == 0 else ((g * torch.sigmoid(g)) * u).bfloat16()
        _check(hip_ops.swiglu_linear(p, gu, uu, up_off=R, mode=mode), ref, f"mode {mode}")


@pytest.mark.parametrize("B,T,H,Hk,R", [(1, 16, 8, 8, 64), (2, 77, 32, 8, 128), (1, 333, 5, 1, 192), (3, 43, 4, 2, 256), (1, 513, 32, 32, 320)])
def test_head_expansion(B, T, H, Hk, R):
    """One expansion alone and two in a launch; destinations by position, the later rows of a cache that is too short dropped."""
    from flashsvd_amd import hip_ops
    Dh, start = 128, 5
    p = _rand(B, T, 2 * R, seed=1)
    qu, ku, bq = _rand(H * Dh, R, std=R ** -0.5, seed=2), _rand(Hk * Dh, R, std=R ** -0.5, seed=3), _rand(H * Dh, seed=4)
    pos = torch.arange(T + start + B, device="cuda", dtype=torch.float32)
    ang = pos[:, None] * (1.0 / (10000.0 ** (torch.arange(0, 64, device="cuda", dtype=torch.float32) / 64)))[None]
    cos, sin = ang.cos().bfloat16(), ang.sin().bfloat16()
    first = torch.arange(B, device="cuda", dtype=torch.int32) + start
    q = torch.zeros(B, T, H, Dh, device="cuda", dtype=torch.bfloat16)
    k = torch.zeros(B, T + start + 1, Hk, Dh, device="cuda", dtype=torch.bfloat16)
    hip_ops.lowrank_expand_heads_multi([dict(p=p[..., :R], u=qu, num_heads=H, out=q, rotate=True, bias=bq),
                                        dict(p=p[..., R:], u=ku, num_heads=Hk, out=k, rotate=True, dst_by_position=True)],
                                       head_dim=Dh, cos=cos, sin=sin, positions=first)
    odd = torch.zeros(B, T, H, Dh + 1, device="cuda", dtype=torch.bfloat16)[..., 1:]      # rows off the 8-byte grid
    hip_ops.lowrank_expand_heads(p[..., :R], qu, num_heads=H, head_dim=Dh, bias=bq, out=odd, cos=cos, sin=sin, positions=first)
    assert torch.equal(odd, q)
    for b in range(B):
        s0 = start + b
        c, s = cos[s0:s0 + T, None], sin[s0:s0 + T, None]

        def rope(x):
            x0, x1 = x[..., :64], x[..., 64:]
            return torch.cat([x0 * c - x1 * s, x1 * c + x0 * s], -1)

        _check(q[b], rope((p[b, :, :R].float() @ qu.float().t() + bq.float()).bfloat16().view(T, H, Dh)), f"q of row {b}")
        n = min(T, k.shape[1] - s0)
        _check(k[b, s0:s0 + n], rope((p[b, :, R:].float() @ ku.float().t()).bfloat16().view(T, Hk, Dh))[:n], f"k of row {b}")
        assert not k[b, :s0].any()


# every tiling by name, each with a partial last row and column tile
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,K,form", [(200, 4035, 256, "ring 64 x 64"), (333, 3077, 128, "ring 128 x 64"), (1000, 4009, 192, "ring 128 x 128")])
def test_linear_forms(B, N, K, form, dtype):
    from flashsvd_amd import hip_ops
    x, w = _rand(B, K, seed=1, dtype=dtype), _rand(N, K, std=K ** -0.5, seed=2, dtype=dtype)
    bias, res = _rand(N, seed=3, dtype=dtype), _rand(B, N, seed=4, dtype=dtype)
    y = hip_ops.linear(x, w, bias, residual=res)
    assert form_taken() == form
    _check(y, (((x.float() @ w.float().t()) + bias.float()).to(dtype).float() + res.float()).to(dtype), form)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,D,R,form", [(333, 11005, 128, "ring 128 x 192 pair"), (154, 11005, 192, "ring 64 x 192 pair")])
def test_pair_forms(B, D, R, form, dtype):
    from flashsvd_amd import hip_ops
    p = _rand(B, 2 * R, seed=1, dtype=dtype)
    gu, uu = _rand(D, R, std=R ** -0.5, seed=2, dtype=dtype), _rand(D, R, std=R ** -0.5, seed=3, dtype=dtype)
    g, u = p[:, :R].float() @ gu.float().t(), p[:, R:].float() @ uu.float().t()
    for mode in (0, 1):
        ref = torch.nn.functional.silu(g.to(dtype)) * u.to(dtype) if mode == 0 else ((g * torch.sigmoid(g)) * u).to(dtype)
        h = hip_ops.swiglu_linear(p, gu, uu, up_off=R, mode=mode)
        assert form_taken() == form
        _check(h, ref, f"mode {mode}")
