"""Projections and head expansions on the four-wave tiles (csrc/mfma_quad.hpp) at the edges of every tiling: partial row and column
tiles, one and several tiles per workgroup, K of five steps and ragged K, K halved and cut in ranges, rows off the 16-byte grid, bias and
residual; and the vocabulary of one and two rows as a stream (csrc/gemv.hip), against the same product in fp32."""
import pytest
import torch

from tests.test_gpu_big_tiles import _check, _expand_and_compare, _rand
from tests.util import form_taken

pytestmark = pytest.mark.gpu


def _linear(B, N, K, dtype, any_grid=False):
    """plain, and with bias and residual into the middle of a larger output; the form taken"""
    from flashsvd_amd import hip_ops
    lead = 2 if any_grid else 8                                                       # rows from the 4-byte or the 16-byte grid
    pad = lead + (K & 1)
    x, w = _rand(B, K + pad, seed=1, dtype=dtype)[:, pad - (K & 1):][:, :K], _rand(N, K + pad, std=K ** -0.5, seed=2, dtype=dtype)[:, :K]
    bias, res = _rand(N, seed=3, dtype=dtype), _rand(B, N + 1, seed=4, dtype=dtype)[:, 1:]
    ref = x.float() @ w.float().t()
    y = hip_ops.linear(x, w)
    form = form_taken()
    _check(y, ref.to(dtype), "plain")
    ref = ((ref + bias.float()).to(dtype).float() + res.float()).to(dtype)
    out = torch.full((B + 1, N + 3), 7.0, device="cuda", dtype=dtype)                 # rows and columns around the output stay as they are
    hip_ops.linear(x, w, bias, residual=res, out=out[:B, 1:N + 1])
    _check(out[:B, 1:N + 1], ref, "bias, residual, odd output")
    assert bool((out[B] == 7).all()) and bool((out[:, 0] == 7).all()) and bool((out[:, N + 1:] == 7).all())
    return form


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,K,form", [
    (1036, 11077, 320, "quad 256 x 256"), (706, 11209, 320, "quad 256 x 192"), (341, 12357, 320, "quad 128 x 192"),
    (777, 7569, 320, "quad 256 x 128"), (514, 9972, 320, "quad 192 x 128"), (130, 11060, 320, "quad 128 x 128"),
    (519, 11227, 320, "quad 128 x 128 alone"), (69, 17004, 1024, "quad 128 x 96"), (99, 8635, 320, "quad 64 x 96"), (99, 12400, 320, "quad 128 x 64"),
    (133, 9272, 320, "quad 64 x 128"), (66, 8328, 320, "quad 96 x 64"), (3648, 1056, 320, "quad 128 x 64"),
    (33, 4170, 320, "quad 64 x 64"), (190, 13257, 1280, "quad 128 x 128 alone"), (190, 13257, 1216, "quad 96 x 64"), (300, 24001, 320, "quad 256 x 192"),
    (130, 259, 320, "quad 64 x 64"),
    (197, 5541, 384, "quad 64 x 96 halves"), (197, 6201, 384, "quad 128 x 64 halves"), (132, 5545, 384, "quad 96 x 64 halves"), (128, 8256, 384, "quad 64 x 96 halves"), (135, 1362, 384, "quad 64 x 64 halves"),
    (130, 259, 1088, "quad 64 x 64 ranges"), (300, 517, 1088, "quad 64 x 64 ranges"), (301, 261, 1408, "quad 64 x 64 ranges"),
])
def test_linear(B, N, K, form, dtype):
    assert _linear(B, N, K, dtype) == form


@pytest.mark.parametrize("B,N,K,single,pair", [
    (64, 4090, 3072, "tiles 32 x 64", "tiles 32 x 64 pair"), (33, 4096, 1984, "quad 64 x 64", "tiles 32 x 64 pair"), (100, 4096, 960, "quad 64 x 64", "quad 64 x 96 pair"),
    (127, 4090, 5184, "tiles 32 x 64", "tiles 32 x 64 pair"), (127, 4096, 2048, "quad 64 x 64", "tiles 32 x 64 pair"), (64, 5500, 1280, "quad 64 x 64", "tiles 32 x 64 pair"),
    (70, 8192, 5184, "quad 64 x 64", "quad 64 x 96 pair"), (65, 4096, 5184, "quad 64 x 64", "tiles 32 x 64 pair"), (65, 4096, 2048, "quad 64 x 64", "quad 64 x 96 pair"),
])
def test_few_tiles_of_a_long_k_split(B, N, K, single, pair):
    """33 to 127 rows: on either side of the lines, with the registered buffer; without it everything runs here."""
    from flashsvd_amd import _lib, hip_ops
    x, w, w2 = _rand(B, K, seed=1), _rand(N, K, std=K ** -0.5, seed=2), _rand(N, K, std=K ** -0.5, seed=3)
    ref = x.float() @ w.float().t()
    act = torch.nn.functional.silu(ref.bfloat16()) * (x.float() @ w2.float().t()).bfloat16()
    _check(hip_ops.linear(x, w), ref.bfloat16(), "single")
    assert form_taken() == single
    _check(hip_ops.swiglu_linear(x, w, w2, up_off=0), act, "pair")
    assert form_taken() == pair
    hip_ops.release_split_workspace(x.device)
    y = torch.empty(B, N, device="cuda", dtype=torch.bfloat16)
    try:
        rc = _lib.load().fsvd_linear(x.data_ptr(), K, w.data_ptr(), K, None, None, 0.0, None, 0, y.data_ptr(), N, B, N, K, 0, 0, hip_ops._stream())
        assert rc == 0 and form_taken() == ("quad 64 x 64" if (N + 63) // 64 * ((B + 63) // 64) >= 128 or K < 4096 else "rows 16")
        _check(y, ref.bfloat16(), "no buffer")
    finally:
        assert hip_ops.ensure_split_workspace(x.device)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,K,form", [
    (297, 12319, 323, "any quad 192 x 128"), (128, 8256, 322, "any quad 128 x 128"), (130, 5559, 383, "any quad 96 x 64"),
    (131, 4103, 321, "any quad 64 x 64"), (8230, 8, 385, "any quad 64 x 64"), (200, 4096, 1281, "any quad 64 x 64"),
    # on either side of the lines to the other tiles
    (128, 259, 321, "any rows 32 x 64"), (130, 259, 321, "any quad 64 x 64"), (130, 259, 1025, "any rows 32 x 64"), (131, 8, 385, "any quad 64 x 64"),
    (200, 1002, 1025, "any quad 64 x 64"), (200, 1002, 2050, "any rows 32 x 64"), (128, 4096, 1490, "any rows 32 x 64"), (200, 4096, 2050, "any quad 64 x 64"),
    (200, 5504, 2050, "any rows 64 x 64"), (256, 4096, 1281, "any rows 64 x 64"), (500, 4090, 1490, "any ring 64 x 128"), (1500, 700, 1490, "any quad 96 x 64"),
    (154, 11008, 1282, "any ring 128 x 128"),
    (154, 11008, 1274, "any quad 96 x 64"), (154, 5500, 2050, "any rows 64 x 64"), (420, 5504, 1490, "any quad 96 x 64"),
])
def test_linear_any_grid(B, N, K, form, dtype):
    assert _linear(B, N, K, dtype, any_grid=True) == form


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,D,R,form", [
    (341, 12357, 320, "quad 128 x 192 pair"), (783, 9447, 320, "quad 160 x 192 pair"), (409, 10404, 320, "quad 160 x 128 pair"),
    (168, 27083, 1280, "quad 256 x 128 pair"), (261, 9918, 320, "quad 128 x 128 pair"), (67, 25091, 832, "quad 128 x 128 pair alone"),
    (129, 17205, 896, "quad 96 x 192 pair"), (72, 12319, 320, "quad 96 x 96 pair"), (66, 8328, 320, "quad 64 x 96 pair"),
    (130, 259, 320, "quad 64 x 64 pair"), (250, 4090, 960, "quad 64 x 96 pair"), (250, 4090, 1024, "tiles 64 x 64 pair"), (260, 4090, 1152, "quad 64 x 96 pair"),
    (790, 2750, 1536, "quad 64 x 96 pair"), (250, 11001, 960, "quad 64 x 96 pair"), (250, 11001, 1024, "ring 64 x 192 pair"),
    (341, 12357, 323, "any quad 128 x 192 pair"), (261, 9918, 322, "any quad 128 x 128 pair"), (129, 17205, 894, "any quad 96 x 192 pair"),
    (130, 8954, 383, "any quad 96 x 96 pair"), (130, 259, 321, "any quad 64 x 96 pair"), (40, 8300, 330, "any quad 64 x 96 pair"),
    (40, 8190, 330, "any rows 32 x 64 pair"), (130, 2750, 1153, "any rows 64 x 64 pair"), (130, 2750, 1151, "any quad 64 x 96 pair"),
])
def test_pair(B, D, R, form, dtype):
    from flashsvd_amd import hip_ops
    up = R + (R & 1)                                                                  # the up half starts on the 4-byte grid
    p = _rand(B, 2 * up, seed=1, dtype=dtype)
    gu, uu = (_rand(D, up, std=R ** -0.5, seed=s, dtype=dtype)[:, :R] for s in (2, 3))
    g, u = p[:, :R].float() @ gu.float().t(), p[:, up:up + R].float() @ uu.float().t()
    out = torch.full((B + 1, D + 3), 7.0, device="cuda", dtype=dtype)
    hip_ops.swiglu_linear(p, gu, uu, up_off=up, out=out[:B, 1:D + 1])
    assert form_taken() == form
    _check(out[:B, 1:D + 1], torch.nn.functional.silu(g.to(dtype)) * u.to(dtype), form)
    assert bool((out[B] == 7).all()) and bool((out[:, 0] == 7).all()) and bool((out[:, D + 1:] == 7).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,H,Hk,R,form", [
    (2, 866, 46, 9, 320, "quad 256 x 256 heads"), (2, 641, 48, 9, 320, "quad 192 x 128 heads"), (1, 650, 36, 7, 320, "quad 160 x 128 heads"),
    (1, 391, 45, 9, 320, "quad 128 x 128 heads"), (2, 166, 36, 7, 320, "quad 96 x 128 heads"), (1, 130, 36, 7, 320, "quad 64 x 128 heads"),
    (3, 11, 2, 1, 320, "quad 64 x 64 heads"), (1, 17, 3, 1, 384, "quad 64 x 64 heads"),
    (1, 391, 45, 9, 322, "any quad 128 x 128 heads"), (2, 166, 36, 7, 322, "any quad 96 x 128 heads"), (3, 11, 2, 1, 382, "any quad 64 x 64 heads"),
])
def test_heads(B, T, H, Hk, R, form, dtype):
    """Row tiles across sequences, rows past the cache dropped, tiles that straddle heads."""
    assert _expand_and_compare(B, T, H, Hk, R, dtype) == form


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,K", [(16384, 4096), (16387, 2048), (32001, 4096), (128257, 2048), (16385, 512), (32003, 1024), (32769, 1024), (50304, 512),
                                 (20479, 512), (20480, 512), (102401, 4096)])
@pytest.mark.parametrize("B", [1, 2])
def test_vocabulary_stream(B, N, K, dtype):
    """Slabs of unequal length, rows that are no multiple of the window, strided weight rows, norm, bias and residual."""
    from flashsvd_amd import hip_ops
    x, w = _rand(B, K + 8, seed=1, dtype=dtype)[:, 8:], _rand(N, K + 8, std=K ** -0.5, seed=2, dtype=dtype)[:, :K]
    bias, res, nw = _rand(N, seed=3, dtype=dtype), _rand(B, N, seed=4, dtype=dtype), _rand(K, seed=5, dtype=dtype)
    ref = x.float() @ w.float().t()
    y = hip_ops.linear(x, w)
    beside = {(1, 512): N < 20480, (1, 1024): N > 32768, (2, 4096): N > 102400}        # what stays with the kernel beside it
    assert form_taken() == ("vector" if beside.get((B, K)) else "rows in a window")
    _check(y, ref.to(dtype), "plain")
    assert torch.equal(y, hip_ops.linear(x, w, cfg=4)) and form_taken() == "vector"      # the same bits as four rows to a wave
    out = torch.full((B + 1, N + 3), 7.0, device="cuda", dtype=dtype)
    hip_ops.linear(x, w, bias, residual=res, out=out[:B, 1:N + 1])
    _check(out[:B, 1:N + 1], ((ref + bias.float()).to(dtype).float() + res.float()).to(dtype), "bias and residual")
    assert bool((out[B] == 7).all()) and bool((out[:, 0] == 7).all()) and bool((out[:, N + 1:] == 7).all())
    xn = hip_ops.rmsnorm(x, nw, 1e-6)
    _check(hip_ops.linear(x, w, norm_weight=nw), (xn.float() @ w.float().t()).to(dtype), "norm")
    assert torch.equal(y, torch.cat([hip_ops.linear(x[b:b + 1], w) for b in range(B)]))
