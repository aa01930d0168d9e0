"""Ragged projections of 128 rows and more on the tiles of csrc/mfma_mid.hip: K off the step (an odd and an even number of whole steps,
one element past and short of them), rows at odd addresses, partial row and column tiles, bias and residual,
both rounding modes of the pair, against the same product in fp32; memory around the rows is NaN and must not be read into them."""
import pytest
import torch

from tests.test_gpu_big_tiles import _check, _rand
from tests.util import form_taken

pytestmark = pytest.mark.gpu


def _among_nan(rows, cols, off, std, seed, dtype):
    """[rows, cols] at odd addresses inside a buffer of NaN (one after every row, `off` in front)."""
    buf = torch.full((rows * (cols + 3) + 64,), float("nan"), dtype=dtype, device="cuda")
    v = buf.as_strided((rows, cols), (cols + 3, 1), off)
    v.copy_(_rand(rows, cols, std=std, seed=seed, dtype=dtype))
    return v


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,K,form", [
    (770, 4090, 1492, "any ring 128 x 128"), (1000, 4001, 131, "any ring 128 x 128"), (641, 3977, 255, "any ring 128 x 128"), (700, 3970, 129, "any ring 128 x 128"),
    (512, 4095, 1491, "any ring 64 x 128"), (333, 3000, 1001, "any ring 64 x 128"), (500, 4090, 2390, "any ring 64 x 128"), (450, 4000, 193, "any ring 64 x 128"),
    (333, 4096, 2390, "any rows 64 x 64"), (1500, 4096, 190, "any rows 128 x 128"), (127, 4096, 1491, "any rows 32 x 64"), (512, 4095, 127, "any rows 64 x 64"),
])
def test_linear(B, N, K, form, dtype):
    from flashsvd_amd import hip_ops
    x, w = _among_nan(B, K, 1, 1.0, 1, dtype), _among_nan(N, K, 3, K ** -0.5, 2, dtype)
    bias, res = _rand(N, seed=3, dtype=dtype), _rand(B, N + 1, seed=4, dtype=dtype)[:, 1:]
    y = hip_ops.linear(x, w, bias, residual=res)
    assert form_taken() == form
    _check(y, (((x.float() @ w.float().t()) + bias.float()).to(dtype).float() + res.float()).to(dtype), form)
    assert torch.equal(y, hip_ops.linear(x, w, bias, residual=res)), "repeat differs"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,D,R,form", [
    (333, 11005, 1492, "any ring 128 x 192 pair"), (512, 11008, 131, "any ring 128 x 192 pair"), (700, 5500, 191, "any ring 128 x 192 pair"),
    (154, 11001, 129, "any ring 64 x 192 pair"), (400, 5504, 747, "any ring 64 x 192 pair"), (128, 11008, 190, "any rows 64 x 64 pair"),
])
def test_pair(B, D, R, form, dtype):
    from flashsvd_amd import hip_ops
    p = _among_nan(B, 2 * R + 1, 1, 1.0, 1, dtype)
    gu, uu = _among_nan(D, R, 5, R ** -0.5, 2, dtype), _among_nan(D, R, 7, R ** -0.5, 3, dtype)
    off = R + 1                                                            # the two halves one element apart
    g, u = p[:, :R].float() @ gu.float().t(), p[:, off:].float() @ uu.float().t()
    for mode in (0, 1):
        ref = torch.nn.functional.silu(g.to(dtype)) * u.to(dtype) if mode == 0 else ((g * torch.sigmoid(g)) * u).to(dtype)
        h = hip_ops.swiglu_linear(p, gu, uu, up_off=off, mode=mode)
        assert form_taken() == form
        _check(h, ref, f"mode {mode}")
