"""Projections and head expansions whose operands span gigabytes (few long rows in a far wider buffer): byte offsets between 2 and
4 GiB, which the direct loads of the tiled kernels carry in 32 unsigned bits, and operands past 4 GiB, which other kernels take
and which do not come to share the device's split workspace by that, against the same product in fp32."""
import pytest
import torch

from tests.test_gpu_big_tiles import _check, _rand

pytestmark = pytest.mark.gpu

# the operands start 3 GiB into the buffer: an offset taken as signed, or cut short, would read zeros of the same buffer
_BASE = 3 << 29


@pytest.fixture(scope="module")
def pool():
    buf = torch.zeros(_BASE + 9216 * 262144 + 65536, dtype=torch.bfloat16, device="cuda")
    yield buf
    del buf
    torch.cuda.empty_cache()


def _spread(pool, rows, cols, ld, at, seed, std=1.0):
    """[rows, cols] random values, rows ``ld`` elements apart, from column ``at`` of the buffer's rows on"""
    v = pool.as_strided((rows, cols), (ld, 1), _BASE + at)
    v.copy_(_rand(rows, cols, std=std, seed=seed))
    return v


@pytest.mark.parametrize("B,N,K", [(1000, 4096, 128), (300, 4096, 128), (150, 4096, 256), (4096, 4096, 128)])
def test_linear_offsets_past_2_gib(pool, B, N, K):
    """One shape per tiling (128 x 128, 128 x 64, 64 x 64, 256 x 256); the weights, then the activations, spread over 3.3 GiB."""
    from flashsvd_amd import hip_ops
    ld = 420_000 // 8 * 8
    assert (2 << 30) < N * ld * 2 < (4 << 30)
    x, w = _rand(B, K, seed=1), _spread(pool, N, K, ld, 0, 2, K ** -0.5)
    _check(hip_ops.linear(x, w), (x.float() @ w.float().t()).bfloat16(), "weights")
    w = w.contiguous()
    xs = _spread(pool, B, K, ((3 << 30) // (2 * B)) // 8 * 8, 0, 1)
    _check(hip_ops.linear(xs, w), (xs.float() @ w.float().t()).bfloat16(), "activations")


@pytest.mark.parametrize("B,D,R", [(333, 11008, 64), (1100, 11000, 128)])
def test_pair_offsets_past_2_gib(pool, B, D, R):
    from flashsvd_amd import hip_ops
    ld = 160_000
    assert (2 << 30) < D * ld * 2 < (4 << 30)
    gu, uu = _spread(pool, D, R, ld, 0, 2, R ** -0.5), _spread(pool, D, R, ld, 1024, 3, R ** -0.5)
    p = _rand(B, 2 * R, seed=1)
    g, u = p[:, :R].float() @ gu.float().t(), p[:, R:].float() @ uu.float().t()
    ref = torch.nn.functional.silu(g.bfloat16()) * u.bfloat16()
    _check(hip_ops.swiglu_linear(p, gu, uu, up_off=R), ref, "weights")
    gu, uu = gu.contiguous(), uu.contiguous()
    p = _spread(pool, B, 2 * R, ((3 << 30) // (2 * B)) // 8 * 8, 0, 1)
    _check(hip_ops.swiglu_linear(p, gu, uu, up_off=R), ref, "activations")


@pytest.mark.parametrize("T,H", [(100, 32), (3100, 33)])
def test_head_expansion_offsets_past_2_gib(pool, T, H):
    from flashsvd_amd import hip_ops
    R, Dh = 128, 128
    p, u = _spread(pool, T, R, ((3 << 30) // (2 * T)) // 8 * 8, 0, 1), _rand(H * Dh, R, std=R ** -0.5, seed=2)
    out = torch.zeros(1, T, H, Dh, dtype=torch.bfloat16, device="cuda")
    hip_ops.lowrank_expand_heads(p[None], u, num_heads=H, head_dim=Dh, out=out)
    _check(out[0], (p.float() @ u.float().t()).bfloat16().view(T, H, Dh), "coefficients")
    p = p.contiguous()
    u = _spread(pool, H * Dh, R, ((3 << 30) // (2 * H * Dh)) // 8 * 8, 0, 3, R ** -0.5)
    out.zero_()
    hip_ops.lowrank_expand_heads(p[None], u, num_heads=H, head_dim=Dh, out=out)
    _check(out[0], (p.float() @ u.float().t()).bfloat16().view(T, H, Dh), "bases")


def test_operands_past_4_gib(pool):
    """130 rows of 8192 against 9216 weight rows spread over 4.5 GiB: 144 tiles of 128 x 128."""
    from flashsvd_amd import hip_ops
    B, N, K = 130, 9216, 8192
    x, w = _rand(B, K, seed=1), _spread(pool, N, K, 262144, 0, 2, K ** -0.5)
    assert hip_ops.ensure_split_workspace(x.device)
    partials = hip_ops._SPLIT_WS[0][64 << 10:]
    partials.fill_(0x5a)
    y = hip_ops.linear(x, w)
    untouched = int((partials != 0x5a).sum()) == 0
    _check(y, (x.float() @ w.float().t()).bfloat16(), "past 4 GiB")
    assert untouched
