"""Projections of a long K in shares over workgroups (csrc/mfma_quad.hip) at the edges of their tilings: partial row and column
tiles, shares of unequal length, strided and odd rows, bias and residual, against the same product in fp32; and the two-stage
ring of the head expansions at its shortest rank."""
import os

import pytest
import torch

from tests import test_gpu_mid_tiles as mid
from tests.test_gpu_big_tiles import _check, _rand
from tests.util import form_taken

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,K,form", [
    (128, 1536, 11008, "shares 64 x 128"), (191, 1027, 8256, "shares 64 x 128"), (130, 3001, 4096, "shares 64 x 128"),
    (193, 1030, 8192, "shares 128 x 128"), (333, 3070, 4160, "shares 128 x 128"),
    (512, 1500, 5504, "shares 256 x 128"), (769, 1533, 8320, "shares 128 x 128"), (1000, 1533, 8320, "shares 256 x 128"), (2047, 2390, 8192, "shares 256 x 128"),
    (150, 1027, 4096, "shares 64 x 64"), (200, 515, 4096, "shares 64 x 64"), (512, 1024, 4160, "shares 64 x 64"),
    (128, 3070, 5120, "shares 64 x 128"), (191, 2050, 5504, "shares 64 x 128"),       # cut in ranges, but enough shares to fill the chip
    (512, 1536, 11008, "shares 128 x 128"), (420, 3072, 4096, "quad 64 x 96 halves"), (520, 3072, 4096, "quad 128 x 64 halves"), (512, 4096, 4096, "quad 128 x 64 halves"), (127, 3072, 4096, "tiles 32 x 64"),
])
def test_linear(B, N, K, form, dtype):
    from flashsvd_amd import hip_ops
    x, w = _rand(B, K + 8, seed=1, dtype=dtype)[:, 8:], _rand(N, K + 16, std=K ** -0.5, seed=2, dtype=dtype)[:, :K]
    bias, res = _rand(N, seed=3, dtype=dtype), _rand(B, N + 1, seed=4, dtype=dtype)[:, 1:]
    ref = x.float() @ w.float().t()
    y = hip_ops.linear(x, w)
    assert form_taken() == form
    _check(y, ref.to(dtype), "plain")
    ref = ((ref + bias.float()).to(dtype).float() + res.float()).to(dtype)
    out = torch.full((B + 1, N + 3), 7.0, device="cuda", dtype=dtype)                 # rows and columns around the output stay as they are
    hip_ops.linear(x, w, bias, residual=res, out=out[:B, 1:N + 1])
    _check(out[:B, 1:N + 1], ref, "bias, residual, odd output")
    assert bool((out[B] == 7).all()) and bool((out[:, 0] == 7).all()) and bool((out[:, N + 1:] == 7).all())
    assert torch.equal(y, hip_ops.linear(x, w)), "repeat differs"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,K", [(150, 1027, 4096), (200, 515, 4096), (333, 259, 6208)])
def test_ranges_apart_and_in_a_row_give_the_same_bits(B, N, K, dtype):
    """A K in ranges: one workgroup each with scratch of the call's own, without it as the registered buffer or one workgroup has them."""
    from flashsvd_amd import _lib, hip_ops
    x, w = _rand(B, K, seed=1, dtype=dtype), _rand(N, K, std=K ** -0.5, seed=2, dtype=dtype)
    apart = hip_ops.linear(x, w)
    assert form_taken() == "shares 64 x 64"
    y = torch.empty_like(apart)
    code = 1 if dtype == torch.float16 else 0
    assert _lib.load().fsvd_linear(x.data_ptr(), K, w.data_ptr(), K, None, None, 0.0, None, 0, y.data_ptr(), N, B, N, K, 0, code, hip_ops._stream()) == 0
    assert not form_taken().startswith("shares")
    assert torch.equal(apart, y)


@pytest.mark.parametrize("B,N,K,form", [
    (128, 1024, 4096, "tiles 64 x 64"), (128, 256, 8192, "tiles 64 x 64"), (150, 1027, 7168, "tiles 64 x 64"), (129, 1530, 11008, "tiles 64 x 64"),
    (512, 1536, 11008, "tiles 64 x 64"), (333, 1536, 8192, "quad 64 x 64"), (333, 1280, 4096, "quad 64 x 64 ranges"),
])
def test_calls_without_scratch_split_in_the_registered_buffer(B, N, K, form):
    """fsvd_linear, whose only scratch is the registered buffer; with that too small for the split, or with none, the same call runs unsplit."""
    from flashsvd_amd import _lib, hip_ops
    lib = _lib.load()
    x, w = _rand(B, K, seed=1), _rand(N, K, std=K ** -0.5, seed=2)
    y = torch.empty(B, N, device="cuda", dtype=torch.bfloat16)
    ref = (x.float() @ w.float().t()).bfloat16()

    def call():
        y.fill_(7.0)
        assert lib.fsvd_linear(x.data_ptr(), K, w.data_ptr(), K, None, None, 0.0, None, 0, y.data_ptr(), N, B, N, K, 0, 0, hip_ops._stream()) == 0
        _check(y, ref, "without scratch")
        return form_taken(), y.clone()

    assert hip_ops.ensure_split_workspace(x.device)
    taken, split = call()
    assert taken == form
    hip_ops.release_split_workspace(x.device)
    small = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    try:
        for buf, nbytes in ((small.data_ptr(), small.numel()), (None, 0)):
            assert lib.fsvd_set_workspace(buf, nbytes, hip_ops._stream()) == 0
            taken, y1 = call()
            assert taken.startswith("quad")
            assert K >= 8192 or torch.equal(y1, split)                                 # ranges of K are added up in the same order
    finally:
        assert hip_ops.ensure_split_workspace(x.device)


@pytest.mark.parametrize("B,N,K,form", [(128, 1024, 3584, "tiles 64 x 64"), (130, 259, 2048, "tiles 64 x 64"), (512, 1024, 3328, "tiles 64 x 64"),
                                        (128, 1024, 1536, "tiles 64 x 64"), (128, 2559, 3840, "tiles 64 x 64"),
                                        (512, 768, 3584, "tiles 64 x 64"), (512, 768, 3072, "quad 64 x 64 ranges"), (200, 1024, 1600, "quad 64 x 64 ranges"), (128, 1024, 1472, "quad 64 x 64 ranges")])
def test_a_k_too_short_for_scratch(B, N, K, form):
    from flashsvd_amd import hip_ops
    x, w = _rand(B, K, seed=1), _rand(N, K, std=K ** -0.5, seed=2)
    y = hip_ops.linear(x, w)
    assert form_taken() == form
    _check(y, (x.float() @ w.float().t()).bfloat16(), form)


def test_calls_on_two_streams_are_independent():
    """Each call's sums lie in scratch of its own, the registered buffer stays as it is."""
    from flashsvd_amd import hip_ops
    xs = [_rand(333, 8192, seed=s) for s in (1, 2)]
    ws = [_rand(1536, 8192, std=8192 ** -0.5, seed=s) for s in (3, 4)]
    assert hip_ops.ensure_split_workspace(xs[0].device)
    partials = hip_ops._SPLIT_WS[0][64 << 10:]
    partials.fill_(0x5a)
    want = [hip_ops.linear(x, w) for x, w in zip(xs, ws)]
    assert int((partials != 0x5a).sum()) == 0
    streams = [torch.cuda.Stream() for _ in xs]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i].append(hip_ops.linear(xs[i], ws[i]))
    torch.cuda.synchronize()
    for i in (0, 1):
        assert all(torch.equal(g, want[i]) for g in got[i])


def test_a_buffer_that_is_too_small_means_fewer_shares():
    from flashsvd_amd import _lib, hip_ops
    lib = _lib.load()
    x, w = _rand(333, 8192, seed=1), _rand(1536, 8192, std=8192 ** -0.5, seed=2)
    y = torch.empty(333, 1536, dtype=torch.bfloat16, device="cuda")
    args = (x.data_ptr(), 8192, w.data_ptr(), 8192, None, None, 0.0, None, 0, y.data_ptr(), 1536, 333, 1536, 8192, 0, 0)
    full = lib.fsvd_linear_scratch_bytes(x.data_ptr(), 8192, w.data_ptr(), 8192, None, 0, y.data_ptr(), 1536, 333, 1536, 8192)
    ref = (x.float() @ w.float().t()).bfloat16()
    for nbytes in (full, full - 1, full // 3, 1 << 16, 0):
        scratch = torch.full((nbytes + 4096,), 0x5a, dtype=torch.uint8, device="cuda")
        rc = lib.fsvd_linear_scratch(*args, scratch.data_ptr(), nbytes, hip_ops._stream())
        assert rc == 0
        _check(y, ref, f"{nbytes} bytes")
        assert bool((scratch[nbytes:] == 0x5a).all())


@pytest.mark.parametrize("B,T,H,Hk,R", [(1, 520, 32, 32, 64), (3, 400, 20, 10, 128)])
def test_head_expansion_in_two_stages(B, T, H, Hk, R):
    mid.test_head_expansion(B, T, H, Hk, R)
    assert form_taken().startswith("ring 64 x 128")


def test_blocks_hand_their_projections_scratch():
    from flashsvd_amd import hip_ops as ops
    B, K, R, D = 333, 4096, 1500, 8192                                     # both long projections in shares
    x, gu_v, dv, du = _rand(B, K, seed=1), _rand(2 * R, K, std=K ** -0.5, seed=2), _rand(R, D, std=D ** -0.5, seed=5), _rand(K, R, std=R ** -0.5, seed=6)
    gu, uu = _rand(D, R, std=R ** -0.5, seed=3), _rand(D, R, std=R ** -0.5, seed=4)
    p = ops.linear(x, gu_v)
    assert form_taken().startswith("shares")
    s = ops.linear(ops.swiglu_linear(p, gu, uu, up_off=R), dv)
    assert form_taken().startswith("shares")
    assert torch.equal(ops.lowrank_mlp(x, gu_v, gu, uu, dv, du, residual=x), ops.linear(s, du, residual=x))


def test_the_switch_keeps_every_call_unsplit():
    """FLASHSVD_AMD_SPLITK=0 with no buffer registered: single projections and those of both blocks run in one share each."""
    from flashsvd_amd import hip_ops as ops
    B, K, R, D, H = 333, 4096, 1500, 8192, 64
    x, gu_v, dv, du = _rand(B, K, seed=1), _rand(2 * R, K, std=K ** -0.5, seed=2), _rand(R, D, std=D ** -0.5, seed=5), _rand(K, R, std=R ** -0.5, seed=6)
    gu, uu = _rand(D, R, std=R ** -0.5, seed=3), _rand(D, R, std=R ** -0.5, seed=4)
    pg, pu = _rand(B, 1504, seed=7)[:, :R], _rand(B, 1504, seed=8)[:, :R]
    qkv_v, ov, ou = _rand(3 * 64, K, std=K ** -0.5, seed=9), _rand(R, H * 128, std=(H * 128) ** -0.5, seed=10), _rand(K, R, std=R ** -0.5, seed=11)
    qu, ku, vu = (_rand(H * 128, 64, std=0.125, seed=12 + i) for i in range(3))
    cos, sin = _rand(B, 64, seed=15), _rand(B, 64, seed=16)
    k, v = torch.zeros(1, B, H, 128, device="cuda", dtype=torch.bfloat16), torch.zeros(1, B, H, 128, device="cuda", dtype=torch.bfloat16)

    def long(a, w):
        y = ops.linear(a, w)
        assert not form_taken().startswith("shares"), form_taken()
        return y

    os.environ["FLASHSVD_AMD_SPLITK"] = "0"
    ops.release_split_workspace(x.device)
    try:
        y = long(ops.swiglu_linear(long(x, gu_v), gu, uu, up_off=R), dv)
        assert torch.equal(ops.lowrank_mlp(x, gu_v, gu, uu, dv, du, residual=x), ops.linear(y, du, residual=x))
        y = long(ops.swiglu_linear(torch.cat([pg, pu], 1), gu, uu, up_off=R, mode=1), dv)
        assert torch.equal(ops._mlp_from_coefficients(pg, pu, gu, uu, dv, du, None, 1), ops.linear(y, du))
        got = ops.lowrank_attn_prefill(x[None], qkv_v, qu, ku, vu, ov, ou, k, v, cos, sin, start=0, num_heads=H, num_kv_heads=H)
        p = long(x, qkv_v)
        q = ops.lowrank_expand_heads(p[None, :, :64], qu, num_heads=H, head_dim=128, out=torch.empty_like(k), cos=cos, sin=sin)
        a = ops.attn_prefill(q, k, v, causal=True)
        assert torch.equal(got[0], ops.linear(long(a.view(B, -1), ov), ou))
    finally:
        del os.environ["FLASHSVD_AMD_SPLITK"]
        assert ops.ensure_split_workspace(x.device)
