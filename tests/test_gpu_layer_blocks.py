"""The halves of a layer in one native call (fsvd_mlp_block_run, fsvd_attn_block_prefill) give the bits of the single operators, at
the row counts where those change kernels, with and without norm, residual and bias, over strided rows and a used cache."""
import pytest
import torch

from tests.test_gpu_big_tiles import _rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,K,R,D,N", [(1, 512, 128, 1376, 512), (2, 264, 136, 520, 264), (3, 512, 128, 1376, 512), (16, 512, 122, 1376, 512), (33, 512, 128, 1376, 512),
                                       (130, 512, 192, 1408, 512), (300, 1024, 250, 2048, 1024)])
def test_mlp_block(B, K, R, D, N, dtype):
    from flashsvd_amd import hip_ops as ops
    x = _rand(B, K + 8, seed=1, dtype=dtype)[:, :K]
    gu_v, gu, uu = _rand(2 * R, K, std=K ** -0.5, seed=2, dtype=dtype), _rand(D, R, std=R ** -0.5, seed=3, dtype=dtype), _rand(D, R, std=R ** -0.5, seed=4, dtype=dtype)
    dv, du = _rand(R + 2, D, std=D ** -0.5, seed=5, dtype=dtype), _rand(N, R + 2, std=R ** -0.5, seed=6, dtype=dtype)
    nw, res = 1 + _rand(K, std=0.1, seed=7, dtype=dtype), _rand(B, N, seed=8, dtype=dtype)
    for norm, r, mode in ((nw, res, 0), (None, None, 1), (nw, None, 0)):
        p = ops.linear(x, gu_v, norm_weight=norm, eps=1e-5)
        want = ops.linear(ops.linear(ops.swiglu_linear(p, gu, uu, up_off=R, mode=mode), dv), du, residual=r)
        assert torch.equal(ops.lowrank_mlp(x, gu_v, gu, uu, dv, du, norm_weight=norm, eps=1e-5, residual=r, mode=mode), want)
    pg, pu = p[:, :R].contiguous(), p[:, R:].contiguous()
    bias = _rand(N, seed=9, dtype=dtype)
    h = ops.swiglu_linear(torch.cat([pg, pu], 1), gu, uu, up_off=R, mode=1)
    want = ops.linear(ops.linear(h, dv), du, bias)
    for a, b in ((pg, pu), (p[:, :R], p[:, R:])):                          # tensors of their own in either order of address, views of a packed one
        assert torch.equal(ops._mlp_from_coefficients(a, b, gu, uu, dv, du, bias, 1), want)
    both = torch.stack([pu, pg])
    assert torch.equal(ops._mlp_from_coefficients(both[1], both[0], gu, uu, dv, du, bias, 1), want)


@pytest.mark.parametrize("B,K,R,D,pad,off", [(239, 512, 128, 256, 0, 0), (240, 512, 128, 256, 0, 1), (256, 512, 130, 256, 64, 3), (1536, 8, 8, 64, 0, 7), (1537, 512, 128, 256, 0, 0),
                                             (320, 512, 128, 256, 72, 0), (256, 16384, 64, 64, 8, 5), (64, 512, 384, 4096, 0, 0), (160, 1024, 384, 2816, 8, 8),
                                             (512, 1024, 330, 2818, 2, 2), (512, 512, 320, 5504, 64, 0), (130, 512, 321, 1411, 0, 1)])
def test_weights_asked_for_ahead(B, K, R, D, pad, off):
    """The norm's launch and the compute units that a projection leaves idle read the weights of the launches behind them: row strides up to
    an eighth over the row and more, weights at any element's address, ranges with no whole piece beside them, all compute units taken."""
    from flashsvd_amd import hip_ops as ops

    def weight(n, k, seed):
        return _rand(n * (k + pad) + off, std=k ** -0.5, seed=seed)[off:].view(n, k + pad)[:, :k]

    x, nw = _rand(B, K, seed=1), 1 + _rand(K, std=0.1, seed=7)
    gu_v, gu, uu, dv, du = weight(2 * R, K, 2), weight(D, R, 3), weight(D, R, 4), weight(R, D, 5), weight(K, R, 6)
    p = ops.linear(x, gu_v, norm_weight=nw)
    want = ops.linear(ops.linear(ops.swiglu_linear(p, gu, uu, up_off=R), dv), du, residual=x)
    for _ in range(2):
        assert torch.equal(ops.lowrank_mlp(x, gu_v, gu, uu, dv, du, norm_weight=nw, residual=x), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,start,H,Hk,R", [(1, 16, 0, 4, 4, 128), (2, 77, 131, 8, 2, 128), (1, 333, 7, 4, 4, 122), (1, 700, 0, 32, 32, 64), (3, 512, 5, 16, 4, 192)])
def test_attention_block(B, T, start, H, Hk, R, dtype):
    from flashsvd_amd import hip_ops as ops
    K, Dh, S = 512, 128, start + T + 3
    x = _rand(B, T, K, seed=1, dtype=dtype)
    qkv_v = _rand(3 * R, K, std=K ** -0.5, seed=2, dtype=dtype)
    qu, ku, vu = (_rand(h * Dh, R, std=R ** -0.5, seed=3 + i, dtype=dtype) for i, h in enumerate((H, Hk, Hk)))
    ov, ou = _rand(R + 8, H * Dh, std=(H * Dh) ** -0.5, seed=6, dtype=dtype), _rand(K, R + 8, std=R ** -0.5, seed=7, dtype=dtype)
    bv, bu, nw = _rand(R + 8, seed=8, dtype=dtype), _rand(K, seed=9, dtype=dtype), 1 + _rand(K, std=0.1, seed=10, dtype=dtype)
    ang = torch.arange(S, device="cuda")[:, None] * (10000.0 ** (-torch.arange(0, 64, device="cuda") / 64))[None]
    cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)
    caches = [[_rand(B + 1, S, Hk, Dh, seed=11, dtype=dtype), _rand(B + 1, S, Hk, Dh, seed=12, dtype=dtype)] for _ in range(2)]
    p = ops.linear(x, qkv_v, norm_weight=nw)
    pos0 = torch.full((B,), start, device="cuda", dtype=torch.int32)
    q, (k, v) = torch.empty(B, T, H, Dh, device="cuda", dtype=dtype), caches[0]
    ops.lowrank_expand_heads_multi([dict(p=p[..., :R], u=qu, num_heads=H, out=q, rotate=True),
                                    dict(p=p[..., R:2 * R], u=ku, num_heads=Hk, out=k[:B], rotate=True, dst_by_position=True),
                                    dict(p=p[..., 2 * R:], u=vu, num_heads=Hk, out=v[:B], dst_by_position=True)],
                                   head_dim=Dh, cos=cos, sin=sin, positions=pos0)
    a = ops.attn_prefill(q, k[:B], v[:B], q_pos0=pos0, causal=True)
    want = ops.linear(ops.linear(a.view(B, T, H * Dh), ov, bv), ou, bu, residual=x)
    got = ops.lowrank_attn_prefill(x, qkv_v, qu, ku, vu, ov, ou, *caches[1], cos, sin, start=start, num_heads=H, num_kv_heads=Hk, norm_weight=nw,
                                   residual=x, o_v_bias=bv, o_u_bias=bu)
    assert torch.equal(got, want) and torch.equal(caches[0][0], caches[1][0]) and torch.equal(caches[0][1], caches[1][1])


def test_refusals():
    from flashsvd_amd import hip_ops as ops
    x = _rand(4, 64, seed=1)
    f = dict(gu_v=_rand(32, 64, seed=2), gate_u=_rand(48, 16, seed=3), up_u=_rand(48, 16, seed=4), down_v=_rand(16, 48, seed=5), down_u=_rand(64, 16, seed=6))
    ops.lowrank_mlp(x, **f)
    for name, bad in (("gu_v", _rand(30, 64, seed=2)), ("up_u", _rand(48, 17, seed=3)), ("down_v", _rand(16, 47, seed=4)), ("down_u", _rand(64, 15, seed=4)),
                      ("gate_u", f["gate_u"].float()), ("down_u", f["down_u"].t())):
        with pytest.raises((ValueError, RuntimeError)):
            ops.lowrank_mlp(x, **{**f, name: bad})
    for kw in (dict(residual=_rand(3, 64, seed=1)), dict(norm_weight=_rand(63, seed=1)), dict(mode=2)):
        with pytest.raises((ValueError, RuntimeError)):
            ops.lowrank_mlp(x, **f, **kw)
    k = _rand(1, 20, 1, 128, seed=1)
    cs = _rand(20, 64, seed=1)
    w = dict(qkv_v=_rand(48, 64, seed=2), q_u=_rand(128, 16, seed=3), k_u=_rand(128, 16, seed=3), v_u=_rand(128, 16, seed=3), o_v=_rand(16, 128, seed=3),
             o_u=_rand(64, 16, seed=3))
    with pytest.raises((ValueError, RuntimeError)):                        # past the end of the cache
        ops.lowrank_attn_prefill(_rand(1, 16, 64, seed=1), **w, k_cache=k, v_cache=k.clone(), cos=cs, sin=cs, start=5, num_heads=1, num_kv_heads=1)


def test_dual_split_operator_takes_rows_of_any_stride():
    """The operator's coefficient rows may be one row expanded, overlap, or start off the 16-byte grid."""
    T, R, D, N = 5, 64, 128, 96
    w = [_rand(*s, std=s[0] ** -0.5, seed=i) for i, s in enumerate(((R, D), (R, D), (D, R), (R, N)))]
    base = _rand(T * (R + 8) + 8, seed=9)
    from flashsvd_amd.torch_ops import ops as registered
    for size, start in ((0, 0), (8, 0), (R, 1), (R + 3, 0), (R + 8, 8)):
        pu, pg = base.as_strided((T, R), (size, 1), start), base.flip(0).as_strided((T, R), (size, 1), start)
        got, want = (registered.mlp_dual_split(u, g, *w, None, 2, 64, True, None) for u, g in ((pu, pg), (pu.clone(memory_format=torch.contiguous_format), pg.clone(memory_format=torch.contiguous_format))))
        assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,start,H,Hk,R", [(1, 17, 0, 4, 4, 320), (2, 77, 131, 8, 2, 384), (1, 333, 7, 4, 4, 330), (1, 128, 0, 32, 8, 320), (1, 257, 3, 8, 8, 576)])
def test_attention_block_of_large_ranks(B, T, start, H, Hk, R, dtype):
    """Ranks whose head expansions run on few four-wave tiles: the compute units that these leave idle read o_v and o_u."""
    test_attention_block(B, T, start, H, Hk, R, dtype)
