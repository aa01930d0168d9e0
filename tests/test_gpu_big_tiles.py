"""The 256 x 256 tile projections of long prompts at the edges of their range: rows and columns that are no multiple of the
tile, the shortest K (two steps), one and several tiles per compute unit, strided rows, bias and residual, both element
types, the gate / up pair and the head expansion with odd head counts and positions, against the same product in fp32."""
import pytest
import torch

from tests.util import bounds, form_taken

pytestmark = pytest.mark.gpu


def _rand(*shape, std=1.0, seed=0, dtype=torch.bfloat16):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return (torch.randn(*shape, generator=gen, device="cuda") * std).to(dtype)


def _check(got, ref, what):
    """One rounding of the output apart (two ulps at the largest value) and 1e-2 of it, as for every other kernel."""
    b = bounds(ref)
    err = (got.float() - ref.float()).abs().max().item()
    assert torch.isfinite(got).all() and err <= b["abs_tol"] and err <= b["rel_tol"] * ref.float().abs().max().item(), f"{what}: {err}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,K", [(3000, 3080, 128), (2049, 4616, 192), (4096, 4096, 256), (9000, 4104, 128), (256, 40000, 128)])
def test_linear(B, N, K, dtype):
    from flashsvd_amd import hip_ops
    x, w = _rand(B, K + 8, seed=1, dtype=dtype)[:, 8:], _rand(N, K + 16, std=K ** -0.5, seed=2, dtype=dtype)[:, :K]
    bias, res = _rand(N, seed=3, dtype=dtype), _rand(B, N, seed=4, dtype=dtype)
    ref = x.float() @ w.float().t()
    _check(hip_ops.linear(x, w), ref.to(dtype), "plain")
    ref = (ref + bias.float()).to(dtype).float() + res.float()
    _check(hip_ops.linear(x, w, bias, residual=res), ref.to(dtype), "bias and residual")


@pytest.mark.parametrize("B,D,R", [(3000, 3080, 128), (1025, 8200, 192), (256, 33000, 128), (5000, 7000, 64)])
def test_swiglu(B, D, R):
    from flashsvd_amd import hip_ops
    p = _rand(B, 2 * R, seed=1)
    gu, uu = _rand(D, R, std=R ** -0.5, seed=2), _rand(D, R, std=R ** -0.5, seed=3)
    for mode in (0, 1):
        h = hip_ops.swiglu_linear(p, gu, uu, up_off=R, mode=mode)
        g, u = p[:, :R].float() @ gu.float().t(), p[:, R:].float() @ uu.float().t()
        ref = torch.nn.functional.silu(g.bfloat16()) * u.bfloat16() if mode == 0 else ((g * torch.sigmoid(g)) * u).bfloat16()
        _check(h, ref, f"mode {mode}")


@pytest.mark.parametrize("B,T,H,Hk,R", [(3, 700, 32, 3, 128), (1, 2049, 33, 1, 192), (4, 1024, 32, 8, 128)])
def test_head_expansion(B, T, H, Hk, R):
    _expand_and_compare(B, T, H, Hk, R, torch.bfloat16)


def _expand_and_compare(B, T, H, Hk, R, dtype):
    from flashsvd_amd import hip_ops
    Dh, start = 128, 5
    p = _rand(B, T, 2 * R, seed=1, dtype=dtype)
    qu, ku, bq = (_rand(H * Dh, R, std=R ** -0.5, seed=2, dtype=dtype), _rand(Hk * Dh, R, std=R ** -0.5, seed=3, dtype=dtype),
                  _rand(H * Dh, seed=4, dtype=dtype))
    pos = torch.arange(T + start + B, device="cuda", dtype=torch.float32)
    ang = pos[:, None] * (1.0 / (10000.0 ** (torch.arange(0, 64, device="cuda", dtype=torch.float32) / 64)))[None]
    cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)
    first = torch.arange(B, device="cuda", dtype=torch.int32) + start            # every row of the batch starts elsewhere
    q = torch.zeros(B, T, H, Dh, device="cuda", dtype=dtype)
    k = torch.zeros(B, T + start + 1, Hk, Dh, device="cuda", dtype=dtype)       # too short for the later rows: dropped
    hip_ops.lowrank_expand_heads_multi([dict(p=p[..., :R], u=qu, num_heads=H, out=q, rotate=True, bias=bq),
                                        dict(p=p[..., R:], u=ku, num_heads=Hk, out=k, rotate=True, dst_by_position=True)],
                                       head_dim=Dh, cos=cos, sin=sin, positions=first)
    form = form_taken()
    for b in range(B):
        s0 = start + b
        c, s = cos[s0:s0 + T, None], sin[s0:s0 + T, None]

        def rope(x):
            x0, x1 = x[..., :64], x[..., 64:]
            return torch.cat([x0 * c - x1 * s, x1 * c + x0 * s], -1)

        ref_q = rope((p[b, :, :R].float() @ qu.float().t() + bq.float()).to(dtype).view(T, H, Dh))
        _check(q[b], ref_q, f"q of row {b}")
        ref_k = rope((p[b, :, R:].float() @ ku.float().t()).to(dtype).view(T, Hk, Dh))
        n = min(T, k.shape[1] - s0)
        _check(k[b, s0:s0 + n], ref_k[:n], f"k of row {b}")
        assert not k[b, :s0].any()
    return form


# ---- the three forms of the 256 x 256 kernel by name: shapes that the rules of the dispatch leave to it
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,N,K", [(3000, 3083, 128), (3500, 4097, 192)])
def test_linear_with_a_column_tail(B, N, K, dtype):
    """N off the grid of eight, in an output and from a residual whose rows are on the 16-byte grid."""
    from flashsvd_amd import hip_ops
    x, w, bias = _rand(B, K, seed=1, dtype=dtype), _rand(N, K, std=K ** -0.5, seed=2, dtype=dtype), _rand(N, seed=3, dtype=dtype)
    ld = (N + 15) // 8 * 8
    out, res = torch.full((B, ld), 7.0, device="cuda", dtype=dtype), _rand(B, ld, seed=4, dtype=dtype)[:, :N]
    ref = x.float() @ w.float().t()
    hip_ops.linear(x, w, out=out[:, :N])
    assert form_taken() == "256 x 256"
    _check(out[:, :N], ref.to(dtype), "plain")
    hip_ops.linear(x, w, bias, residual=res, out=out[:, :N])
    assert form_taken() == "256 x 256"
    _check(out[:, :N], ((ref + bias.float()).to(dtype).float() + res.float()).to(dtype), "bias and residual")
    assert bool((out[:, N:] == 7).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,D,R", [(1100, 11000, 128), (1101, 11003, 192), (4100, 11008, 64)])
def test_pair_form(B, D, R, dtype):
    """One and several tiles per workgroup, whole and partial column groups."""
    from flashsvd_amd import hip_ops
    p = _rand(B, 2 * R, seed=1, dtype=dtype)
    gu, uu = _rand(D, R, std=R ** -0.5, seed=2, dtype=dtype), _rand(D, R, std=R ** -0.5, seed=3, dtype=dtype)
    out = torch.full((B, (D + 15) // 8 * 8), 7.0, device="cuda", dtype=dtype)
    hip_ops.swiglu_linear(p, gu, uu, up_off=R, out=out[:, :D])
    assert form_taken() == "256 x 256 pair"
    g, u = p[:, :R].float() @ gu.float().t(), p[:, R:].float() @ uu.float().t()
    _check(out[:, :D], torch.nn.functional.silu(g.to(dtype)) * u.to(dtype), "pair")
    assert bool((out[:, D:] == 7).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,H,Hk,R", [(1, 2049, 39, 1, 192), (3, 700, 40, 3, 128), (4, 1025, 33, 9, 128)])
def test_heads_form(B, T, H, Hk, R, dtype):
    """Odd head counts (half a tile past the last head), partial row tiles, row tiles across sequences, dropped rows."""
    assert _expand_and_compare(B, T, H, Hk, R, dtype) == "256 x 256 heads"
