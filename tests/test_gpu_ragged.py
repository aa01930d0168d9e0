"""Projections and head expansions whose rank or row length is no multiple of the matrix-core steps, or whose rows start
off the 16-byte grid (three rows and more): edges of K steps (one element below and above a multiple of 64, less than one
step), of row and column tiles, K split over workgroups, against the CPU oracle."""
import pytest
import torch

from oracle import flashsvd_oracle as O
from tests.util import assert_close_bf16, bounds, form_taken, rand_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N,K", [(3, 17, 1), (3, 64, 7), (5, 130, 63), (16, 100, 65), (40, 515, 1492), (127, 33, 2049), (128, 65, 63),
                                   (130, 129, 1638), (129, 4100, 1025), (300, 257, 96), (1030, 4096, 130)])
def test_linear_any_k(B, N, K):
    from flashsvd_amd import hip_ops
    x, w = rand_bf16(B, K, seed=1), rand_bf16(N, K, std=K ** -0.5, seed=2)
    res, bias = rand_bf16(B, N, seed=3), rand_bf16(N, seed=4)
    y = hip_ops.linear(x.cuda(), w.cuda(), bias.cuda(), residual=res.cuda())
    ref = res + O.lin(x, w, bias)
    assert_close_bf16(y, ref, f"linear {B}x{N}x{K}", **bounds(ref))


@pytest.mark.parametrize("off", [1, 2, 4])
@pytest.mark.parametrize("B", [4, 200])
def test_linear_rows_off_the_grid(B, off):
    """K is a whole number of steps, the rows of x and W start ``off`` elements past a 16-byte boundary."""
    from flashsvd_amd import hip_ops
    x, w = rand_bf16(B, 136, seed=1).cuda(), rand_bf16(96, 136, std=0.1, seed=2).cuda()
    y = hip_ops.linear(x[:, off:off + 128], w[:, off:off + 128])
    assert_close_bf16(y, O.lin(x[:, off:off + 128].cpu(), w[:, off:off + 128].cpu()), f"offset {off}")


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("B,D,R", [(3, 100, 52), (33, 1376, 375), (128, 130, 1), (200, 688, 100), (1040, 8200, 67)])
def test_swiglu_any_rank(B, D, R, mode):
    from flashsvd_amd import hip_ops
    p = rand_bf16(B, 2 * R, seed=1)
    gu, uu = rand_bf16(D, R, std=R ** -0.5, seed=2), rand_bf16(D, R, std=R ** -0.5, seed=3)
    h = hip_ops.swiglu_linear(p.cuda(), gu.cuda(), uu.cuda(), up_off=R, mode=mode)
    g, u = p[:, :R].float() @ gu.float().t(), p[:, R:].float() @ uu.float().t()
    if mode == 0:
        ref = torch.nn.functional.silu(g.to(torch.bfloat16)) * u.to(torch.bfloat16)
    else:
        ref = ((g * torch.sigmoid(g)) * u).to(torch.bfloat16)
    assert_close_bf16(h, ref, f"swiglu {B}x{D}x{R}", **bounds(ref))


@pytest.mark.parametrize("B,T,R", [(1, 16, 1), (2, 37, 52), (1, 130, 1638), (2, 333, 65), (1, 1, 52), (1, 15, 52), (3, 4, 65)])
def test_head_expansion_any_rank(B, T, R):
    """q with the rotation and v without, as one launch and as two, at positions behind a cached prefix."""
    from flashsvd_amd import hip_ops
    H, Hk, Dh = 4, 2, 128
    p = rand_bf16(B, T, 2 * R, seed=1)
    qu, vu = rand_bf16(H * Dh, R, std=R ** -0.5, seed=2), rand_bf16(Hk * Dh, R, std=R ** -0.5, seed=3)
    cos, sin = O.rope_tables(T + 9, Dh, dtype=torch.bfloat16)
    pos = torch.full((B,), 9, dtype=torch.int32)
    q = torch.zeros(B, T, H, Dh, dtype=torch.bfloat16, device="cuda")
    v = torch.zeros(B, T + 9, Hk, Dh, dtype=torch.bfloat16, device="cuda")
    pc = p.cuda()
    items = [dict(p=pc[..., :R], u=qu.cuda(), num_heads=H, out=q, rotate=True),
             dict(p=pc[..., R:], u=vu.cuda(), num_heads=Hk, out=v, dst_by_position=True)]
    kw = dict(head_dim=Dh, cos=cos.cuda(), sin=sin.cuda(), positions=pos.cuda())
    hip_ops.lowrank_expand_heads_multi(items, **kw)
    ref_q = O.apply_rope(O.lin(p[..., :R], qu).view(B, T, H, Dh), cos[9:, None], sin[9:, None])
    ref_v = O.lin(p[..., R:], vu).view(B, T, Hk, Dh)
    assert_close_bf16(q, ref_q, "q", **bounds(ref_q))
    assert_close_bf16(v[:, 9:], ref_v, "v", **bounds(ref_v))
    q2 = torch.zeros_like(q)
    hip_ops.lowrank_expand_heads(pc[..., :R], qu.cuda(), num_heads=H, out=q2, **kw)
    assert torch.equal(q, q2)


# pairs and single matrices of 3 to 500 rows, from less than one K step to a long K; every form that ragged rows take
_INDEPENDENT = [("pair", 4, 11008, 1492), ("pair", 40, 5504, 746), ("pair", 20, 2048, 1001), ("pair", 130, 1376, 375),
                ("single", 5, 1492, 4104), ("single", 30, 100, 4000), ("single", 40, 1536, 4100), ("single", 100, 515, 1492),
                ("single", 128, 1000, 2050), ("single", 200, 300, 8200), ("single", 500, 1492, 4104)]


def _ragged_call(kind, B, N, K, seed):
    from flashsvd_amd import hip_ops
    if kind == "pair":
        p, gu, uu = rand_bf16(B, 2 * K, seed=seed).cuda(), rand_bf16(N, K, std=K ** -0.5, seed=seed + 1).cuda(), rand_bf16(N, K, std=K ** -0.5, seed=seed + 2).cuda()
        return lambda: hip_ops.swiglu_linear(p, gu, uu, up_off=K)
    x, w = rand_bf16(B, K, seed=seed).cuda(), rand_bf16(N, K, std=K ** -0.5, seed=seed + 1).cuda()
    return lambda: hip_ops.linear(x, w)


@pytest.mark.parametrize("kind,B,N,K", _INDEPENDENT)
def test_ragged_rows_leave_the_shared_workspace_alone(kind, B, N, K):
    """One workspace serves a device, so whatever uses it is bound to one stream; ragged rows do not use it."""
    from flashsvd_amd import hip_ops
    assert hip_ops.ensure_split_workspace(torch.device("cuda", 0))
    ws = hip_ops._SPLIT_WS[0]
    call = _ragged_call(kind, B, N, K, seed=1)
    torch.cuda.synchronize()
    partials = ws[64 << 10:]                            # behind the arrival counters, which are zero between calls
    partials.fill_(0x5a)
    call()
    torch.cuda.synchronize()
    untouched, at_rest = int((partials != 0x5a).sum()) == 0, int(ws[:64 << 10].sum()) == 0
    assert untouched and at_rest


def test_ragged_rows_on_two_streams():
    """The same projections issued on two streams at once give the bits that each gives alone."""
    calls = [_ragged_call(*c, seed=10 * i) for i, c in enumerate(_INDEPENDENT)]
    alone = [c() for c in calls]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(5):
        got = [[], []]
        for i in range(len(calls)):
            for s, st in enumerate(streams):            # the two streams are at different calls at any time
                with torch.cuda.stream(st):
                    j = (i + s * 3) % len(calls)
                    got[s].append((j, calls[j]()))
        torch.cuda.synchronize()
        for s in range(2):
            for j, y in got[s]:
                assert torch.equal(y, alone[j]), f"{_INDEPENDENT[j]} on stream {s}"


def _rand16(*shape, std=1.0, seed=0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed), dtype=torch.float32) * std).to(torch.float16)


def _close16(got, ref, what):
    """A quarter of the bf16 bounds: float16 has three more mantissa bits (two of its ulps where max|ref| is 2 and more)."""
    m = float(ref.float().abs().max())
    assert got.dtype == torch.float16
    assert_close_bf16(got, ref, what, abs_tol=5e-3 if m < 2.0 else 2.0 * m * 2.0 ** -10, rel_tol=2.5e-3)


@pytest.mark.parametrize("B,N,K,form", [
    (16, 4097, 1492, "any rows 16"), (31, 4097, 1003, "any rows 16"), (12, 8200, 333, "any rows 32 x 64"), (100, 3970, 1492, "any rows 32 x 64"),
    (500, 4097, 333, "any rows 64 x 64"), (1030, 4096, 130, "any rows 128 x 128")])
def test_linear_forms(B, N, K, form):
    """Every form that ragged rows of a single matrix take, in both element types."""
    from flashsvd_amd import hip_ops
    for rand, close in ((rand_bf16, lambda y, r, w: assert_close_bf16(y, r, w, **bounds(r))), (_rand16, _close16)):
        x, w, bias, res = rand(B, K, seed=1), rand(N, K, std=K ** -0.5, seed=2), rand(N, seed=3), rand(B, N, seed=4)
        y = hip_ops.linear(x.cuda(), w.cuda(), bias.cuda(), residual=res.cuda())
        assert form_taken() == form
        close(y, res + O.lin(x, w, bias), form)


@pytest.mark.parametrize("B,D,R,form", [
    (16, 1000, 517, "any rows 16 pair"), (30, 4090, 517, "any rows 16 pair"), (33, 1000, 517, "any rows 32 x 64 pair"), (5, 5000, 130, "any rows 32 x 64 pair"),
    (200, 4090, 67, "any rows 64 x 64 pair"), (1040, 8200, 67, "any rows 128 x 128 pair")])
def test_pair_forms(B, D, R, form):
    from flashsvd_amd import hip_ops
    for rand, close in ((rand_bf16, lambda y, r, w: assert_close_bf16(y, r, w, **bounds(r))), (_rand16, _close16)):
        p, gu, uu = rand(B, 2 * R, seed=1), rand(D, R, std=R ** -0.5, seed=2), rand(D, R, std=R ** -0.5, seed=3)
        g, u = p[:, :R].float() @ gu.float().t(), p[:, R:].float() @ uu.float().t()
        for mode in (0, 1):
            ref = torch.nn.functional.silu(g.to(p.dtype)) * u.to(p.dtype) if mode == 0 else ((g * torch.sigmoid(g)) * u).to(p.dtype)
            h = hip_ops.swiglu_linear(p.cuda(), gu.cuda(), uu.cuda(), up_off=R, mode=mode)
            assert form_taken() == form
            close(h, ref, f"{form}, mode {mode}")


@pytest.mark.parametrize("B,K", [(3, 33), (5, 262), (40, 1001), (150, 100), (9, 4104)])
def test_norm_in_front_of_a_ragged_projection(B, K):
    """RMSNorm with its own rounding in front of a projection whose K is no multiple of 32."""
    from flashsvd_amd import hip_ops
    for rand, close in ((rand_bf16, lambda y, r, w: assert_close_bf16(y, r, w, **bounds(r))), (_rand16, _close16)):
        x, w, nw = rand(B, K, seed=1), rand(300, K, std=K ** -0.5, seed=2), rand(K, seed=3) * 0.1 + 1
        y = hip_ops.linear(x.cuda(), w.cuda(), norm_weight=nw.cuda(), eps=1e-6)
        close(y, O.lin(O.rms_norm(x, nw, 1e-6), w), f"{B} x {K}")


def test_longest_rows():
    """K past what the vector kernels stage in LDS."""
    from flashsvd_amd import hip_ops
    x, w = rand_bf16(3, 33001, seed=1), rand_bf16(20, 33001, std=33001 ** -0.5, seed=2)
    ref = O.lin(x, w)
    assert_close_bf16(hip_ops.linear(x.cuda(), w.cuda()), ref, "linear", **bounds(ref))


@pytest.mark.parametrize("B,T,R", [(2, 37, 52), (1, 333, 65)])
def test_head_expansion_any_rank_float16(B, T, R):
    from flashsvd_amd import hip_ops
    H, Hk, Dh = 4, 2, 128
    p, qu, vu = _rand16(B, T, 2 * R, seed=1), _rand16(H * Dh, R, std=R ** -0.5, seed=2), _rand16(Hk * Dh, R, std=R ** -0.5, seed=3)
    cos, sin = O.rope_tables(T + 9, Dh, dtype=torch.float16)
    q, v = torch.zeros(B, T, H, Dh, dtype=torch.float16, device="cuda"), torch.zeros(B, T + 9, Hk, Dh, dtype=torch.float16, device="cuda")
    pc = p.cuda()
    hip_ops.lowrank_expand_heads_multi([dict(p=pc[..., :R], u=qu.cuda(), num_heads=H, out=q, rotate=True),
                                        dict(p=pc[..., R:], u=vu.cuda(), num_heads=Hk, out=v, dst_by_position=True)],
                                       head_dim=Dh, cos=cos.cuda(), sin=sin.cuda(), positions=torch.full((B,), 9, dtype=torch.int32, device="cuda"))
    assert form_taken() == "tiles 64 x 128 heads"
    _close16(q, O.apply_rope(O.lin(p[..., :R], qu).view(B, T, H, Dh), cos[9:, None], sin[9:, None]), "q")
    _close16(v[:, 9:], O.lin(p[..., R:], vu).view(B, T, Hk, Dh), "v")
