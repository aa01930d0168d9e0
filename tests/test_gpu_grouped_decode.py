"""Decode attention over grouped-query caches, four and two query heads per workgroup (512 workgroups and more): key ranges
around a pass of 128 keys, several passes, sequences without keys, splits without keys, more splits than one round of the
merge loads, one workspace for calls that group differently."""
import pytest
import torch

from tests.util import assert_close_bf16, rand_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from flashsvd_amd import hip_ops
    return hip_ops


def _reference(q, kc, vc, n):
    """softmax(q k^T / sqrt(Dh)) v of one sequence in float64 on the CPU."""
    H, Dh = q.shape
    rep = H // kc.shape[1]
    k, v = (t[:n].double().repeat_interleave(rep, 1) for t in (kc, vc))
    w = torch.softmax(torch.einsum("hd,khd->hk", q.double(), k) / Dh ** 0.5, -1)
    return torch.einsum("hk,khd->hd", w, v)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Hk,nsplit,lens", [(64, 32, 8, 1, (1, 127, 128, 129, 255, 256, 257, 0)), (32, 32, 16, 1, (16, 130, 384, 385, 0)),
                                                (16, 32, 8, 4, (1, 64, 511, 512, 513, 900, 0)), (8, 32, 8, 9, (3, 143, 145, 1296, 0)),
                                                (4, 32, 16, 17, (1, 16, 17, 273, 0))])
def test_grouped_decode_attention(ops, dtype, B, H, Hk, nsplit, lens):
    S = max(lens) + 3
    q, kc, vc = (rand_bf16(*shape, seed=i).to(dtype) for i, shape in enumerate(((B, H, 128), (B, S, Hk, 128), (B, S, Hk, 128))))
    lens = torch.tensor([lens[b % len(lens)] for b in range(B)], dtype=torch.int32)
    qd, kd, vd, ld = (t.cuda() for t in (q, kc, vc, lens))
    ws = ops.attn_workspace(B, H, 128, max(nsplit, 2), "cuda")
    out = ops.attn_decode_densekv(qd, kd, vd, ld, nsplit=nsplit, workspace=ws)
    few = ops.attn_decode_densekv(qd[:1], kd[:1], vd[:1], ld[:1], nsplit=nsplit, workspace=ws)        # one head per workgroup
    again = ops.attn_decode_densekv(qd, kd, vd, ld, nsplit=nsplit, workspace=ws)
    assert torch.equal(out, again)
    assert_close_bf16(few[0], _reference(q[0], kc[0], vc[0], int(lens[0])), "one sequence")
    for b in range(min(B, 8)):
        n = int(lens[b])
        if n:
            assert_close_bf16(out[b], _reference(q[b], kc[b], vc[b], n), f"sequence {b}, {n} keys")
        else:
            assert torch.all(out[b] == 0)


def _pair_of_caches(B, S, Hk, Dh, dtype):
    """The same values with the rows of a token together (a workgroup may append its own row) and with the rows of a head
    together (the append is a launch of its own)."""
    kc, vc = (rand_bf16(B, S, Hk, Dh, seed=i).to(dtype).cuda() for i in (3, 4))
    return (kc, vc), tuple(t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for t in (kc, vc))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Hk,Dh,nsplit,lens", [(2, 8, 8, 128, 1, (0, 128)), (3, 16, 16, 128, 4, (63, 64, 300)), (16, 32, 8, 128, 4, (0, 1, 127, 128, 511, 512, 400)),
                                                   (64, 32, 8, 128, 1, (0, 15, 128, 255)), (16, 32, 16, 128, 2, (31, 32, 33, 256)), (32, 16, 2, 128, 4, (5, 64, 130)),
                                                   (1, 32, 8, 128, 3, (47,)),
                                                   # four heads of 64 per workgroup, which append in the launch; eight per kv head, which do not; one
                                                   (64, 32, 8, 64, 1, (0, 31, 32, 127, 128, 255)), (16, 32, 8, 64, 4, (0, 1, 127, 128, 256, 511, 512, 400)),
                                                   (32, 16, 2, 64, 4, (5, 64, 130)), (3, 8, 8, 64, 2, (63, 64, 300))])
@pytest.mark.parametrize("rotate", [True, False])
def test_append_in_the_attention_launch(ops, dtype, B, H, Hk, Dh, nsplit, lens, rotate):
    """New rows at split and pass borders, at the first and the last row of the cache and past its end (dropped): the caches
    and results are those of an append launched before the attention, bit for bit."""
    S = max(lens) + 1
    lens = torch.tensor([lens[b % len(lens)] for b in range(B)], dtype=torch.int32)
    if B > 2:
        lens[-1] = S                                            # no room: nothing is written, all S rows are attended to
    cos, sin = (rand_bf16(S + 1, Dh // 2, seed=i).to(dtype).cuda() for i in (6, 7)) if rotate else (None, None)
    q, kn, vn = (rand_bf16(B, h, Dh, seed=i).to(dtype).cuda() for i, h in ((0, H), (1, Hk), (2, Hk)))
    results = []
    for kc, vc in _pair_of_caches(B, S, Hk, Dh, dtype):
        for _ in range(2):                                      # a second call finds the row there already
            out = ops.attn_decode_densekv(q, kc, vc, lens.cuda(), k_new=kn, v_new=vn, cos=cos, sin=sin, nsplit=nsplit)
        results.append((out, kc, vc))
    for got, want in zip(*results):
        assert torch.equal(got, want)
    if not rotate:
        for b in range(min(B, 4)):
            n = min(int(lens[b]) + 1, S)
            if lens[b] < S:
                assert torch.equal(results[0][1][b, n - 1], kn[b]) and torch.equal(results[0][2][b, n - 1], vn[b])
            kc, vc = (t[b].cpu() for t in results[0][1:])
            assert_close_bf16(results[0][0][b], _reference(q[b].cpu(), kc, vc, n), f"sequence {b}")


def test_sequences_bound_to_one_cache_row_see_each_other(ops):
    """Three tokens of one sequence as three batch rows over one cache: each attends to the rows that the others append."""
    H, S, n = 8, 64, 20
    kc, vc = (rand_bf16(1, S, H, 128, seed=i).cuda() for i in (3, 4))
    q, kn, vn = (rand_bf16(3, H, 128, seed=i).cuda() for i in (0, 1, 2))
    lens = torch.tensor([n, n + 1, n + 2], dtype=torch.int32).cuda()
    out = ops.attn_decode_densekv(q, kc.expand(3, S, H, 128), vc.expand(3, S, H, 128), lens, k_new=kn, v_new=vn, nsplit=2)
    assert torch.equal(kc[0, n:n + 3], kn) and torch.equal(vc[0, n:n + 3], vn)
    for b in range(3):
        assert_close_bf16(out[b], _reference(q[b].cpu(), kc[0].cpu(), vc[0].cpu(), n + 1 + b), f"token {b}")
