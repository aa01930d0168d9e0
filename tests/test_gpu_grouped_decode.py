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
