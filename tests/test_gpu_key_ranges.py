"""Decode attention: the key ranges follow each sequence's length, whatever the split that the scratch was sized for."""
import pytest
import torch

from tests.util import assert_close_bf16, rand_bf16

pytestmark = pytest.mark.gpu


def _reference(q, kc, vc, n):
    """softmax(q k^T / sqrt(Dh)) v of one sequence in float64 on the CPU."""
    H, Dh = q.shape
    k, v = (t[:n].double().repeat_interleave(H // kc.shape[1], 1) for t in (kc, vc))
    w = torch.softmax(torch.einsum("hd,khd->hk", q.double(), k) / Dh ** 0.5, -1)
    return torch.einsum("hk,khd->hd", w, v)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Hk,Dh,nsplit,lens", [
    (1, 8, 8, 128, 40, (128,)), (1, 8, 8, 128, 40, (129,)), (2, 5, 5, 64, 7, (255, 700)), (3, 8, 2, 128, 5, (0, 1, 641)),  # one pass and more
    (8, 32, 32, 128, 8, (511, 512, 1023, 1024, 1535, 1536, 0, 1)), (8, 32, 32, 64, 2, (1024, 1100, 30)),                 # from 2 keys a pair
    (17, 16, 16, 128, 3, (1087, 1088, 64)), (64, 16, 16, 128, 2, (9, 300, 300, 17, 140)), (65, 8, 8, 128, 2, (300, 17)), (33, 9, 9, 64, 3, (593, 594, 595)),
    (48, 32, 32, 128, 2, (300, 17, 129)), (4, 12, 12, 128, 3, (300, 40)),                                                   # odd batches and heads, more than 1024 pairs
    # longest first, a group of heads per workgroup: around 1000 keys, alike and not, a last round that is not full, without ranges on more than one XCD, around 257 keys
    (16, 32, 8, 128, 4, (999, 1000, 1024, 3)), (14, 64, 8, 128, 2, (1000, 830, 999)), (14, 64, 8, 128, 2, (1024, 300, 0)), (5, 40, 8, 128, 10, (1001, 1, 130)),
    (36, 32, 4, 128, 1, (1100, 9, 300)), (36, 32, 4, 128, 1, (999, 9, 300)), (40, 32, 8, 128, 1, (257, 20, 90)), (40, 32, 8, 128, 1, (256, 20, 90)),
    (64, 32, 8, 64, 1, (1, 31, 32, 127, 128, 129, 0, 300)), (16, 32, 8, 64, 4, (511, 512, 513, 40, 0)), (4, 64, 8, 64, 9, (3, 1160))])  # groups of 64
def test_ranges_follow_the_length(dtype, B, H, Hk, Dh, nsplit, lens):
    from flashsvd_amd import hip_ops as ops
    S = max(lens) + 5
    q, kc, vc = (rand_bf16(*shape, seed=i).to(dtype) for i, shape in enumerate(((B, H, Dh), (B, S, Hk, Dh), (B, S, Hk, Dh))))
    n = torch.tensor([lens[b % len(lens)] for b in range(B)], dtype=torch.int32)
    qd, kd, vd, nd = (t.cuda() for t in (q, kc, vc, n))
    ws = ops.attn_workspace(B, H, Dh, nsplit, "cuda")
    out = ops.attn_decode_densekv(qd, kd, vd, nd, nsplit=nsplit, workspace=ws)
    other = ops.attn_decode_densekv(qd, kd, vd, nd.flip(0), nsplit=nsplit, workspace=ws)        # other ranges over the same scratch
    assert torch.equal(out, ops.attn_decode_densekv(qd, kd, vd, nd, nsplit=nsplit, workspace=ws))
    for got, length in ((out, n), (other, n.flip(0))):
        for b in range(B):
            if int(length[b]):
                assert_close_bf16(got[b], _reference(q[b], kc[b], vc[b], int(length[b])), f"sequence {b}, {int(length[b])} keys")
            else:
                assert torch.all(got[b] == 0)
