"""Head expansion of a batch of decoded tokens (three and more) on the matrix cores: rotation, append and the bounds of the
cache against the CPU oracle at the edges of its batch tiles (16, 32 tokens), chunks of the rank and forms."""
import pytest
import torch

from oracle import flashsvd_oracle as O
from tests.util import assert_close_bf16, bounds, rand_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rope", [True, False])
@pytest.mark.parametrize("B,H,Hk,Dh,Rq,Rk,Rv", [
    (3, 4, 2, 128, 64, 128, 192), (16, 2, 2, 64, 576, 64, 64), (17, 4, 4, 128, 1024, 1024, 512), (32, 2, 1, 64, 64, 64, 64),
    (33, 2, 2, 128, 128, 64, 64), (5, 2, 2, 128, 52, 33, 100), (70, 4, 2, 128, 65, 64, 1), (4, 2, 2, 64, 100, 100, 100)])
def test_qkv_batch(B, H, Hk, Dh, Rq, Rk, Rv, rope):
    from flashsvd_amd import hip_ops
    S = 50
    p = rand_bf16(B, Rq + Rk + Rv, seed=1)
    qu, ku, vu = (rand_bf16(h * Dh, r, std=r ** -0.5, seed=2 + i) for i, (h, r) in enumerate(((H, Rq), (Hk, Rk), (Hk, Rv))))
    cos, sin = O.rope_tables(S, Dh, dtype=torch.bfloat16)
    pos = torch.tensor([(7 * b + 5) % S for b in range(B)], dtype=torch.int32)
    pos[1] = S                                           # outside the cache: q is produced, k and v are dropped
    kc = torch.zeros(B, S, Hk, Dh, dtype=torch.bfloat16, device="cuda")
    vc = torch.zeros_like(kc)
    q = hip_ops.qkv_rope_append(p.cuda(), qu.cuda(), ku.cuda(), vu.cuda(), cos.cuda() if rope else None, sin.cuda() if rope else None,
                                pos.cuda(), kc, vc, num_heads=H, num_kv_heads=Hk, head_dim=Dh)
    pq, pk, pv = p[:, :Rq], p[:, Rq:Rq + Rk], p[:, Rq + Rk:]
    at = pos.clamp(max=S - 1).long()
    rot = (lambda x: O.apply_rope(x, cos[at][:, None], sin[at][:, None])) if rope else (lambda x: x)
    ref_q = rot(O.lin(pq, qu).view(B, H, Dh))
    ref_k, ref_v = rot(O.lin(pk, ku).view(B, Hk, Dh)), O.lin(pv, vu).view(B, Hk, Dh)
    assert_close_bf16(q, ref_q, "q", **bounds(ref_q))
    kc, vc = kc.cpu(), vc.cpu()
    kept = [b for b in range(B) if b != 1]
    assert_close_bf16(kc[kept, at[kept]], ref_k[kept], "k rows", **bounds(ref_k))
    assert_close_bf16(vc[kept, at[kept]], ref_v[kept], "v rows", **bounds(ref_v))
    for b in kept:
        kc[b, at[b]] = 0
        vc[b, at[b]] = 0
    assert not kc.any() and not vc.any()                 # nothing else in the caches was touched
