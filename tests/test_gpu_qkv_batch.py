"""Head expansion of a batch of decoded tokens (three and more) on the matrix cores: rotation, append and the bounds of the
cache against the CPU oracle at the edges of its batch tiles (16, 32 tokens), chunks of the rank and forms."""
import pytest
import torch

from oracle import flashsvd_oracle as O
from tests.util import assert_close_bf16, bounds, form_taken, rand_bf16

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


@pytest.mark.parametrize("B,H,Hk,Dh,R,form", [
    (3, 4, 2, 128, 64, "stream q k v"), (17, 4, 4, 64, 576, "stream q k v"), (33, 2, 2, 128, 128, "ring 64 x 128 heads"),
    (5, 2, 2, 128, 65, "tiles 64 x 128 heads"), (4, 2, 2, 64, 100, "vector q k v")])
def test_qkv_batch_float16(B, H, Hk, Dh, R, form):
    from flashsvd_amd import hip_ops
    from tests.test_gpu_ragged import _close16, _rand16
    S = 50
    p = _rand16(B, 3 * R, seed=1)
    qu, ku, vu = (_rand16(h * Dh, R, std=R ** -0.5, seed=2 + i) for i, h in enumerate((H, Hk, Hk)))
    cos, sin = O.rope_tables(S, Dh, dtype=torch.float16)
    pos = torch.tensor([(7 * b + 5) % S for b in range(B)], dtype=torch.int32)
    kc, vc = (torch.zeros(B, S, Hk, Dh, dtype=torch.float16, device="cuda") for _ in range(2))
    q = hip_ops.qkv_rope_append(p.cuda(), qu.cuda(), ku.cuda(), vu.cuda(), cos.cuda(), sin.cuda(), pos.cuda(), kc, vc,
                                num_heads=H, num_kv_heads=Hk, head_dim=Dh)
    assert form_taken() == form
    at, rows = pos.long(), torch.arange(B)
    rot = lambda x: O.apply_rope(x, cos[at][:, None], sin[at][:, None])
    _close16(q, rot(O.lin(p[:, :R], qu).view(B, H, Dh)), "q")
    _close16(kc.cpu()[rows, at], rot(O.lin(p[:, R:2 * R], ku).view(B, Hk, Dh)), "k rows")
    _close16(vc.cpu()[rows, at], O.lin(p[:, 2 * R:], vu).view(B, Hk, Dh), "v rows")
