"""GPU parity of the rank-space KV-cache decode attention (MFMA K rebuild, rank-space V accumulation)
against the CPU oracle's streaming decode; bf16 within max-abs 2e-2 / max-rel 1e-2."""
import pytest
import torch

from oracle import flashsvd_oracle as O
from tests.util import assert_close_bf16, model_from_oracle, rand_bf16

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def RD():
    assert torch.cuda.is_available()
    from flashsvd_amd.kernels import rank_decode
    return rank_decode


def _lin_layout(V):   # [heads,R,Dh] -> nn.Linear weight [heads*Dh, R]
    h, r, d = V.shape
    return V.transpose(1, 2).reshape(h * d, r).contiguous()


CASES = [(1, 32, 32, 512, 560, 1024, 1024, None), (1, 32, 32, 512, 560, 1024, 1024, 1), (2, 8, 2, 100, 128, 72, 40, 3),
         (3, 4, 4, 1, 64, 64, 64, 2), (2, 16, 4, 333, 400, 1664, 1664, 4), (1, 2, 2, 65, 80, 8, 2048, None),
         # long splits take the 2- and 4-sub-tile variants of stage 1 (ragged tails, MHA and 2 query heads per kv head)
         (2, 8, 4, 700, 720, 136, 264, 2), (2, 4, 4, 450, 500, 200, 72, 2), (1, 4, 4, 1500, 1536, 64, 64, 1)]


@pytest.mark.parametrize("B,H,Hk,L,S,Rk,Rv,nsplit", CASES)
def test_rank_decode_vs_oracle(RD, B, H, Hk, L, S, Rk, Rv, nsplit):
    Dh = 128
    cos, sin = O.rope_tables(S, Dh, dtype=BF16)
    q = rand_bf16(B, H, Dh, seed=1)
    Pk, Pv = rand_bf16(B, S, Rk, seed=2), rand_bf16(B, S, Rv, seed=3)
    Vk, Vv = rand_bf16(Hk, Rk, Dh, std=Rk ** -0.5, seed=4), rand_bf16(Hk, Rv, Dh, std=Rv ** -0.5, seed=5)
    lens = torch.tensor([max(1, L - 17 * b) for b in range(B)], dtype=torch.int32)
    out = RD.rank_decode(q.cuda(), Pk.cuda(), Pv.cuda(), _lin_layout(Vk).cuda(), _lin_layout(Vv).cuda(), cos.cuda(), sin.cuda(),
                         lens.cuda(), num_kv_heads=Hk, nsplit=nsplit)
    for b in range(B):
        n = int(lens[b])
        ref = O.rank_decode_attn(q[b:b + 1], Pk[b:b + 1, :n], Pv[b:b + 1, :n], Vk, Vv, cos[:n], sin[:n])
        assert_close_bf16(out[b:b + 1], ref, f"b={b} n={n}")
    # equals dense decode on the reconstructed cache (the reference's own --check)
    K = O.apply_rope_fp32(torch.einsum("blr,krd->blkd", Pk.float(), Vk.float()), cos[None, :, None], sin[None, :, None])
    V = torch.einsum("blr,krd->blkd", Pv.float(), Vv.float())
    n = int(lens[0])
    assert_close_bf16(out[:1], O.dense_decode_attn(q[:1].float(), K[:1, :n], V[:1, :n]), "vs dense")


LONG_CASES = [  # B, H, Hk, S, Rk, Rv, nsplit: shared caches of 2^17 (head, key) pairs and more take the three-launch form
    (4, 32, 32, 8200, 192, 200, 2),     # one query head per kv head: two heads per workgroup share the Pk rows, four key sub-tiles per wave
    (4, 32, 8, 8200, 128, 64, 3),       # four query heads per kv head
    (4, 32, 16, 8200, 72, 136, 2),      # two query heads per kv head, ranks off the 64 grid (fragments straight from memory)
    (9, 16, 16, 7300, 64, 72, 5),       # 16 heads: one head tile; short last split
    (2, 32, 32, 2100, 128, 128, None),  # just above the size from which the form is taken; the wrapper's own split count
    (16, 8, 4, 1030, 64, 64, 2),        # 8 heads in a 16-head tile
    (4, 32, 32, 8200, 72, 72, 2),       # one query head per kv head, ranks off the 64 grid: one head per workgroup
    (12, 3, 3, 4000, 64, 64, 2),        # an odd number of heads: one head per workgroup, operands straight into LDS
]


@pytest.mark.parametrize("B,H,Hk,S,Rk,Rv,nsplit", LONG_CASES)
def test_long_cache_three_launch_form(RD, monkeypatch, B, H, Hk, S, Rk, Rv, nsplit):
    """Scores -> softmax -> rank-space accumulation per head tile (long caches shared by the heads, the call brings a score
    buffer) against the one-kernel form on the same inputs (same arithmetic up to the order of fp32 sums: one bf16 ulp) and
    against the oracle on sampled batch rows."""
    Dh = 128
    cos, sin = O.rope_tables(S, Dh, dtype=BF16)
    q = rand_bf16(B, H, Dh, seed=11)
    Pk, Pv = rand_bf16(B, S, Rk, seed=12), rand_bf16(B, S, Rv, seed=13)
    Vk, Vv = rand_bf16(Hk, Rk, Dh, std=Rk ** -0.5, seed=14), rand_bf16(Hk, Rv, Dh, std=Rv ** -0.5, seed=15)
    lens = torch.tensor([max(0, S - 5 - (S // (B + 1)) * b) for b in range(B)], dtype=torch.int32)
    lens[-1] = 0 if B > 4 else lens[-1]                 # an empty batch row in the widest case
    args = (q.cuda(), Pk.cuda(), Pv.cuda(), _lin_layout(Vk).cuda(), _lin_layout(Vv).cuda(), cos.cuda(), sin.cuda(), lens.cuda())
    # one-kernel form: the call brings no score buffer
    monkeypatch.setattr(RD, "_FORCE_ONE_KERNEL", True)
    one = RD.rank_decode(*args, num_kv_heads=Hk, nsplit=nsplit).float().cpu()
    monkeypatch.setattr(RD, "_FORCE_ONE_KERNEL", False)
    kept = []
    monkeypatch.setattr(RD, "_KEEP_SCORES", kept)
    three = RD.rank_decode(*args, num_kv_heads=Hk, nsplit=nsplit)
    torch.cuda.synchronize()
    # the call's score buffer now holds its softmax weights, [B,H,ld] words, per 8 keys four words of bf16 pairs hi(p) and
    # four of lo(p) = bf16(p - hi): the largest weight of a non-empty row is exp(0) in at least one split -- which proves
    # the form that ran
    assert len(kept) == 1 and kept[0] is not None
    ld = (S + 63) // 64 * 64
    w = kept[0][:B * H * ld].view(torch.int32).view(B, H, ld // 8, 2, 4)[0].cpu()
    n0 = int(lens[0])
    def pairs(x):                                       # [H, groups, 4] words -> [H, groups * 8] values
        lo16 = ((x & 0xffff) << 16).view(torch.float32)
        hi16 = (x & -65536).view(torch.float32)
        return torch.stack([lo16, hi16], dim=-1).reshape(x.shape[0], -1)
    p_hi, p_lo = pairs(w[:, :, 0].contiguous()), pairs(w[:, :, 1].contiguous())
    p = (p_hi + p_lo)[:, :n0]
    assert float(p.max(dim=-1).values.min()) == 1.0 and float(p.min()) >= 0.0
    assert float((p_hi + p_lo)[:, n0:(n0 + 63) // 64 * 64].abs().max() if n0 % 64 else 0.0) == 0.0   # the tail of the last block
    three = three.float().cpu()
    assert torch.isfinite(three).all()
    assert_close_bf16(three, one, "three-launch form vs one-kernel form", abs_tol=2e-3, rel_tol=1e-2)
    for b in (0, B - 1):
        n = int(lens[b])
        if n == 0:
            assert float(three[b].abs().max()) == 0.0 and float(one[b].abs().max()) == 0.0
            continue
        ref = O.rank_decode_attn(q[b:b + 1], Pk[b:b + 1, :n], Pv[b:b + 1, :n], Vk, Vv, cos[:n], sin[:n])
        assert_close_bf16(three[b:b + 1], ref, f"three-launch form, b={b} n={n}")


def test_score_buffer_follows_the_capacity_of_a_long_cache(RD, monkeypatch):
    """The scores of a call are indexed by cache position: a cache with room for 600 000 tokens takes a 77 MB score buffer
    whatever its fill.  The buffer belongs to the call; nothing registered with the library is involved."""
    from flashsvd_amd import hip_ops
    B, H, Hk, S, R, Dh, n = 1, 32, 32, 600_000, 64, 128, 3000
    dev = torch.device("cuda", torch.cuda.current_device())
    hip_ops.release_split_workspace(dev)
    cos, sin = O.rope_tables(n, Dh, dtype=BF16)
    q = rand_bf16(B, H, Dh, seed=21)
    Pk, Pv = rand_bf16(B, n, R, seed=22), rand_bf16(B, n, R, seed=23)
    Vk, Vv = rand_bf16(Hk, R, Dh, std=R ** -0.5, seed=24), rand_bf16(Hk, R, Dh, std=R ** -0.5, seed=25)
    pkc = torch.zeros(B, S, R, dtype=BF16, device="cuda")
    pvc = torch.zeros(B, S, R, dtype=BF16, device="cuda")
    pkc[:, :n], pvc[:, :n] = Pk.cuda(), Pv.cuda()
    lens = torch.tensor([n], dtype=torch.int32, device="cuda")
    kept = []
    monkeypatch.setattr(RD, "_KEEP_SCORES", kept)
    out = RD.rank_decode(q.cuda(), pkc, pvc, _lin_layout(Vk).cuda(), _lin_layout(Vv).cuda(), cos.cuda(), sin.cuda(), lens,
                         num_kv_heads=Hk, nsplit=4)
    assert len(kept) == 1 and kept[0].numel() == B * H * ((S + 63) // 64 * 64)
    assert dev.index not in hip_ops._SPLIT_WS
    ref = O.rank_decode_attn(q, Pk, Pv, Vk, Vv, cos, sin)
    assert_close_bf16(out, ref, "long-capacity cache")
    # the weights of the call sit in its buffer (row 0: head 0): the three-launch form ran
    assert int(kept[0][:64].view(torch.int32).abs().max()) != 0


def test_graph_and_eager_take_the_same_form(RD, monkeypatch):
    """Which form runs depends on the shape alone: a call captured into a HIP graph and the same call made eagerly give
    the same bits, replay after replay, and a second stream with its own call does not disturb them."""
    B, H, Hk, S, R, Dh = 4, 32, 32, 2048, 256, 128
    cos, sin = O.rope_tables(S, Dh, dtype=BF16)
    q = rand_bf16(B, H, Dh, seed=31).cuda()
    Pk, Pv = rand_bf16(B, S, R, seed=32).cuda(), rand_bf16(B, S, R, seed=33).cuda()
    Vk, Vv = rand_bf16(Hk, R, Dh, std=R ** -0.5, seed=34), rand_bf16(Hk, R, Dh, std=R ** -0.5, seed=35)
    ku, vu = _lin_layout(Vk).cuda(), _lin_layout(Vv).cuda()
    lens = torch.tensor([S - 3, S // 2, 700, 64], dtype=torch.int32, device="cuda")
    cosg, sing = cos.cuda(), sin.cuda()
    kept = []
    monkeypatch.setattr(RD, "_KEEP_SCORES", kept)
    eager = RD.rank_decode(q, Pk, Pv, ku, vu, cosg, sing, lens, num_kv_heads=Hk, nsplit=4).clone()
    assert kept[-1] is not None                       # this shape takes the three-launch form
    out = torch.empty_like(eager)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            RD.rank_decode(q, Pk, Pv, ku, vu, cosg, sing, lens, num_kv_heads=Hk, nsplit=4, out=out)
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        RD.rank_decode(q, Pk, Pv, ku, vu, cosg, sing, lens, num_kv_heads=Hk, nsplit=4, out=out)
    assert kept[-1] is not None                       # and so does the captured call
    for rep in range(3):
        out.zero_()
        g.replay()
        with torch.cuda.stream(side):                 # an eager call of another shape on another stream, its own buffers
            other = RD.rank_decode(q[:2], Pk[:2], Pv[:2], ku, vu, cosg, sing, lens[:2].contiguous(), num_kv_heads=Hk, nsplit=4)
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {rep} differs from the eager call"
        assert torch.equal(other, eager[:2])


def test_packed_api_shared_and_headwise(RD):
    B, H, Hk, L, R, Dh = 2, 8, 4, 150, 96, 128
    cos, sin = O.rope_tables(L, Dh, dtype=BF16)
    Pq = rand_bf16(B, H, R, seed=1)
    Pk, Pv = rand_bf16(B, L, R, seed=2), rand_bf16(B, L, R, seed=3)
    Vq, Vk, Vv = rand_bf16(H, R, Dh, std=0.1, seed=4), rand_bf16(Hk, R, Dh, std=0.1, seed=5), rand_bf16(Hk, R, Dh, std=0.1, seed=6)
    bq = rand_bf16(H, Dh, std=0.1, seed=7)
    g = lambda t: t.cuda()
    f = RD.DecodePackedFactors(Pq=g(Pq), Pk=g(Pk).unsqueeze(2).expand(B, L, Hk, R), Pv=g(Pv).unsqueeze(2).expand(B, L, Hk, R),
                               Vq=g(Vq), Vk=g(Vk), Vv=g(Vv), bq=g(bq))
    M = torch.empty(B, H, 3, device="cuda"); Lw = torch.empty_like(M); Acc = torch.empty(B, H, 3, R, device="cuda")
    o_ws = torch.empty(B, H, Dh, device="cuda", dtype=BF16)
    out = RD.flashsvd_attn_decode_packed(f, g(cos), g(sin), seqlen_k=L, causal=True, split_k=64, bn=64, br=64,
                                         workspace=(M, Lw, Acc), out=o_ws, pad_to_16=True, vk_resident=True)
    assert out.data_ptr() == o_ws.data_ptr()
    qd, _, _ = O.reconstruct_qkv_token(Pq, Pq[:, :1], Pq[:, :1], Vq, Vq[:1], Vq[:1], bq)
    qr = O.apply_rope_fp32(qd, cos[L - 1], sin[L - 1])
    ref = O.rank_decode_attn(qr, Pk, Pv, Vk, Vv, cos, sin)
    assert_close_bf16(out, ref, "packed shared")
    # shorter seqlen_k uses a prefix of the cache and rotates q at seqlen_k-1
    out2 = RD.flashsvd_attn_decode_packed_v1(f, g(cos), g(sin), seqlen_k=70)
    ref2 = O.rank_decode_attn(O.apply_rope_fp32(qd, cos[69], sin[69]), Pk[:, :70], Pv[:, :70], Vk, Vv, cos[:70], sin[:70])
    assert_close_bf16(out2, ref2, "seqlen_k prefix")
    # head-wise coefficients
    Pkh, Pvh = rand_bf16(B, L, Hk, R, seed=8), rand_bf16(B, L, Hk, R, seed=9)
    fh = RD.DecodePackedFactors(Pq=g(Pq), Pk=g(Pkh), Pv=g(Pvh), Vq=g(Vq), Vk=g(Vk), Vv=g(Vv), bq=g(bq))
    outh = RD.flashsvd_attn_decode_packed(fh, g(cos), g(sin), seqlen_k=L)
    refh = O.rank_decode_attn_headwise(qr, Pkh, Pvh, Vk, Vv, cos, sin)
    assert_close_bf16(outh, refh, "packed headwise")


@pytest.mark.parametrize("B,H,Hk,L,S,R", [(1, 32, 32, 512, 560, 1024), (2, 16, 4, 333, 400, 1664), (4, 8, 8, 130, 192, 192)])
def test_short_splits_repeat_bit_identically(RD, B, H, Hk, L, S, R):
    """Short splits stream k_u and Pk two chunks ahead into LDS rings guarded only by the wave's load counter and a bare
    barrier: a chunk read before it has landed, or a stage refilled while still being read, would show as a difference
    between calls."""
    Dh = 128
    cos, sin = O.rope_tables(S, Dh, dtype=BF16)
    q = rand_bf16(B, H, Dh, seed=1).cuda()
    Pk, Pv = rand_bf16(B, S, R, seed=2).cuda(), rand_bf16(B, S, R, seed=3).cuda()
    ku, vu = rand_bf16(Hk * Dh, R, std=R ** -0.5, seed=4).cuda(), rand_bf16(Hk * Dh, R, std=R ** -0.5, seed=5).cuda()
    lens = torch.tensor([max(1, L - 17 * b) for b in range(B)], dtype=torch.int32).cuda()
    first = RD.rank_decode(q, Pk, Pv, ku, vu, cos.cuda(), sin.cuda(), lens, num_kv_heads=Hk)
    for _ in range(20):
        assert torch.equal(RD.rank_decode(q, Pk, Pv, ku, vu, cos.cuda(), sin.cuda(), lens, num_kv_heads=Hk), first)


def test_rankkv_append_matches_index_copy(RD):
    B, S, Rk, Rv = 3, 40, 72, 136
    p = rand_bf16(B, 64 + Rk + Rv, seed=1).cuda()                       # coefficients as row slices of a wider buffer
    pkc, pvc = rand_bf16(B + 1, S, Rk, seed=2).cuda(), rand_bf16(B + 1, S, Rv, seed=3).cuda()
    ek, ev = pkc.clone(), pvc.clone()
    pos = torch.tensor([0, 39, 40], dtype=torch.int32).cuda()           # the last row is outside the cache: dropped
    RD.rankkv_append(p[:, 64:64 + Rk], p[:, 64 + Rk:], pkc, pvc, pos)
    for b in range(2):
        ek[b, int(pos[b])] = p[b, 64:64 + Rk]
        ev[b, int(pos[b])] = p[b, 64 + Rk:]
    assert torch.equal(pkc, ek) and torch.equal(pvc, ev)
    with pytest.raises(ValueError, match="int32"):
        RD.rankkv_append(p[:, 64:64 + Rk], p[:, 64 + Rk:], pkc, pvc, pos.long())
    from flashsvd_amd._lib import FlashSVDHipError
    with pytest.raises(FlashSVDHipError, match="aligned"):
        RD.rankkv_append(p[:, 60:60 + Rk], p[:, 64 + Rk:], pkc, pvc, pos)


@pytest.mark.parametrize("B,rq,rk,rv", [(1, 1024, 1024, 1024), (2, 72, 40, 136), (1, 64, 52, 52)])
def test_projection_with_append_epilogue_equals_projection_then_append(RD, B, rq, rk, rv):
    """fsvd_linear_rankkv_append: one launch, the bits of fsvd_linear followed by fsvd_rankkv_append (or by the indexed
    copy, for ranks off the 8 grid), fused RMSNorm included; rows outside the cache are not appended."""
    from flashsvd_amd import hip_ops
    from flashsvd_amd._lib import FlashSVDHipError
    K, S = 512, 24
    x, w = rand_bf16(B, K, seed=1).cuda(), rand_bf16(rq + rk + rv, K, std=0.05, seed=2).cuda()
    nw = (rand_bf16(K, seed=3) * 0.1 + 1).cuda()
    pos = torch.tensor([5, 30][:B], dtype=torch.int32).cuda()       # the second row lies outside the cache
    pkc = rand_bf16(B, S, rk, seed=4).cuda()
    pvc = rand_bf16(B, S, rv, seed=5).cuda()
    want_k, want_v = pkc.clone(), pvc.clone()
    p_ref = hip_ops.linear(x, w, norm_weight=nw, eps=1e-6)
    want_k[0, 5], want_v[0, 5] = p_ref[0, rq:rq + rk], p_ref[0, rq + rk:]
    p = hip_ops.linear_rankkv_append(x, w, pkc, pvc, pos, ranks=(rq, rk, rv), norm_weight=nw, eps=1e-6)
    assert torch.equal(p, p_ref) and torch.equal(pkc, want_k) and torch.equal(pvc, want_v)
    assert_close_bf16(p, O.lin(O.rms_norm(x.cpu(), nw.cpu(), 1e-6), w.cpu()), "projection")
    with pytest.raises(ValueError, match="one or two rows"):
        hip_ops.linear_rankkv_append(rand_bf16(3, K).cuda(), w, rand_bf16(3, S, rk).cuda(), rand_bf16(3, S, rv).cuda(),
                                     torch.zeros(3, dtype=torch.int32).cuda(), ranks=(rq, rk, rv))


def test_rank_decode_rejects_unsupported(RD):
    from flashsvd_amd._lib import FlashSVDHipError
    c = lambda *s: rand_bf16(*s).cuda()
    lens = torch.tensor([4], dtype=torch.int32).cuda()
    with pytest.raises(FlashSVDHipError, match="head_dim"):
        RD.rank_decode(c(1, 2, 64), c(1, 8, 16), c(1, 8, 16), c(128, 16), c(128, 16), None, None, lens, num_kv_heads=2)
    with pytest.raises(FlashSVDHipError, match="multiples of 8"):
        RD.rank_decode(c(1, 2, 128), c(1, 8, 12), c(1, 8, 12), c(256, 12), c(256, 12), None, None, lens, num_kv_heads=2)
    with pytest.raises(ValueError, match="bfloat16 or float16"):
        RD.rank_decode(c(1, 2, 128).float(), c(1, 8, 16), c(1, 8, 16), c(256, 16), c(256, 16), None, None, lens, num_kv_heads=2)


def test_model_rank_cache_greedy_matches_oracle_rank_cache():
    from flashsvd_amd.graphs import GraphedDecoder
    from flashsvd_amd.runtime.cache import FlashSVDLegacySparseKVCache
    mw = O.make_model(d=256, n_heads=2, n_kv_heads=2, head_dim=128, ffn=512, attn_rank=64, mlp_rank=96, n_layers=2,
                      vocab=500, dtype=BF16, seed=5, std=0.05)
    prompt = torch.randint(0, 500, (1, 21), generator=torch.Generator().manual_seed(4))
    n_new = 8
    ref_tok, ref_hid, ref_cache = O.greedy_decode(mw, prompt, n_new, "rank", return_hidden=True)
    model = model_from_oracle(mw)
    cache = FlashSVDLegacySparseKVCache(model.config, max_batch_size=1, max_cache_len=40, device="cuda", dtype=BF16)
    out = model(prompt.cuda(), past_key_values=cache, cache_position=torch.arange(21))
    assert_close_bf16(cache.key_cache[0][:, :21], ref_cache.pk[0][:, :21], "Pk cache layer 0")
    assert_close_bf16(out.hidden_states[:, -1], ref_hid[:, 0], "prefill hidden", rel_tol=3e-2)
    # teacher-forced with the oracle's tokens: the rank path rounds differently from the oracle's
    # (fp32 K rebuild, V applied in rank space), so near-tied logits may pick another token
    tok = out.logits[:, -1].float().argmax(-1, keepdim=True)
    same = int(torch.equal(tok.cpu(), ref_tok[:, :1]))
    dec = GraphedDecoder(model, cache, 1)
    dec.set_state(ref_tok[:, :1].cuda(), 21)
    for s in range(1, n_new):
        nxt = dec.eager_step().clone().cpu()
        assert_close_bf16(dec.hidden, ref_hid[:, s], f"hidden step {s}", rel_tol=3e-2)
        same += int(torch.equal(nxt, ref_tok[:, s:s + 1]))
        dec.tokens.copy_(ref_tok[:, s:s + 1])
    assert same >= n_new - 2, f"only {same}/{n_new} teacher-forced tokens identical"


def test_graph_replays_of_the_three_launch_form_match_eager_steps():
    """Batch 16 over a 1000-token rank-space context (8 heads: 2^17 (head, key) pairs): the decode step captured in a HIP
    graph (score, softmax, accumulation and merge launches, scores in the registered scratch) replayed three times, with
    synchronisations between the replays, gives the tokens and hidden states of eager steps from the same state."""
    from flashsvd_amd import hip_ops
    from flashsvd_amd.graphs import GraphedDecoder
    from flashsvd_amd.runtime.cache import FlashSVDLegacySparseKVCache
    mw = O.make_model(d=1024, n_heads=8, n_kv_heads=8, head_dim=128, ffn=512, attn_rank=64, mlp_rank=64, n_layers=1,
                      vocab=300, dtype=BF16, seed=9, std=0.05)
    model = model_from_oracle(mw)
    B, Lp, S = 16, 1000, 1100
    prompt = torch.randint(0, 300, (B, Lp), generator=torch.Generator().manual_seed(6)).cuda()
    runs = []
    for graphed in (True, False):
        cache = FlashSVDLegacySparseKVCache(model.config, max_batch_size=B, max_cache_len=S, device="cuda", dtype=BF16)
        out = model(prompt, past_key_values=cache, cache_position=torch.arange(Lp), logits_to_keep=1)
        tok = out.logits[:, -1].float().argmax(-1, keepdim=True)
        dec = GraphedDecoder(model, cache, B)
        dec.set_state(tok, Lp)
        if graphed:
            dec.capture()
        toks, hids = [tok.cpu()], []
        for _ in range(3):
            t = dec.step() if graphed else dec.eager_step()
            torch.cuda.synchronize()
            toks.append(t.clone().cpu())
            hids.append(dec.hidden.float().cpu().clone())
        runs.append((torch.cat(toks, 1), torch.stack(hids)))
    assert torch.equal(runs[0][0], runs[1][0]), "graph replays and eager steps disagree on tokens"
    assert torch.equal(runs[0][1], runs[1][1]), "graph replays and eager steps disagree on hidden states"
    assert torch.isfinite(runs[0][1]).all()
    # (the projections that follow the attention in a step reuse the scratch, so the weights cannot be read back here;
    # the shape is above the size from which fsvd_attn_decode_rankkv takes the form, with scratch registered)
    assert hip_ops._SPLIT_WS.get(torch.cuda.current_device()) is not None and B * 8 * ((S + 63) // 64 * 64) >= 1 << 17


def test_decode_driver_serves_the_rank_space_cache(monkeypatch):
    """decode_kvcache_eval(lowrank_cache=True) (utils/evaluator.py:358-371) decodes over FlashSVDLegacySparseKVCache through
    the per-operator graph engine, with per-layer and unequal q/k/v ranks; generate_text takes the same cache when the
    checkpoint's config asks for it, and then produces the oracle's rank-cache tokens."""
    from flashsvd_amd import api, llama
    from types import SimpleNamespace
    monkeypatch.setenv("FLASHSVD_AMD_DECODE_ENGINE", "auto")
    cfg = SimpleNamespace(hidden_size=256, num_attention_heads=2, num_key_value_heads=2, head_dim=128, intermediate_size=512,
                          num_hidden_layers=2, vocab_size=500, rope_theta=10000.0, rms_norm_eps=1e-6, hidden_act="silu",
                          max_position_embeddings=256)
    with torch.device("meta"):
        hetero = llama.SVDLlamaForCausalLM(cfg, attn_ranks=dict(q=64, k=40, v=72, o=64), mlp_rank=96)
    hetero = llama.materialize(hetero, "cuda", BF16, seed=1, std=0.05)
    r = api.decode_kvcache_eval(hetero, prompt_len=33, new_tokens=5, warmup=2, batch_size=2, lowrank_cache=True)
    assert r["lowrank_cache"] and not r["flashsvd_dense_cache"] and r["decode_engine"] == "graph" and r["decode_tok_s"] > 0
    with pytest.raises(ValueError, match="mutually exclusive"):
        api.decode_kvcache_eval(hetero, prompt_len=8, new_tokens=1, warmup=0, lowrank_cache=True, flashsvd_dense_cache=True)

    mw = O.make_model(d=256, n_heads=2, n_kv_heads=2, head_dim=128, ffn=512, attn_rank=64, mlp_rank=96, n_layers=2,
                      vocab=500, dtype=BF16, seed=5, std=0.05)
    model = model_from_oracle(mw)
    model.config.flash_svd_use_lowrank_cache = True
    prompt = torch.randint(0, 500, (1, 21), generator=torch.Generator().manual_seed(4))

    class Tok:
        eos_token_id = None
        pad_token_id = 0

        def __call__(self, text, return_tensors="pt", add_special_tokens=False):
            return {"input_ids": prompt}

        def decode(self, ids, skip_special_tokens=False):
            return " ".join(map(str, ids))

    out = api.generate_text(model, Tok(), prompt="x", max_new_tokens=6, use_graph=True)
    ref_tok, _, _, ref_logits = O.greedy_decode(mw, prompt, 6, "rank", return_logits=True)
    got, ref = out["completion_ids"], ref_tok[0].tolist()
    same = next((s for s in range(6) if got[s] != ref[s]), 6)
    if same < 6:    # the first differing token must be a near-tie in the oracle (rank path: fp32 K rebuild, V applied in rank space)
        lo = ref_logits[0, same].float()
        assert float(lo[ref[same]] - lo[got[same]]) <= 2e-2 * float(lo.abs().max()), f"{got} vs {ref}"
    assert same >= 3, f"{got} vs {ref}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,start,rq,rk,rv", [(1, 1, 0, 8, 8, 8), (2, 17, 3, 64, 520, 256), (3, 5, 0, 40, 1664, 2048), (2, 9, 4, 6, 8, 8), (2, 9, 4, 8, 12, 4)])
def test_rankkv_fill_matches_copies(RD, B, T, start, rq, rk, rv, dtype):
    """Rows of one piece to several rounds of a wave, a last workgroup that is not full, rows off the grid; nothing beside them is written."""
    S = start + T + 2
    p = torch.randn(B, T, rq + rk + rv, device="cuda").to(dtype)
    caches = [torch.full((B + 1, S, r), 7.0, device="cuda", dtype=dtype) for r in (rk, rv)]
    want = [c.clone() for c in caches]
    want[0][:B, start:start + T], want[1][:B, start:start + T] = p[..., rq:rq + rk], p[..., rq + rk:]
    RD.rankkv_fill(p, *caches, start)
    assert torch.equal(caches[0], want[0]) and torch.equal(caches[1], want[1])
    if rk % 8 == 0 and rq % 8 == 0:
        with pytest.raises((ValueError, RuntimeError)):                    # past the end of the caches
            torch.ops.flashsvd_hip.rankkv_fill(p, *caches, start + 3)
    wide = [torch.full((B + 1, S + 1, r + 8), 7.0, device="cuda", dtype=dtype) for r in (rk, rv)]
    views = [w[:, 1:, :r] for w, r in zip(wide, (rk, rv))]
    RD.rankkv_fill(p, *views, start)
    for v, c, w in zip(views, want, wide):
        assert torch.equal(v, c) and bool((w[:, 0] == 7).all()) and bool((w[..., v.shape[2]:] == 7).all())
    off = [torch.full((B + 1, S, r + 8), 7.0, device="cuda", dtype=dtype) for r in (rk, rv)]
    RD.rankkv_fill(p, *(o[..., 4:4 + r] for o, r in zip(off, (rk, rv))), start)                  # strides on the grid, addresses off it
    for o, c, r in zip(off, want, (rk, rv)):
        assert torch.equal(o[..., 4:4 + r], c) and bool((o[..., :4] == 7).all()) and bool((o[..., 4 + r:] == 7).all())
