"""The launches between two decoded tokens (csrc/token.hip) against torch: whole numbers, so they agree exactly."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,V,off", [(1, 1, 0), (2, 7, 1), (3, 8, 0), (1, 9, 3), (5, 1023, 1), (16, 32000, 0), (2, 32771, 5), (1, 65543, 0)])
def test_greedy_token_is_the_argmax(dtype, B, V, off):
    from flashsvd_amd import hip_ops
    gen = torch.Generator().manual_seed(B * V + off)
    rows = torch.randn(B, V + off + 3, generator=gen).to(dtype).cuda()
    x = rows[:, off:off + V]                            # rows at any element's address
    cases = [x.clone()]
    cases.append(torch.zeros_like(x))                   # all equal, zeros of both signs: the first
    cases[-1][:, ::2] = -0.0
    cases.append(torch.full_like(x, float("-inf")))
    top = x.clone()                                     # the largest value twice, the last element among them
    top[:, V - 1] = top[:, V // 2] = 100.0
    cases.append(top)
    nan = x.clone()
    nan[:, V // 3] = float("nan")
    nan[:, V // 2] = float("inf")
    cases.append(nan)
    for c in cases:
        x.copy_(c)
        tokens = torch.full((B, 1), -7, dtype=torch.long, device="cuda")
        pos = torch.arange(B, dtype=torch.int32, device="cuda")
        hip_ops.greedy_token_(x, tokens, pos)
        ref = c.float()
        want = torch.where(ref.isnan().any(1), ref.isnan().float().argmax(1), ref.argmax(1)) if ref.isnan().any() else (ref == ref.amax(1, keepdim=True)).float().argmax(1)
        assert tokens[:, 0].tolist() == want.tolist()
        assert pos.tolist() == list(range(1, B + 1))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V,off", [(5, 0), (8191, 1), (8200, 0), (14336, 3), (14337, 0), (14343, 0), (32768, 0), (32769, 2), (65535, 1), (70007, 0)])
def test_greedy_token_where_the_largest_lies(V, off, dtype):
    """The largest value in the first piece, in the first and a later round, in the last round, behind the last whole piece; only zeros above the
    rest, of either sign; a NaN of either sign; the lowest finite value."""
    from flashsvd_amd import hip_ops
    x = -torch.rand(14, V + off, generator=torch.Generator().manual_seed(V)).to(dtype)[:, off:] - 1
    first, mid, last = 0, V // 2, V - 1               # up to 14336 logits in one pass, from there on in two
    spots = [(first,), (mid,), (last,), (mid, last), (first, mid), (max(0, V - V % 8 - 1),), (min(V - 1, 32767), last)]
    want = []
    for r, s in enumerate(spots):
        x[r, list(s)] = 3.0
        want.append(min(s))
    x[7, [mid, last]] = torch.tensor([-0.0, 0.0], dtype=dtype)
    x[8, [mid, last]] = torch.tensor([0.0, -0.0], dtype=dtype)
    x[9, [mid, last]] = -0.0
    x[10, last] = float("nan")
    x[11, first], x[12, mid] = float("inf"), float("nan")
    x.view(torch.int16)[11:13, last] = -1               # a negative NaN
    x[13] = torch.finfo(dtype).min
    want += [mid, mid, mid, last, last, mid, 0]
    rows = torch.empty(14, V + off, dtype=dtype, device="cuda")
    got = rows[:, off:]
    got.copy_(x.cuda())
    tokens = torch.full((14, 1), -7, dtype=torch.long, device="cuda")
    hip_ops.greedy_token_(got, tokens)
    assert tokens[:, 0].tolist() == want


def test_refusals_and_state_rows():
    from flashsvd_amd import hip_ops
    x = torch.zeros(2, 64, dtype=torch.bfloat16, device="cuda")
    t, p = torch.zeros(2, 1, dtype=torch.long, device="cuda"), torch.zeros(2, dtype=torch.int32, device="cuda")
    for bad in ((x.float(), t, p), (x.t(), t, p), (x, t[:1], p), (x, t.int(), p), (x, t, p[:1]), (x[:, :0], t, p)):
        with pytest.raises((ValueError, RuntimeError)):
            hip_ops.greedy_token_(*bad)
    hip_ops.set_token_rows_(t, torch.tensor([[5], [9]], device="cuda"), p, 31)
    assert t[:, 0].tolist() == [5, 9] and p.tolist() == [31, 31]
