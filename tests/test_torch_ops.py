"""The custom operators flashsvd_hip::* (flashsvd_amd/torch_ops.py): registration, schemas and the fake / meta shape
functions run here without a GPU; the device implementations are exercised by every GPU test, which reach the library
through these operators, and by torch.library.opcheck in the GPU part below."""
import pytest
import torch

import flashsvd_amd.torch_ops  # noqa: F401  (registers the operators, whichever test runs first)

BF16 = torch.bfloat16


def _m(*shape, dtype=BF16):
    return torch.empty(*shape, dtype=dtype, device="meta")


def test_every_operator_is_registered_with_a_schema():
    from flashsvd_amd import torch_ops as T
    for name in T.OP_NAMES:
        packet = getattr(torch.ops.flashsvd_hip, name)
        schema = str(packet.default._schema)
        assert schema.startswith(f"flashsvd_hip::{name}("), schema
    # mutated arguments are declared: the caches of the append / attention operators, the output overloads
    assert "Tensor(a!) k_cache" in str(torch.ops.flashsvd_hip.qkv_rope_append.default._schema)
    assert "Tensor(a!) out" in str(torch.ops.flashsvd_hip.linear.out._schema)
    assert "Tensor(a!) pk_cache" in str(torch.ops.flashsvd_hip.rankkv_append.default._schema)


def test_meta_shape_functions():
    ops = torch.ops.flashsvd_hip
    B, d, R, D, H, Hk, Dh, S = 3, 256, 64, 512, 4, 2, 128, 40
    x = _m(B, 1, d)
    assert ops.linear(x, _m(R, d)).shape == (B, 1, R)
    assert ops.linear(x, _m(R, d), None, _m(d), 1e-6, None, 0).dtype == BF16
    out = _m(B, 1, R)
    assert ops.linear.out(x, _m(R, d), out=out) is out
    assert ops.swiglu_linear(_m(B, 2 * R), _m(D, R), _m(D, R), R).shape == (B, D)
    assert ops.rmsnorm(x, _m(d)).shape == x.shape
    kc = _m(B, S, Hk, Dh)
    q = ops.qkv_rope_append(_m(B, 3 * R), _m(H * Dh, R), _m(Hk * Dh, R), _m(Hk * Dh, R), _m(S, Dh // 2), _m(S, Dh // 2),
                            _m(B, dtype=torch.int32), kc, _m(B, S, Hk, Dh), H, Hk, Dh)
    assert q.shape == (B, H, Dh)
    assert ops.attn_decode_densekv(q, kc, kc, _m(B, dtype=torch.int32)).shape == (B, H, Dh)
    assert ops.attn_decode_rankkv(q, _m(B, S, R), _m(B, S, R), _m(Hk * Dh, R), _m(Hk * Dh, R), None, None,
                                  _m(B, dtype=torch.int32), Hk).shape == (B, H, Dh)
    assert ops.rope_attn_prefill(_m(B, 9, H, Dh), _m(B, S, Hk, Dh), _m(B, S, Hk, Dh)).shape == (B, 9, H, Dh)
    Q, K, V = ops.reconstruct_qkv_token(_m(B, H, R), _m(B, Hk, R), _m(B, Hk, R), _m(H, R, Dh), _m(Hk, R, Dh), _m(Hk, R, Dh))
    assert Q.shape == (B, H, Dh) and K.shape == V.shape == (B, Hk, Dh)
    assert ops.xw_linear(_m(B, d), _m(d, R)).shape == (B, R)
    assert ops.mlp_dual_split(_m(B, R), _m(B, R), _m(R, D), _m(R, D), _m(D, R), _m(R, d), None, 2, 128).shape == (B, d)
    assert ops.rankkv_append(_m(B, R), _m(B, R), _m(B, S, R), _m(B, S, R), _m(B, dtype=torch.int32)) is None
    assert ops.lowrank_expand_heads(_m(B, 9, R), _m(H * Dh, R), H, Dh, _m(B, 9, H, Dh)) is None


def test_host_tensors_raise_value_error_through_the_dispatcher():
    from flashsvd_amd import hip_ops
    with pytest.raises(ValueError, match="GPU tensor"):
        hip_ops.linear(torch.zeros(1, 64, dtype=BF16), torch.zeros(8, 64, dtype=BF16))
    with pytest.raises(ValueError, match="GPU tensor"):
        torch.ops.flashsvd_hip.rmsnorm(torch.zeros(1, 64, dtype=BF16), torch.ones(64, dtype=BF16))


def test_token_rows_are_an_operator_of_one_device():
    """set_token_rows_ writes through raw addresses: it declares what it writes, and refuses tensors of another device."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from flashsvd_amd import hip_ops
    schema = str(torch.ops.flashsvd_hip.set_token_rows_.default._schema)
    assert "Tensor(a!) tokens" in schema and "Tensor(b!) positions" in schema
    with FakeTensorMode():
        on = lambda dtype, i: torch.empty(4, dtype=dtype, device=f"cuda:{i}")
        for devices in ((0, 1, 0), (0, 0, 1), (1, 0, 0)):
            with pytest.raises(ValueError, match="one device"):
                hip_ops._set_token_rows_impl(*(on(dt, i) for dt, i in zip((torch.long, torch.long, torch.int32), devices)), 3)


def test_greedy_tokens_and_rotation_tables_are_of_one_device():
    """Both take raw addresses; as tensor operations a table of two devices was refused."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from flashsvd_amd import hip_ops
    with FakeTensorMode():
        on = lambda i, dtype, *s: torch.empty(*s, dtype=dtype, device=f"cuda:{i}")
        for a, b, c in ((0, 0, 1), (0, 1, 0), (1, 0, 0)):
            with pytest.raises(ValueError, match="one device"):
                hip_ops._greedy_token_impl(on(a, BF16, 4, 100), on(b, torch.long, 4, 1), on(c, torch.int32, 4))
        with pytest.raises(ValueError, match="one device"):
            hip_ops._rope_tables_impl(on(0, torch.long, 9), on(1, torch.float32, 64), BF16)


def test_prompt_attention_refuses_masks_of_another_device():
    """The kernel reads the masks through raw addresses: one that was left on the host is refused, not read."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from flashsvd_amd import hip_ops
    with FakeTensorMode():
        q, kv = torch.empty(2, 9, 4, 128, dtype=BF16, device="cuda:0"), torch.empty(2, 9, 4, 128, dtype=BF16, device="cuda:0")
        for device in ("cpu", "cuda:1"):
            for pad, add in ((torch.empty(2, 9, dtype=torch.uint8, device=device), None), (None, torch.empty(2, 9, 9, device=device))):
                with pytest.raises(ValueError, match="on the device of q"):
                    hip_ops._attn_prefill_impl(q, kv, kv, None, True, pad, add, None, None)


def test_prompt_coefficients_without_addresses_and_into_any_pair_of_caches():
    """The route of rankkv_fill is known from shapes and strides (a traced tensor has no address); caches of unequal length
    and caches that overlap are not for the kernel."""
    import warnings
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.utils._python_dispatch import TorchDispatchMode
    from flashsvd_amd.kernels.rank_decode import rankkv_fill

    class Names(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func.name())
            return func(*args, **(kwargs or {}))

    with FakeTensorMode(), warnings.catch_warnings():
        warnings.simplefilter("error")
        new = lambda *s: torch.empty(*s, dtype=BF16, device="cuda:0")
        p, rows = new(2, 9, 192), new(2, 32, 64)
        for pk, pv, in_one in ((rows, new(2, 32, 64), True), (rows, new(2, 40, 64), False), (rows, new(1, 32, 64).expand(2, 32, 64), False),
                               (new(2, 32, 72)[..., 8:], rows, True), (new(32, 2, 64).transpose(0, 1), rows, False)):
            seen = []
            with Names():
                try:
                    rankkv_fill(p, pk, pv, 0)
                except RuntimeError:
                    assert not in_one                          # copies refuse to write rows that overlap
            assert ("flashsvd_hip::rankkv_fill" in seen) == in_one, (pk.shape, pk.stride(), pv.shape, pv.stride())


def test_coefficients_of_different_devices_are_refused():
    """The dual-split MLP reads both sets of coefficients through raw addresses, one as a distance from the other."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from flashsvd_amd import hip_ops
    with FakeTensorMode():
        t = lambda *s, i=0: torch.empty(*s, dtype=BF16, device=f"cuda:{i}")
        with pytest.raises(ValueError, match="one device"):
            hip_ops._mlp_from_coefficients(t(4, 64), t(4, 64, i=1), t(128, 64), t(128, 64), t(64, 128), t(32, 64), None, 1)


@pytest.mark.gpu
def test_opcheck_and_fake_tensor_tracing_on_the_device():
    """torch.library.opcheck (schema and fake-tensor consistency against the real kernels) on the hot operators, and a
    make_fx trace of a low-rank MLP through fake tensors that records the custom operators as graph nodes."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from tests.util import rand_bf16
    ops = torch.ops.flashsvd_hip
    d, R, D = 512, 128, 768
    x = rand_bf16(1, d, seed=1).cuda()
    vw, gu, uu = rand_bf16(2 * R, d, std=0.05, seed=2).cuda(), rand_bf16(D, R, std=0.05, seed=3).cuda(), rand_bf16(D, R, std=0.05, seed=4).cuda()
    dv, du, nw = rand_bf16(R, D, std=0.05, seed=5).cuda(), rand_bf16(d, R, std=0.05, seed=6).cuda(), torch.ones(d, dtype=BF16, device="cuda")
    checks = ("test_schema", "test_faketensor")
    torch.library.opcheck(ops.linear.default, (x, vw, None, nw, 1e-6, None, 0), test_utils=checks)
    torch.library.opcheck(ops.linear.out, (x, vw), dict(out=torch.empty(1, 2 * R, dtype=BF16, device="cuda")), test_utils=checks)
    p = ops.linear(x, vw, None, nw)
    torch.library.opcheck(ops.swiglu_linear.default, (p, gu, uu, R), test_utils=checks)
    torch.library.opcheck(ops.rmsnorm.default, (x, nw), test_utils=checks)
    H, Dh, S = 2, 128, 32
    kc, vc = rand_bf16(1, S, H, Dh, seed=7).cuda(), rand_bf16(1, S, H, Dh, seed=8).cuda()
    lens = torch.tensor([20], dtype=torch.int32, device="cuda")
    q = rand_bf16(1, H, Dh, seed=9).cuda()
    torch.library.opcheck(ops.attn_decode_densekv.default, (q, kc, vc, lens), dict(nsplit=2), test_utils=checks)

    def mlp(x, vw, gu, uu, dv, du, nw):
        p = ops.linear(x, vw, None, nw, 1e-6)
        h = ops.swiglu_linear(p, gu, uu, R)
        return ops.linear(ops.linear(h, dv), du, None, None, 1e-6, x)

    args = (x, vw, gu, uu, dv, du, nw)
    g = make_fx(mlp, tracing_mode="fake")(*args)
    targets = [n.target for n in g.graph.nodes if n.op == "call_function"]
    assert targets.count(ops.linear.default) == 3 and ops.swiglu_linear.default in targets
    assert torch.equal(g(*args), mlp(*args))
