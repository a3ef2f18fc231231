"""The decode operators called by themselves check what their kernels read and
write, and decode refuses torch.func transforms of its arguments."""

import pytest
import torch

from fa_rdna3 import _native, flash_attention_decode, flash_attention_decode_paged, flash_attention_with_kvcache

pytestmark = pytest.mark.gpu
B, HQ, HKV, ROWS, KEYS, D = 2, 8, 2, 1, 300, 64


def _rand(*shape, dtype=torch.float16):
    return torch.randn(shape, device="cuda").to(dtype)


def _decode_args():
    lens = torch.tensor([250, 100], dtype=torch.int32, device="cuda")
    return dict(q=_rand(B, HQ, ROWS, D), k=_rand(B, HKV, KEYS, D), v=_rand(B, HKV, KEYS, D),
                new_k=_rand(B, HKV, ROWS, D), new_v=_rand(B, HKV, ROWS, D), lens=lens, causal=False, scale=0.125,
                num_splits=2, kv_fp8=False, k_scale=1.0, v_scale=1.0,
                tickets=torch.zeros(B * HQ * ROWS, dtype=torch.int32, device="cuda"))


def _paged_args():
    pages = B * 20
    return dict(q=_rand(B, HQ, ROWS, D), k_cache=_rand(pages, 16, HKV, D), v_cache=_rand(pages, 16, HKV, D),
                block_table=torch.arange(pages, dtype=torch.int32, device="cuda").view(B, 20),
                context_lens=torch.tensor([250, 100], dtype=torch.int32, device="cuda"), causal=False, scale=0.125,
                num_splits=2, kv_fp8=False, k_scale=1.0, v_scale=1.0,
                tickets=torch.zeros(B * HQ * ROWS, dtype=torch.int32, device="cuda"))


BAD = [
    ("lens", lambda t: t.cpu()), ("lens", lambda t: t.long()), ("lens", lambda t: t[:1]), ("lens", lambda t: None),
    ("tickets", lambda t: t.cpu()), ("tickets", lambda t: t[:-1]), ("tickets", lambda t: t.long()),
    ("tickets", lambda t: t.repeat(2)[::2]),
    ("new_k", lambda t: t.cpu()), ("new_k", lambda t: t[:1]), ("new_k", lambda t: t[:, :1]),
    ("new_k", lambda t: t[..., :32]), ("new_k", lambda t: t.bfloat16()), ("new_k", lambda t: None),
    ("new_v", lambda t: t.repeat(1, 1, 2, 1)), ("new_v", lambda t: None), ("new_v", lambda t: t[0]),
    ("k", lambda t: t.cpu()), ("k", lambda t: t.float()), ("k", lambda t: t[..., :32]), ("k", lambda t: t[:1]),
    ("k", lambda t: t.transpose(2, 3).contiguous().transpose(2, 3)), ("v", lambda t: t[:, :, :100]),
    ("kv_fp8", lambda t: True), ("q", lambda t: t[0]), ("num_splits", lambda t: 0),
]


@pytest.mark.parametrize("case", range(len(BAD)))
def test_decode_operator_refuses(case):
    name, change = BAD[case]
    args = _decode_args()
    before = args["k"].clone(), args["v"].clone()
    args[name] = change(args[name])
    with pytest.raises((RuntimeError, NotImplementedError)):
        _native.ops().decode(**args)
    torch.cuda.synchronize()
    if name not in ("k", "v", "num_splits"):
        assert torch.equal(args["k"], before[0]) and torch.equal(args["v"], before[1])


BAD_PAGED = [
    ("block_table", lambda t: t.cpu()), ("block_table", lambda t: t.long()), ("block_table", lambda t: t[:1]),
    ("block_table", lambda t: t[0]), ("context_lens", lambda t: t.cpu()), ("context_lens", lambda t: t[:1]),
    ("context_lens", lambda t: t.long()), ("tickets", lambda t: t.cpu()), ("tickets", lambda t: t[:-1]),
    ("k_cache", lambda t: t.bfloat16()), ("v_cache", lambda t: t[:4]), ("v_cache", lambda t: t.cpu()),
    ("q", lambda t: t[..., :32]),
]


@pytest.mark.parametrize("case", range(len(BAD_PAGED)))
def test_paged_operator_refuses(case):
    name, change = BAD_PAGED[case]
    args = _paged_args()
    args[name] = change(args[name])
    with pytest.raises((RuntimeError, NotImplementedError)):
        _native.ops().decode_paged(**args)
    torch.cuda.synchronize()


def test_operators_run_with_what_they_ask_for():
    args = _decode_args()
    want = flash_attention_with_kvcache(args["q"], args["k"].clone(), args["v"].clone(), args["new_k"], args["new_v"],
                                        cache_seqlens=args["lens"])
    torch.testing.assert_close(_native.ops().decode(**args), want, rtol=4e-3, atol=4e-3)
    args = _paged_args()
    want = flash_attention_decode_paged(args["q"].squeeze(2), args["k_cache"], args["v_cache"], args["block_table"],
                                        args["context_lens"])
    torch.testing.assert_close(_native.ops().decode_paged(**args).squeeze(2), want, rtol=4e-3, atol=4e-3)


def _calls():
    a, p = _decode_args(), _paged_args()
    return [
        (lambda q: flash_attention_decode(q, a["k"], a["v"], cache_seqlens=a["lens"]), a["q"]),
        (lambda q: flash_attention_with_kvcache(q, a["k"], a["v"], a["new_k"], a["new_v"], cache_seqlens=a["lens"]),
         a["q"]),
        (lambda q: flash_attention_decode_paged(q, p["k_cache"], p["v_cache"], p["block_table"], p["context_lens"]),
         p["q"].squeeze(2)),
    ]


@pytest.mark.parametrize("which", range(3))
def test_transforms_of_the_arguments_are_refused(which):
    """A jvp used to come back with a zero tangent."""
    call, q = _calls()[which]
    with pytest.raises(RuntimeError, match="torch.func transforms"):
        torch.func.jvp(call, (q,), (torch.ones_like(q),))
    with pytest.raises(RuntimeError, match="torch.func transforms"):
        torch.vmap(call)(q[None].clone())
    with pytest.raises(RuntimeError):
        torch.func.functionalize(call)(q)


@pytest.mark.parametrize("which", range(3))
def test_plain_tensors_inside_a_transform(which):
    call, q = _calls()[which]
    want = call(q)
    if which < 2:  # (one-row paged decode reshapes its query, which jvp wraps)
        out, tangent = torch.func.jvp(lambda x: call(q).float() * x, (torch.tensor(2.0, device="cuda"),),
                                      (torch.tensor(1.0, device="cuda"),))
        assert torch.equal(out, 2 * want.float()) and torch.equal(tangent, want.float())
    out = torch.vmap(lambda x: call(q).float() * x)(torch.tensor([1.0, 3.0], device="cuda"))
    assert torch.equal(out[1], 3 * want.float())
