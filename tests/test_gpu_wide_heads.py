"""16-bit forward and backward at head dims 256 and 512 (one wave per SIMD,
key-split forward, dK/dV with its two products on two waves) against 64-bit
attention, at tile edges, splits and modifiers."""

import ctypes
import math

import pytest
import torch

from attn_refs import attention, grads, varlen_attention
from fa_rdna3 import _native, alibi_slopes, flash_attention, flash_attention_varlen
from fa_rdna3.interface import _fwd_params

pytestmark = pytest.mark.gpu
# Largest relative 2-norm error: four roundings to the 16-bit type lie on any
# result's path (P or dS, out in delta, the operand products' inputs are
# exact, the result), each at most one unit 2^-11 / 2^-8 of what it rounds.
BOUND = {torch.float16: 4 * 2.0 ** -11, torch.bfloat16: 4 * 2.0 ** -8}


def _rand(shape, dtype, gen):
    return torch.randn(shape, generator=gen).to(dtype).cuda()


def _close(got, want, dtype):
    want = want.double()
    assert torch.isfinite(got).all()
    err = (got.double() - want).norm() / want.norm().clamp_min(1e-30)
    assert err <= BOUND[dtype], float(err)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim", [256, 512])
@pytest.mark.parametrize("sq,sk,opts", [
    (1, 1, {}), (33, 31, {"causal": True}), (127, 129, {}), (128, 128, {"causal": True}),
    (129, 1024, {}), (700, 700, {"causal": True, "window": (200, 0)}), (300, 2000, {"softcap": 20.0}),
    (257, 1500, {"scale": 0.0}), (64, 640, {"causal": True, "softcap": 5.0}),
])
def test_forward(dtype, head_dim, sq, sk, opts):
    gen = torch.Generator().manual_seed(sq * 7 + sk)
    q = _rand((2, sq, 2, head_dim), dtype, gen).transpose(1, 2)  # heads within a row
    k, v = (_rand((2, 1, sk, head_dim), dtype, gen) for _ in range(2))
    opts = dict(opts)
    window, scale = opts.pop("window", (-1, -1)), opts.pop("scale", None)
    out = flash_attention(q, k, v, softmax_scale=scale, window_size=window, **opts)
    ref = attention(q.double(), k.double(), v.double(), scale=scale, window=window, **opts)
    _close(out, ref, dtype)


@pytest.mark.parametrize("head_dim", [256, 512])
@pytest.mark.parametrize("hidden", ["none", "row", "share"])
def test_key_splits_agree_with_one_workgroup(head_dim, hidden):
    """fa_fwd_ws with and without its scratch, output and LSE; a row that sees
    no key at all, and one whose first share of the keys is hidden."""
    gen = torch.Generator().manual_seed(5)
    dtype, sq, sk = torch.float16, 150, 1100
    q, k, v = (_rand((1, 1, n, head_dim), dtype, gen) for n in (sq, sk, sk))
    bias = torch.zeros((1, 1, sq, sk), device="cuda")
    if hidden == "row":
        bias[:, :, 7] = float("-inf")
    elif hidden == "share":
        bias[:, :, 7, :600] = float("-inf")
    lib, got = _native.lib(), []
    for split in (True, False):
        out = torch.full((1, 1, sq, head_dim), float("nan"), device="cuda", dtype=dtype)
        lse = torch.full((1, 1, sq), float("nan"), device="cuda")
        p = _fwd_params(q, k, v, out, lse, dense=True, causal=False, softmax_scale=1 / math.sqrt(head_dim),
                        window=(-1, -1), softcap=0.0, bias=bias, alibi=None, dropout_p=0.0, dropout_seed=0)
        need = lib.fa_fwd_workspace_bytes(ctypes.byref(p))
        assert need > 0
        ws = torch.empty(need if split else 0, dtype=torch.uint8, device="cuda")
        rc = lib.fa_fwd_ws(ctypes.byref(p), ws.data_ptr() if split else None, need if split else 0,
                           torch.cuda.current_stream().cuda_stream)
        assert rc == 0, lib.fa_last_error_string()
        got.append((out, lse))
    ref = attention(q.double(), k.double(), v.double(), bias=bias.double())
    for out, lse in got:
        _close(out, ref, dtype)
        if hidden == "row":
            assert (out[:, :, 7] == 0).all() and lse[0, 0, 7] == float("-inf")
    finite = torch.isfinite(got[0][1])
    assert torch.equal(finite, torch.isfinite(got[1][1]))
    # fp32 sums of at most 1100 terms taken in another order
    assert (got[0][1] - got[1][1])[finite].abs().max() <= 1100 * 2.0 ** -24 * 8


def test_no_splits_without_room_to_gain():
    p = _native.FwdParams()
    p.dtype, p.head_dim, p.batch, p.heads_q, p.heads_kv, p.seqlen_q, p.seqlen_k = 0, 256, 1, 16, 16, 2048, 2048
    p.window_left = p.window_right = -1  # none (0 would be a window of one key)
    need = _native.lib().fa_fwd_workspace_bytes
    assert need(ctypes.byref(p)) == 0  # 256 row blocks fill the CUs
    p.heads_q = p.heads_kv = 1
    assert need(ctypes.byref(p)) > 0
    p.seqlen_k = 200  # fewer than two shares of four tiles
    assert need(ctypes.byref(p)) == 0
    p.seqlen_k, p.head_dim = 2048, 128
    assert need(ctypes.byref(p)) == 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads,kv,sq,sk,opts", [
    (2, 2, 1, 1, {}), (2, 1, 31, 33, {"causal": True}), (2, 2, 64, 64, {"causal": True}), (4, 2, 129, 65, {}),
    (4, 2, 333, 700, {"causal": True}), (2, 1, 500, 500, {"softcap": 10.0}),
    (2, 2, 500, 500, {"causal": True, "window": (90, 0), "softcap": 30.0}),
    (2, 2, 400, 257, {"bias": True, "window": (100, 60)}), (2, 2, 257, 400, {"alibi": True, "causal": True}),
    (2, 1, 1100, 900, {"causal": True, "softcap": 20.0}),  # dK/dV in four shares of the query steps
    (4, 2, 2000, 300, {}), (16, 8, 2000, 2048, {"causal": True}),  # seven shares; a full grid in two
])
def test_backward_256(dtype, heads, kv, sq, sk, opts):
    gen = torch.Generator().manual_seed(sq + 3 * sk)
    opts = dict(opts)
    q, do = (_rand((1, sq, heads, 256), dtype, gen).transpose(1, 2) for _ in range(2))
    k, v = (_rand((1, kv, sk, 256), dtype, gen) for _ in range(2))
    window = opts.pop("window", (-1, -1))
    bias = _rand((1, heads, sq, sk), torch.float32, gen) if opts.pop("bias", False) else None
    slopes = alibi_slopes(heads) if opts.pop("alibi", False) else None
    got = grads(lambda a, b, c: flash_attention(a, b, c, window_size=window, bias=bias, alibi_slopes=slopes, **opts),
                q, k, v, do)
    want = grads(lambda a, b, c: attention(a, b, c, window=window, bias=None if bias is None else bias.double(),
                                           alibi=None if slopes is None else slopes.double(), **opts),
                 q.double(), k.double(), v.double(), do.double())
    scale = max(float(w.norm()) for w in want)
    for g, w in zip(got, want):
        if float(w.norm()) <= 1e-6 * scale:  # one visible key: dQ and dK are rounding noise around zero
            assert float(g.double().norm()) <= BOUND[dtype] * scale
        else:
            _close(g, w, dtype)


@pytest.mark.parametrize("opts", [{}, {"causal": True}, {"window": (150, 40)}])
@pytest.mark.parametrize("upstream", [1.0, 1e-2, 1e-3, 1e-4])
def test_softcap_256_keeps_small_gradients(upstream, opts):
    """fp16 holds dS in full: the products of dQ and dK read dS rounded to
    fp16 once, and below its smallest normal number (a mean loss without loss
    scaling is there) the error follows from that rounding.  Modelled in 64
    bits, with the results' own rounding; 1.15 covers the fp32 sums, delta and
    the row sums' rounding (a dS stored as a quarter is at 1.06 to 3.6)."""
    gen = torch.Generator().manual_seed(3)
    dtype, n, cap = torch.float16, 512, 50.0
    q, k, v = (_rand((1, 2, n, 256), dtype, gen) for _ in range(3))
    do = (torch.randn((1, 2, n, 256), generator=gen) * upstream).to(dtype).cuda()
    opts = dict(opts)
    window = opts.pop("window", (-1, -1))
    got = grads(lambda a, b, c: flash_attention(a, b, c, softcap=cap, window_size=window, **opts), q, k, v, do)
    qd, kd, vd, dod = (t.double() for t in (q, k, v, do))
    exact = grads(lambda a, b, c: attention(a, b, c, softcap=cap, window=window, **opts), qd, kd, vd, dod)
    raw = torch.matmul(qd, kd.transpose(-1, -2).contiguous()) / 16
    t = torch.tanh(raw / cap)
    keep = torch.ones((n, n), dtype=torch.bool, device="cuda")
    i, j = torch.arange(n, device="cuda")[:, None], torch.arange(n, device="cuda")[None, :]
    if opts.get("causal"):
        keep &= j <= i
    if window[0] >= 0:
        keep &= (j >= i - window[0]) & (j <= i + window[1])
    p = torch.softmax((cap * t).masked_fill(~keep, float("-inf")), -1)
    dp = torch.matmul(dod, vd.transpose(-1, -2).contiguous())
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * (1 - t * t)
    r16 = lambda x: x.to(torch.float16).double()
    model = (r16(torch.matmul(r16(ds), kd) / 16), r16(torch.matmul(r16(ds).transpose(-1, -2).contiguous(), qd) / 16))
    for g, m, w in zip(got, model, exact):
        err, floor = float((g.double() - w).norm()), float((m - w).norm())
        assert err <= 1.15 * floor, (err / float(w.norm()), floor / float(w.norm()))


def test_dropout_256_equals_zero_padded_128():
    """The dropout mask depends on positions and seed only, so a head of 128
    padded with zeros to 256 must give the 128-wide kernels' result."""
    gen = torch.Generator().manual_seed(9)
    q, k, v, do = (_rand((1, 2, 300, 128), torch.float16, gen) for _ in range(4))
    pad = lambda t: torch.nn.functional.pad(t, (0, 128))
    tail = (False, 0.1, -1, -1, 0.0, None, None, 0.3, 1234)
    ops = _native.ops()
    out, lse = ops.forward(q, k, v, *tail)
    wide, wlse = ops.forward(pad(q), pad(k), pad(v), *tail)
    _close(wide[..., :128], out, torch.float16)
    assert (wlse - lse).abs().max() <= 1e-5
    for g, w in zip(ops.backward(pad(do), pad(q), pad(k), pad(v), wide, wlse, *tail),
                    ops.backward(do, q, k, v, out, lse, *tail)):
        _close(g[..., :128], w, torch.float16)
        assert (g[..., 128:] == 0).all()


@pytest.mark.parametrize("limit", [0, None])
def test_backward_256_varlen_and_without_scratch(limit):
    gen = torch.Generator().manual_seed(11)
    lens = [1, 70, 300, 129]
    q, do = (_rand((sum(lens), 4, 256), torch.bfloat16, gen) for _ in range(2))
    k, v = (_rand((sum(lens), 2, 256), torch.bfloat16, gen) for _ in range(2))
    cu = torch.tensor([0, 1, 71, 371, 500], dtype=torch.int32, device="cuda")
    before = _native.ds_scratch_limit()
    try:
        if limit is not None:
            _native.set_ds_scratch_limit(limit)
        got = grads(lambda a, b, c: flash_attention_varlen(a, b, c, cu, cu, 300, 300, causal=True), q, k, v, do)
        dense = grads(lambda a, b, c: flash_attention(a, b, c, causal=True), *(
            t[71:371].transpose(0, 1)[None] for t in (q, k, v, do)))
    finally:
        _native.set_ds_scratch_limit(before)
    want = grads(lambda a, b, c: varlen_attention(a, b, c, lens, lens, causal=True),
                 q.double(), k.double(), v.double(), do.double())
    for g, d, w in zip(got, dense, want):
        _close(g, w, torch.bfloat16)
        _close(d[0].transpose(0, 1), w[71:371], torch.bfloat16)
