"""Choice of the forward's form on a dense grid, and its aligned bias loads,
against 64-bit attention."""

import pytest
import torch

from attn_refs import attention
from fa_rdna3 import flash_attention

pytestmark = pytest.mark.gpu
# Relative 2-norm: four 16-bit roundings of at most one unit on a result's path.
BOUND = {torch.float16: 4 * 2.0 ** -11, torch.bfloat16: 4 * 2.0 ** -8}


def _check(out, q, k, v, dtype, **opts):
    ref = attention(q.double(), k.double(), v.double(), **opts)
    assert torch.isfinite(out).all()
    for got, want in zip(out, ref):  # each batch entry by itself: its own bias base, form and loads
        err = (got.double() - want).norm() / want.norm()
        assert err <= BOUND[dtype], float(err)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim", [32, 64, 128])
@pytest.mark.parametrize("heads,seqlen,causal", [
    (32, 900, False),   # 256 row blocks: key halves
    (33, 900, False),   # 264: one key half
    (40, 1700, True),   # 560, in pairs 280 of which a round of 256 leaves 24
    (32, 2048, True),   # 512, in pairs exactly 256
    (64, 2500, True),   # 1280: one key half
    (64, 130, False), (64, 65, True),
])
def test_forms(dtype, head_dim, heads, seqlen, causal):
    gen = torch.Generator(device="cuda").manual_seed(seqlen + heads)
    q, k, v = (torch.randn((1, heads, seqlen, head_dim), generator=gen, device="cuda").to(dtype) for _ in range(3))
    _check(flash_attention(q, k, v, causal=causal), q, k, v, dtype, causal=causal)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bias_dtype", ["same", "fp32"])
@pytest.mark.parametrize("layout", ["keys", "rows_by_4", "rows_odd", "offset", "transposed", "head"])
@pytest.mark.parametrize("sq,sk,head_dim", [(1, 1, 64), (70, 154, 64), (130, 257, 128), (33, 300, 256)])
def test_bias_layouts(dtype, bias_dtype, layout, sq, sk, head_dim):
    """Row strides of a multiple of four keys on an aligned base take four
    keys per load, other strides, offsets and orders one; both read the same
    bias.  The bias fills its storage exactly, and its last elements matter."""
    gen = torch.Generator(device="cuda").manual_seed(sk)
    q, k, v = (torch.randn((2, 3, n, head_dim), generator=gen, device="cuda").to(dtype) for n in (sq, sk, sk))
    bt = torch.float32 if bias_dtype == "fp32" else dtype
    rand = lambda *shape: (2 * torch.randn(shape, generator=gen, device="cuda")).to(bt)
    pad4 = -(-sk // 4) * 4
    bias = {
        "keys": lambda: rand(2, 1, 1, sk),
        "rows_by_4": lambda: rand(1, 3, sq, pad4)[..., :sk],
        "rows_odd": lambda: rand(1, 3, sq, pad4 + 1)[..., :sk],
        "offset": lambda: rand(2, 1, sq, pad4 + 4)[..., 1:sk + 1],
        "transposed": lambda: rand(1, 1, sk, sq).transpose(2, 3),
        "head": lambda: rand(3, sq, sk)[None],
    }[layout]()
    if sk > 8:
        bias[..., -5] = float("-inf")  # one hidden key
    out = flash_attention(q, k, v, bias=bias)
    _check(out, q, k, v, dtype, bias=bias.expand(2, 3, sq, sk).double())


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("sk,hidden", [(77, 0), (100, 0), (128, 0), (154, 38), (300, 200), (1024, 900)])
def test_few_visible_keys_round_against_their_own_tiles(head_dim, sk, hidden):
    """fp16 weights are rounded relative to the max of their own 64 keys, so
    the largest of each tile are exact.  Modelled in 64 bits with the result's
    rounding; 1.004 leaves room for ties that fp32 takes the other way (one
    max for both tiles of 128 keys is at 1.014)."""
    gen = torch.Generator(device="cuda").manual_seed(sk)
    q, k, v = (torch.randn((1, 20, n, head_dim), generator=gen, device="cuda").half() for n in (2048, sk, sk))
    bias = None
    if hidden:
        bias = torch.zeros((1, 1, 1, sk), device="cuda", dtype=torch.float16)
        bias[..., sk - hidden:] = float("-inf")
    out = flash_attention(q, k, v, bias=bias)
    n = sk - hidden
    kd, vd = k[:, :, :n].double(), v[:, :, :n].double()
    x = torch.matmul(q.double(), kd.transpose(-1, -2).contiguous()) / head_dim ** 0.5
    weights = torch.exp(x - x.amax(-1, keepdim=True))
    total = weights.sum(-1, keepdim=True)
    exact = torch.matmul(weights, vd) / total
    rounded = []
    for t in weights.split(64, -1):
        top = t.amax(-1, keepdim=True)
        rounded.append((t / top).half().double() * top)
    model = (torch.matmul(torch.cat(rounded, -1), vd) / total).half().double()
    err, floor = float((out.double() - exact).norm()), float((model - exact).norm())
    assert err <= 1.004 * floor, (err / float(exact.norm()), floor / float(exact.norm()))


@pytest.mark.parametrize("head_dim", [32, 64, 128])
@pytest.mark.parametrize("sk", [1, 65, 200, 400])
@pytest.mark.parametrize("drop", [0.0, 40.0, 4000.0])
def test_tile_maxima_far_apart(head_dim, sk, drop):
    """Scores that fall or rise by `drop` from one 64-key tile to the next
    (the row state is rescaled down and up), rows that see nothing, and rows
    whose first tiles are hidden."""
    gen = torch.Generator(device="cuda").manual_seed(sk)
    heads, sq = 300, 270
    q, k, v = (torch.randn((1, heads, n, head_dim), generator=gen, device="cuda").half() for n in (sq, sk, sk))
    step = (torch.arange(sk, device="cuda") // 64).float() * drop
    bias = torch.stack([-step, step, step.flip(0), -step.flip(0)]).repeat_interleave(68, 0)[:sq].contiguous()
    bias[5] = float("-inf")
    bias[100, :sk * 2 // 3] = float("-inf")
    out = flash_attention(q, k, v, bias=bias[None, None])
    ref = attention(q[:, :4].double(), k[:, :4].double(), v[:, :4].double(), bias=bias[None, None].double())
    err = (out[:, :4].double() - ref).norm() / ref.norm()
    assert torch.isfinite(out).all() and err <= BOUND[torch.float16], float(err)
    assert (out[:, :, 5] == 0).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim", [32, 64])
@pytest.mark.parametrize("heads,seqlen,window", [
    (200, 130, (-1, -1)), (256, 130, (-1, -1)), (257, 130, (-1, -1)),  # 400, 512 and 514 equal blocks
    (200, 300, (40, -1)), (200, 300, (-1, 40)), (200, 300, (200, -1)), (400, 400, (50, -1)), (400, 400, (50, 50)),
    (1030, 130, (-1, -1)), (1030, 130, (20, -1)),  # more than eight rounds
])
def test_equal_and_uneven_blocks(dtype, head_dim, heads, seqlen, window):
    gen = torch.Generator(device="cuda").manual_seed(heads)
    q, k, v = (torch.randn((1, heads, seqlen, head_dim), generator=gen, device="cuda").to(dtype) for _ in range(3))
    out = flash_attention(q, k, v, window_size=window)
    for h in (0, heads // 2, heads - 1):
        ref = attention(*(t[:, h:h + 1].double() for t in (q, k, v)), window=window)
        err = (out[:, h:h + 1].double() - ref).norm() / ref.norm()
        assert err <= BOUND[dtype], (h, float(err))
    assert torch.isfinite(out).all()
