"""Choice of the forward's form on a dense grid, and its aligned bias loads,
against 64-bit attention."""

import pytest
import torch

from attn_refs import attention
from fa_rdna3 import flash_attention

pytestmark = pytest.mark.gpu
# Relative 2-norm: four 16-bit roundings of at most one unit on a result's path.
BOUND = {torch.float16: 4 * 2.0 ** -11, torch.bfloat16: 4 * 2.0 ** -8}


def _check(out, q, k, v, dtype, rows=slice(None), **opts):
    ref = attention(q[:1].double(), k[:1].double(), v[:1].double(), **opts)
    err = (out[:1].double() - ref).norm() / ref.norm()
    assert torch.isfinite(out).all() and err <= BOUND[dtype], float(err)


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
    _check(out, q, k, v, dtype, bias=bias.expand(2, 3, sq, sk)[:1].double())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim", [32, 64])
@pytest.mark.parametrize("heads,seqlen,window", [
    (1020, 130, (-1, -1)), (1024, 130, (50, 50)),
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
