"""fp32 forward and backward, with the key or query range split between two
halves of a workgroup and, on grids that fill the chip, without, against
64-bit attention at tile edges."""

import pytest
import torch

from attn_refs import attention, grads
from fa_rdna3 import flash_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("head_dim", [32, 64, 128, 512])
@pytest.mark.parametrize("heads,kv,sq,sk,opts", [
    (2, 2, 1, 1, {}), (2, 1, 31, 33, {}), (2, 2, 64, 64, {"causal": True}), (4, 2, 65, 63, {"causal": True}),
    (2, 2, 129, 31, {}), (4, 1, 200, 333, {"causal": True}), (2, 2, 300, 300, {"window": (40, 10)}),
    (2, 2, 150, 150, {"softcap": 8.0, "causal": True}),
    # 200 to 900 blocks of 128 rows, odd lengths: whole workgroups where they
    # are the faster form (see f32_halves), halves otherwise
    (100, 50, 131, 70, {}), (150, 150, 140, 129, {}), (260, 130, 65, 131, {}), (300, 300, 129, 31, {"softcap": 8.0}),
    (300, 100, 150, 150, {"causal": True}), (300, 300, 257, 257, {"causal": True}),
    (260, 260, 200, 200, {"window": (30, -1)}), (260, 260, 200, 200, {"causal": True, "window": (30, -1)}),
])
def test_matches_64_bit(head_dim, heads, kv, sq, sk, opts):
    gen = torch.Generator(device="cuda").manual_seed(sq + sk)
    rand = lambda h, n: torch.randn((2, n, h, head_dim), generator=gen, device="cuda").transpose(1, 2)
    q, k, v, do = rand(heads, sq), rand(kv, sk), rand(kv, sk), rand(heads, sq)
    opts = dict(opts)
    window = opts.pop("window", (-1, -1))
    ours = lambda a, b, c: flash_attention(a, b, c, window_size=window, **opts)
    exact = lambda a, b, c: attention(a, b, c, window=window, **opts)
    got = (ours(q, k, v),) + grads(ours, q, k, v, do)
    d = [t.double() for t in (q, k, v, do)]
    want = (exact(*d[:3]),) + grads(exact, *d)
    # fp32 sums of up to D or S terms: error of at most sqrt(n) units of 2^-24
    # on each of four chained sums, doubled for the exponentials.
    bound = 2 * 4 * max(sk, sq, head_dim) ** 0.5 * 2.0 ** -24
    scale = max(float(w.norm()) for w in want)
    for g, w in zip(got, want):
        assert torch.isfinite(g).all()
        # With one visible key dQ and dK are exactly zero: dP - delta cancels
        # sums of the size of the other results, whose error is then left.
        size = float(w.norm())
        assert float((g.double() - w).norm()) <= bound * (size if size > 1e-6 * scale else scale)
