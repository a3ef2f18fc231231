"""Scratch sizes of the split forward and of the head-dim-256 backward: when
blocks are shared out over workgroups, and what their states take (CPU; the
rules assume 256 compute units where no GPU says otherwise)."""

import ctypes

import pytest
import torch

from fa_rdna3 import _native

if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
    pytest.skip("sizes below are for 256 compute units", allow_module_level=True)


def _params(head_dim, heads, kv, sq, sk, causal=0, batch=1, dtype=0):
    p = _native.BwdParams()
    f = p.fwd
    f.abi_version, f.dtype, f.head_dim, f.batch = _native.ABI_VERSION, dtype, head_dim, batch
    f.heads_q, f.heads_kv, f.seqlen_q, f.seqlen_k, f.causal = heads, kv, sq, sk, causal
    return p


@pytest.mark.parametrize("head_dim,heads,sq,sk,causal,shares", [
    (512, 1, 4096, 4096, 0, 4),    # 64 workgroups (two column halves)
    (256, 1, 4096, 4096, 0, 8),
    (256, 16, 2048, 2048, 0, 1),   # one round of equal blocks
    (256, 16, 2048, 2048, 1, 2),   # one round of causal blocks
    (256, 17, 2048, 2048, 1, 1),   # more than one round
    (256, 16, 2048, 992, 1, 1),    # causal, fewer than 32 key tiles
    (512, 1, 1, 10 ** 6, 0, 16),
    (256, 1, 100, 255, 0, 2), (256, 1, 100, 224, 0, 1),
    (128, 1, 4096, 4096, 0, 1),
])
def test_forward_shares(head_dim, heads, sq, sk, causal, shares):
    p = _params(head_dim, heads, heads, sq, sk, causal)
    blocks = -(-sq // 128) * heads
    per_share = 4 * (128 * head_dim + 256 * (2 if head_dim == 512 else 1))
    want = 0 if shares == 1 else blocks * shares * per_share
    assert _native.lib().fa_fwd_workspace_bytes(ctypes.byref(p.fwd)) == want
    p.fwd.dtype = 2
    assert _native.lib().fa_fwd_workspace_bytes(ctypes.byref(p.fwd)) == 0


@pytest.mark.parametrize("heads,kv,sq,sk,causal,shares", [
    (16, 8, 2048, 2048, 1, 2), (16, 8, 2048, 2048, 0, 1), (16, 9, 2048, 2048, 1, 1), (16, 8, 1000, 2048, 1, 2),
    (16, 8, 992, 2048, 1, 1), (4, 4, 500, 500, 0, 2), (1, 1, 4096, 64, 0, 8), (1, 1, 255, 64, 0, 1),
    (8, 1, 16384, 16384, 1, 1),  # 4 GiB of dS: no shares, whole or in chunks
])
def test_backward_256_shares(heads, kv, sq, sk, causal, shares):
    p = _params(256, heads, kv, sq, sk, causal)
    ds = heads * -(-sk // 64) * -(-sq // 128) * 16384 + 1024
    part = -(-sk // 64) * kv * shares * 2 * 64 * 256 * 4 if shares > 1 else 0
    assert _native.lib().fa_bwd_workspace_bytes(ctypes.byref(p)) == ds + part
    p.fwd.head_dim = 512
    assert _native.lib().fa_bwd_workspace_bytes(ctypes.byref(p)) == 0
