"""Scratch sizes of the split forward and of the head-dim-256 backward: when
blocks are shared out over workgroups, and what their states take (CPU; the
rules assume 256 compute units where no GPU says otherwise)."""

import ctypes

import pytest
import torch

from fa_rdna3 import _native

if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
    pytest.skip("sizes below are for 256 compute units", allow_module_level=True)


def _params(head_dim, heads, kv, sq, sk, causal=0, batch=1, dtype=0, window=(-1, -1)):
    p = _native.BwdParams()
    f = p.fwd
    f.abi_version, f.dtype, f.head_dim, f.batch = _native.ABI_VERSION, dtype, head_dim, batch
    f.heads_q, f.heads_kv, f.seqlen_q, f.seqlen_k, f.causal = heads, kv, sq, sk, causal
    f.window_left, f.window_right = window  # (-1: none; 0 would be a window of one key)
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


@pytest.mark.parametrize("sq,sk,causal,window,shares", [
    (4096, 4096, 0, (64, 0), 1),       # 193 keys at most: under two shares of four 32-key tiles
    (4096, 4096, 0, (200, 100), 3),    # 429 keys, 14 tiles
    (4096, 4096, 1, (400, 50), 4),     # causal: 528 keys, 17 tiles
    (4096, 4096, 0, (-1, 64), 8), (4096, 4096, 0, (64, -1), 8),  # one side: some block sees all keys
    (100, 8000, 0, (64, -1), 1),       # the last 164 keys
    (100, 8000, 0, (10000, 10000), 16),
])
def test_forward_shares_count_visible_keys(sq, sk, causal, window, shares):
    p = _params(256, 1, 1, sq, sk, causal, window=window)
    want = 0 if shares == 1 else -(-sq // 128) * shares * 4 * (128 * 256 + 256)
    assert _native.lib().fa_fwd_workspace_bytes(ctypes.byref(p.fwd)) == want


@pytest.mark.parametrize("heads,sq,sk,causal,window,shares", [
    (1, 4096, 256, 0, (64, 0), 1),     # 128 queries at most see a block of 64 keys
    (1, 4096, 256, 0, (300, 300), 2),  # 664 of the 4096, but 556 queries reach the 256 keys: 17 steps
    (1, 4096, 4096, 1, (1000, -1), 4),
    (1, 4096, 256, 1, (-1, -1), 1),    # only the last 256 queries see a key
    (8, 2048, 2048, 1, (-1, -1), 2), (8, 2048, 2048, 1, (300, -1), 1), (8, 2048, 2048, 1, (4000, -1), 2),
])
def test_backward_256_shares_count_visible_queries(heads, sq, sk, causal, window, shares):
    p = _params(256, heads, heads, sq, sk, causal, window=window)
    ds = heads * -(-sk // 64) * -(-sq // 128) * 16384 + 1024
    part = -(-sk // 64) * heads * shares * 2 * 64 * 256 * 4 if shares > 1 else 0
    assert _native.lib().fa_bwd_workspace_bytes(ctypes.byref(p)) == ds + part
    assert _native.lib().fa_bwd_workspace_min_bytes(ctypes.byref(p)) == ds  # the dS path without shares
