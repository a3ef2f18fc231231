"""What a user of this package has it do, as timed cases over its public entry points.

A case is a dict of plain values; `kind` says which entry point it goes through:

* ``forward``   flash_attention without gradients (text, image, latent and prompt passes)
* ``train``     flash_attention forward and backward
* ``varlen``    flash_attention_varlen forward and backward
* ``decode``    flash_attention_decode on a contiguous cache
* ``paged``     flash_attention_decode_paged / _paged_multi on a block-table cache
* ``append``    flash_attention_with_kvcache: append the step's rows, then attend

`listed` holds the fixed cases and `draw` further ones of the same ranges;
`prepare`, `run`, `work`, `tolerance` and `exact` take any of them.
"""

import math
import os
import sys

import torch

_PACKAGE = os.path.abspath("flash-attention-rdna3_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(1, _PACKAGE)

import fa_rdna3  # noqa: E402

_DTYPE = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
_BYTES = {"fp16": 2, "bf16": 2, "fp32": 4, "fp8": 1}


def _dense(kind, dtype, batch, heads, kv_heads, seq_q, seq_k, dim, causal=False, window=-1, softcap=0.0,
           alibi=False, bias="", layout="bhsd"):
    return {"kind": kind, "dtype": dtype, "batch": batch, "heads": heads, "kv_heads": kv_heads, "seq_q": seq_q,
            "seq_k": seq_k, "dim": dim, "causal": causal, "window": window, "softcap": softcap, "alibi": alibi,
            "bias": bias, "layout": layout}


def _varlen(dtype, count, shortest, longest, heads, kv_heads, dim, causal=True, window=-1, softcap=0.0):
    return {"kind": "varlen", "dtype": dtype, "count": count, "shortest": shortest, "longest": longest,
            "heads": heads, "kv_heads": kv_heads, "dim": dim, "causal": causal, "window": window,
            "softcap": softcap}


def _decode(dtype, batch, heads, kv_heads, rows, keys, dim, ragged=True):
    return {"kind": "decode", "dtype": dtype, "batch": batch, "heads": heads, "kv_heads": kv_heads, "rows": rows,
            "keys": keys, "dim": dim, "ragged": ragged}


def _paged(dtype, cache, batch, heads, kv_heads, rows, keys, dim, page, ragged=False):
    return {"kind": "paged", "dtype": dtype, "cache": cache, "batch": batch, "heads": heads, "kv_heads": kv_heads,
            "rows": rows, "keys": keys, "dim": dim, "page": page, "ragged": ragged}


def _append(dtype, batch, heads, kv_heads, rows, keys, dim):
    return {"kind": "append", "dtype": dtype, "batch": batch, "heads": heads, "kv_heads": kv_heads, "rows": rows,
            "keys": keys, "dim": dim}


def listed():
    return [
        # The smallest call a program makes over and over: a text encoder's
        # layer on one 77-token prompt.  Launch and host latency.
        {"name": "text_77", **_dense("forward", "fp16", 1, 8, 8, 77, 77, 64, causal=True)},
        # An image model's cross attention: many image tokens against a
        # padded prompt, the padding masked by an additive bias.
        {"name": "cross_masked", **_dense("forward", "fp16", 2, 10, 10, 4096, 154, 64, bias="keys", layout="bshd")},
        # An image model's self attention (no mask), heads within a row as
        # the projections leave them.
        {"name": "image_self", **_dense("forward", "fp16", 2, 10, 10, 4096, 4096, 64, layout="bshd")},
        # The single wide head of an image autoencoder.
        {"name": "latent_wide", **_dense("forward", "fp16", 1, 1, 1, 4096, 4096, 512)},
        # Prompt pass of a long context, grouped heads, a length that is no
        # multiple of a tile.
        {"name": "prefill_long", **_dense("forward", "bf16", 1, 32, 8, 8000, 8000, 128, causal=True)},
        # The headline training step of this repository's benchmark.
        {"name": "train_dense", **_dense("train", "fp16", 2, 16, 16, 2048, 2048, 128, causal=True)},
        # Training with wide heads and grouped KV.
        {"name": "train_wide", **_dense("train", "bf16", 1, 16, 8, 2048, 2048, 256, causal=True)},
        # Training in full precision (the package's fp32 inputs), a ragged length.
        {"name": "train_fp32", **_dense("train", "fp32", 1, 16, 16, 1000, 1000, 64)},
        # Packed training batch with a sliding window and softcap.
        {"name": "train_packed", **_varlen("bf16", 16, 128, 2048, 32, 8, 128, window=1024, softcap=50.0)},
        # One token per sequence against contiguous caches of uneven length.
        {"name": "decode_ragged", **_decode("fp16", 4, 32, 8, 1, 8192, 128)},
        # One token per sequence against a paged cache.
        {"name": "decode_pages", **_paged("fp16", "fp16", 4, 32, 8, 1, 16384, 128, 16)},
        # A serving step that appends its new rows and attends, short caches.
        {"name": "decode_append", **_append("bf16", 8, 32, 8, 4, 2000, 128)},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    what = rng.randrange(12)
    half = rng.choice(["fp16", "bf16"])
    if what == 0:  # short prompts
        s = _log_int(rng, 8, 256)
        return _dense("forward", half, rng.randint(1, 4), 8, 8, s, s, rng.choice([32, 64, 64, 128]),
                      causal=rng.random() < 0.7)
    if what == 1:  # cross attention with masks
        return _dense("forward", half, rng.randint(1, 2), rng.choice([5, 8, 10, 20]), 0, _log_int(rng, 64, 4096),
                      _log_int(rng, 16, 512), rng.choice([40, 64, 80, 128]), bias=rng.choice(["keys", "full"]),
                      layout="bshd")
    if what == 2:  # image self attention, head dims that need padding among them
        s = _log_int(rng, 64, 4096)
        return _dense("forward", half, rng.randint(1, 2), rng.choice([8, 10, 20]), 0, s, s,
                      rng.choice([40, 64, 64, 80, 128, 160]), layout=rng.choice(["bshd", "bhsd"]))
    if what == 3:  # wide heads, forward
        s = _log_int(rng, 64, 4096)
        return _dense("forward", half, rng.randint(1, 2), rng.choice([1, 2, 4]), 0, s, s, rng.choice([256, 512, 512]),
                      causal=rng.random() < 0.3)
    if what == 4:  # prompt pass
        s = _log_int(rng, 256, 8000)
        kv = rng.choice([4, 8])
        return _dense("forward", half, 1, kv * rng.choice([1, 2, 4]), kv, s, s, rng.choice([64, 128, 128]),
                      causal=True, window=rng.choice([-1, -1, 1024]), softcap=rng.choice([0.0, 0.0, 30.0]))
    if what == 5:  # training
        s = _log_int(rng, 64, 2048)
        kv = rng.choice([4, 8, 16])
        return _dense("train", half, rng.randint(1, 2), kv * rng.choice([1, 2]) if kv < 16 else 16, kv, s, s,
                      rng.choice([32, 64, 128, 128]), causal=rng.random() < 0.7, window=rng.choice([-1, -1, 300]),
                      softcap=rng.choice([0.0, 0.0, 50.0]), alibi=rng.random() < 0.25,
                      layout=rng.choice(["bhsd", "bshd"]))
    if what == 6:  # training with wide heads
        s = _log_int(rng, 64, 2048)
        kv = rng.choice([2, 4, 8])
        return _dense("train", half, 1, kv * rng.choice([1, 2]), kv, s, s, rng.choice([256, 256, 256, 512]),
                      causal=rng.random() < 0.7, softcap=rng.choice([0.0, 0.0, 50.0]))
    if what == 7:  # full precision
        s = _log_int(rng, 32, 1000)
        return _dense("train", "fp32", 1, rng.choice([8, 16]), 0, s, s, rng.choice([32, 64, 64, 128]),
                      causal=rng.random() < 0.5)
    if what == 8:  # packed training
        kv = rng.choice([2, 4, 8])
        return _varlen(half, rng.randint(4, 16), _log_int(rng, 16, 128), _log_int(rng, 192, 2048),
                       kv * rng.choice([1, 4]), kv, rng.choice([64, 128]), causal=rng.random() < 0.8,
                       window=rng.choice([-1, 1024]), softcap=rng.choice([0.0, 50.0]))
    kv = rng.choice([4, 8])
    if what == 9:
        return _decode(half, _log_int(rng, 1, 16), kv * rng.choice([1, 4, 8]), kv, rng.choice([1, 1, 2, 5]),
                       _log_int(rng, 200, 8192), rng.choice([64, 128, 128, 256]), ragged=rng.random() < 0.7)
    if what == 10:
        return _paged(half, rng.choice([half, half, "fp8"]), _log_int(rng, 1, 8), kv * rng.choice([1, 4, 8]), kv,
                      rng.choice([1, 1, 4]), _log_int(rng, 200, 16384), rng.choice([64, 128, 128, 256]),
                      rng.choice([8, 16, 16, 64, 256]), ragged=rng.random() < 0.5)
    return _append(half, _log_int(rng, 1, 16), kv * rng.choice([1, 4]), kv, rng.choice([1, 2, 4]),
                   _log_int(rng, 200, 4000), rng.choice([64, 128, 128]))


# --- inputs -----------------------------------------------------------------

def _kv_heads(case):
    return case["kv_heads"] or case["heads"]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _lengths(count, shortest, longest):
    # Uneven lengths fixed by the case (an even spread, visited out of order),
    # so a case costs the same for every seed.
    step = 7 if count % 7 else 5
    return [shortest + (longest - shortest) * ((i * step) % count) // max(count - 1, 1) for i in range(count)]


def _cache_lengths(case):
    keys, batch = case["keys"], case["batch"]
    if not case.get("ragged", True):
        return [keys] * batch
    if batch == 1:
        return [keys * 7 // 8]
    return _lengths(batch, keys * 5 // 8, keys * 15 // 16)


def _dense_inputs(case, seed):
    gen, dtype = _gen(seed), _DTYPE[case["dtype"]]
    b, d = case["batch"], case["dim"]

    def tensor(heads, seq):
        if case["layout"] == "bshd":
            return _randn(gen, (b, seq, heads, d), dtype).transpose(1, 2)
        return _randn(gen, (b, heads, seq, d), dtype)

    q = tensor(case["heads"], case["seq_q"])
    k = tensor(_kv_heads(case), case["seq_k"])
    v = tensor(_kv_heads(case), case["seq_k"])
    bias = None
    if case["bias"] == "keys":  # padding mask: the last quarter of the first sequence's keys is hidden
        bias = torch.zeros((b, 1, 1, case["seq_k"]), device="cuda", dtype=dtype)
        bias[0, :, :, case["seq_k"] - case["seq_k"] // 4:] = float("-inf")
    elif case["bias"] == "full":
        bias = _randn(gen, (1, case["heads"], case["seq_q"], case["seq_k"]), dtype)
    slopes = fa_rdna3.alibi_slopes(case["heads"], device="cuda") if case["alibi"] else None
    grad = tensor(case["heads"], case["seq_q"]) if case["kind"] == "train" else None
    return q, k, v, bias, slopes, grad


def _varlen_inputs(case, seed):
    gen, dtype = _gen(seed), _DTYPE[case["dtype"]]
    lens = _lengths(case["count"], case["shortest"], case["longest"])
    total, d = sum(lens), case["dim"]
    q = _randn(gen, (total, case["heads"], d), dtype)
    k = _randn(gen, (total, case["kv_heads"], d), dtype)
    v = _randn(gen, (total, case["kv_heads"], d), dtype)
    grad = _randn(gen, (total, case["heads"], d), dtype)
    return lens, q, k, v, grad


def _decode_inputs(case, seed):
    gen, dtype = _gen(seed), _DTYPE[case["dtype"]]
    b, d = case["batch"], case["dim"]
    q = _randn(gen, (b, case["heads"], case["rows"], d), dtype)
    k = _randn(gen, (b, case["kv_heads"], case["keys"], d), dtype)
    v = _randn(gen, (b, case["kv_heads"], case["keys"], d), dtype)
    return gen, q, k, v


_FP8_SCALE = (0.5, 0.25)  # K / k_scale and V / v_scale are what an fp8 cache holds


def _paged_inputs(case, seed):
    gen, dtype = _gen(seed), _DTYPE[case["dtype"]]
    b, d, page = case["batch"], case["dim"], case["page"]
    per_seq = -(-case["keys"] // page)
    q = _randn(gen, (b, case["heads"], case["rows"], d), dtype)
    shape = (b * per_seq, page, case["kv_heads"], d)
    k, v = _randn(gen, shape, torch.float32), _randn(gen, shape, torch.float32)
    if case["cache"] == "fp8":
        k = (k / _FP8_SCALE[0]).to(torch.float8_e4m3fn)
        v = (v / _FP8_SCALE[1]).to(torch.float8_e4m3fn)
    else:
        k, v = k.to(dtype), v.to(dtype)
    table = torch.randperm(b * per_seq, generator=gen, device="cuda").to(torch.int32).view(b, per_seq)
    return q, k, v, table


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("forward", "train"):
        q, k, v, bias, slopes, grad = _dense_inputs(case, seed)
        args = dict(causal=case["causal"], window_size=(case["window"], -1), softcap=case["softcap"], bias=bias,
                    alibi_slopes=slopes)
        if kind == "train":
            q, k, v = (t.requires_grad_() for t in (q, k, v))
        return {"kind": kind, "qkv": (q, k, v), "grad": grad, "args": args}
    if kind == "varlen":
        lens, q, k, v, grad = _varlen_inputs(case, seed)
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        cu = _int32(cu)
        args = dict(causal=case["causal"], window_size=(case["window"], -1), softcap=case["softcap"])
        return {"kind": kind, "qkv": tuple(t.requires_grad_() for t in (q, k, v)), "grad": grad, "cu": cu,
                "longest": max(lens), "args": args}
    if kind == "decode":
        _, q, k, v = _decode_inputs(case, seed)
        lens = _int32(_cache_lengths(case)) if case["ragged"] else None
        return {"kind": kind, "qkv": (q, k, v), "lens": lens}
    if kind == "append":
        gen, q, k, v = _decode_inputs(case, seed)
        shape = (case["batch"], case["kv_heads"], case["rows"], case["dim"])
        return {"kind": kind, "qkv": (q, k, v), "lens": _int32([n - case["rows"] for n in _cache_lengths(case)]),
                "new": (_randn(gen, shape, q.dtype), _randn(gen, shape, q.dtype))}
    q, k, v, table = _paged_inputs(case, seed)
    args = dict(max_context_len=case["keys"])
    if case["cache"] == "fp8":
        args.update(k_scale=_FP8_SCALE[0], v_scale=_FP8_SCALE[1])
    return {"kind": kind, "qkv": (q if case["rows"] > 1 else q.squeeze(2), k, v), "table": table,
            "lens": _int32(_cache_lengths(case)), "args": args}


def run(state):
    kind = state["kind"]
    q, k, v = state["qkv"]
    if kind == "forward":
        return fa_rdna3.flash_attention(q, k, v, **state["args"])
    if kind == "train":
        out = fa_rdna3.flash_attention(q, k, v, **state["args"])
        return (out.detach(),) + torch.autograd.grad(out, (q, k, v), state["grad"])
    if kind == "varlen":
        out = fa_rdna3.flash_attention_varlen(q, k, v, state["cu"], state["cu"], state["longest"], state["longest"],
                                              **state["args"])
        return (out.detach(),) + torch.autograd.grad(out, (q, k, v), state["grad"])
    if kind == "decode":
        return fa_rdna3.flash_attention_decode(q, k, v, cache_seqlens=state["lens"])
    if kind == "append":
        out = fa_rdna3.flash_attention_with_kvcache(q, k, v, *state["new"], cache_seqlens=state["lens"], causal=True)
        return out, k, v
    if q.dim() == 4:
        return fa_rdna3.flash_attention_decode_paged_multi(q, k, v, state["table"], state["lens"], **state["args"])
    return fa_rdna3.flash_attention_decode_paged(q, k, v, state["table"], state["lens"], **state["args"])


# --- what a pass cannot do without ------------------------------------------

def _pairs(seq_q, seq_k, causal, window):
    """Visible (query, key) pairs; query i sits at key position i + seq_k - seq_q."""
    total, off = 0, seq_k - seq_q
    for i in range(seq_q):
        hi = min(seq_k - 1, i + off) if causal else seq_k - 1
        lo = max(0, i + off - window) if window >= 0 else 0
        total += max(0, hi - lo + 1)
    return total


def work(case):
    kind, d, heads, size = case["kind"], case["dim"], case["heads"], _BYTES[case["dtype"]]
    kv = _kv_heads(case)
    if kind in ("forward", "train", "varlen"):
        if kind == "varlen":
            lens = _lengths(case["count"], case["shortest"], case["longest"])
            pairs = heads * sum(_pairs(n, n, case["causal"], case["window"]) for n in lens)
            rows_q = rows_k = sum(lens)
        else:
            pairs = case["batch"] * heads * _pairs(case["seq_q"], case["seq_k"], case["causal"], case["window"])
            rows_q, rows_k = case["batch"] * case["seq_q"], case["batch"] * case["seq_k"]
        tensor_q, tensor_k = rows_q * heads * d * size, rows_k * kv * d * size
        moved, flops = 2 * tensor_q + 2 * tensor_k, 4 * d * pairs  # q, k, v in; out
        if kind != "forward":  # also dout in, dq, dk, dv out; the backward's five products
            moved, flops = moved + 2 * tensor_q + 2 * tensor_k, flops + 10 * d * pairs
        if case.get("bias") == "keys":
            moved += case["batch"] * case["seq_k"] * size
        elif case.get("bias") == "full":
            moved += heads * case["seq_q"] * case["seq_k"] * size
        return {"bytes": moved, "flops": flops}
    keys = sum(_cache_lengths(case))
    cache = _BYTES[case.get("cache", case["dtype"])]
    moved = 2 * keys * kv * d * cache + 2 * case["batch"] * heads * case["rows"] * d * size
    if kind == "append":  # the new rows are read and written; the causal rows see what is there
        moved += 2 * case["batch"] * kv * case["rows"] * d * size
    return {"bytes": moved, "flops": 4 * d * heads * case["rows"] * keys}


# --- accuracy ---------------------------------------------------------------

def tolerance(case):
    # About four times what the path measured against `exact`: 2.3e-4 to
    # 3.3e-4 in fp16, 1.6e-3 to 2.5e-3 in bf16 (the results and the operands
    # of the second products are rounded to 16 bits), 6e-7 to 8e-7 in fp32.
    return {"rel": {"fp16": 1.3e-3, "bf16": 1e-2, "fp32": 3e-6}[case["dtype"]]}


def _attend(q, k, v, scale, causal, window, softcap, slope, bias, grad):
    """One head in 64 bits: out, or (out, dq, dk, dv) when `grad` is given."""
    seq_q, seq_k = q.shape[0], k.shape[0]
    raw = q @ k.t() * scale
    x = softcap * torch.tanh(raw / softcap) if softcap > 0 else raw
    rows = torch.arange(seq_q, device=q.device)[:, None] + (seq_k - seq_q)
    cols = torch.arange(seq_k, device=q.device)[None, :]
    if bias is not None:
        x = x + bias
    if slope is not None:
        x = x - slope * (rows - cols).abs()
    if causal:
        x = x.masked_fill(cols > rows, float("-inf"))
    if window >= 0:
        x = x.masked_fill(cols < rows - window, float("-inf"))
    p = torch.softmax(x, dim=-1)
    p = torch.nan_to_num(p, nan=0.0)  # a row that sees nothing is zero
    out = p @ v
    if grad is None:
        return out
    dv = p.t() @ grad
    ds = p * (grad @ v.t() - (out * grad).sum(-1, keepdim=True))
    if softcap > 0:
        ds = ds * (1 - torch.tanh(raw / softcap) ** 2)
    return out, ds @ k * scale, ds.t() @ q * scale, dv


def _attend_heads(q, k, v, case, slopes, bias, grad):
    """(heads, seq, dim) tensors of one sequence, head by head in 64 bits."""
    group, scale = q.shape[0] // k.shape[0], 1.0 / math.sqrt(q.shape[-1])
    outs, dqs = [], []
    dk, dv = torch.zeros_like(k, dtype=torch.float64), torch.zeros_like(v, dtype=torch.float64)
    for h in range(q.shape[0]):
        got = _attend(q[h].double(), k[h // group].double(), v[h // group].double(), scale, case["causal"],
                      case["window"], case["softcap"], None if slopes is None else slopes[h].double(),
                      None if bias is None else bias[h].double(), None if grad is None else grad[h].double())
        if grad is None:
            outs.append(got)
        else:
            outs.append(got[0])
            dqs.append(got[1])
            dk[h // group] += got[2]
            dv[h // group] += got[3]
    return torch.stack(outs), (torch.stack(dqs) if dqs else None), dk, dv


def _attend_cache(q, k, v, rows_see):
    """(heads, rows, dim) queries against (kv_heads, keys, dim); rows_see[i] keys for row i."""
    group, scale = q.shape[0] // k.shape[0], 1.0 / math.sqrt(q.shape[-1])
    q, k, v = q.double(), k.double(), v.double()
    x = torch.matmul(q.view(k.shape[0], -1, q.shape[-1]), k.transpose(1, 2).contiguous()) * scale
    x = x.view(q.shape[0], q.shape[1], -1)
    cols = torch.arange(k.shape[1], device=q.device)
    x = x.masked_fill(cols[None, None, :] >= rows_see[None, :, None], float("-inf"))
    p = torch.softmax(x, dim=-1).view(k.shape[0], group * q.shape[1], -1)
    return torch.matmul(p, v).view(q.shape)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("forward", "train"):
        q, k, v, bias, slopes, grad = _dense_inputs(case, seed)
        if bias is not None:
            bias = bias.expand(case["batch"], case["heads"], case["seq_q"], case["seq_k"])
        got = [_attend_heads(q[b], k[b], v[b], case, slopes, None if bias is None else bias[b],
                             None if grad is None else grad[b]) for b in range(case["batch"])]
        if kind == "forward":
            return torch.stack([g[0] for g in got])
        return tuple(torch.stack([g[i] for g in got]) for i in range(4))
    if kind == "varlen":
        lens, q, k, v, grad = _varlen_inputs(case, seed)
        got, at = [], 0
        for n in lens:
            part = [t[at:at + n].transpose(0, 1) for t in (q, k, v, grad)]
            got.append(_attend_heads(part[0], part[1], part[2], case, None, None, part[3]))
            at += n
        return tuple(torch.cat([g[i].transpose(0, 1) for g in got]) for i in range(4))
    lens, rows = _cache_lengths(case), case["rows"]
    if kind == "paged":
        q, k, v, table = _paged_inputs(case, seed)
        scale = _FP8_SCALE if case["cache"] == "fp8" else (1.0, 1.0)
    else:
        gen, q, k, v = _decode_inputs(case, seed)
    if kind == "append":
        shape = (case["batch"], case["kv_heads"], rows, case["dim"])
        new = _randn(gen, shape, q.dtype), _randn(gen, shape, q.dtype)
    outs = []
    for b, n in enumerate(lens):
        if kind == "paged":
            kb, vb = (t[table[b].long()].double().mul(s).flatten(0, 1)[:n].transpose(0, 1)
                      for t, s in zip((k, v), scale))
        else:
            if kind == "append":
                k[b, :, n - rows:n], v[b, :, n - rows:n] = new[0][b], new[1][b]
            kb, vb = k[b, :, :n], v[b, :, :n]
        last = torch.arange(rows, device="cuda") + n - rows + 1 if kind != "decode" else torch.full((rows,), n, device="cuda")
        outs.append(_attend_cache(q[b], kb, vb, last))
    out = torch.stack(outs)
    if kind == "append":
        return out, k.double(), v.double()
    return out if kind == "decode" or rows > 1 else out.squeeze(2)
