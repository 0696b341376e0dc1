"""Shared body of the attention types that keep attention sinks plus a sliding window
("stream-llm", "infinite-lm": inf_llm/attention/stream_llm.py:6-111, infinite_lm.py:6-100) and of
plain causal attention ("origin": origin.py:4-79): one native call per layer call (infllm_window_forward).

The reference re-rotates the whole cached window on every call (positions relative to the window).
Here every key is rotated once, at its absolute stream position, when it arrives, and the cache keeps
the rotated rows: q.k then depends on the position difference only, which is what the window-relative
tables produce.  The sink stage uses one fixed query angle:

  infinite-lm   query at position n_local - 1, sink keys un-rotated        (infinite_lm.py:59-66)
  stream-llm    query at position n_local + n_init - 1, sink key j at j     (stream_llm.py:62-73)

A sink key j is visible to the query at stream position p in that stage iff p - j >= n_local (otherwise it
is still inside the window and the local stage sees it).  The cache tuple keeps the reference's first three
fields (keys, values, tokens seen); a fourth holds the un-rotated sink keys when the type needs them.

A cache that still holds every token grows in place: its tensors are the filled part of buffers with room behind it
(a quarter more), and the next call writes its rows there instead of copying everything - when the cache it is given is
the newest one of those buffers.  An older one (a second continuation of the same prompt) gets buffers of its own.  A cache
and the one it continues then share memory: a caller that writes into a cache's tensors clones them first.
"""
import functools
import math
import struct

import torch

from .. import _lib
from ..ops import HEAD_DIM, _stream, rows16
from ._rows import check_head_dim, narrow, wide_inv_freq, widen

_KINDS = {"origin": 0, "stream-llm": 1, "infinite-lm": 2}
_ARGS = struct.Struct("@3P9q8i2qPd2P4q2P4q2i4P2iPqP3qPfi")        # infllm_window_args
_SPLIT_ROWS = 131072                # partial rows that key splits of a call of several queries may take

def _capturing(dev):
    return dev.type == "cuda" and torch.cuda.is_current_stream_capturing()


_STEP_BYTES = 4 << 20               # scratch of a call of one token that is kept for the next one, at most


@functools.lru_cache(maxsize=64)
def _step_bytes(kind, batch, heads, dim):
    """scratch of a call of one token: its rotated queries, up to 64 key splits of its rows, their sums"""
    rows = batch * heads
    splits = 64 * rows if rows <= 2048 else _SPLIT_ROWS if 2 * rows <= _SPLIT_ROWS else 0
    return (2 if kind else 1) * rows * dim * 2 + splits * (2 * dim + 4) + 4 * rows


def _take_words(past_k, n, step_bytes, dev, stream):
    """((tensor, address of n words or more in which a step counts its finished key splits, their number, the stream they belong to,
    address and size of a scratch behind them: of step_bytes or more, or, where that is more than _STEP_BYTES, of any size) and whether
    the call has to clear the words, or None: it counts in words of its own scratch.

    The words are zero between the launches that use them, and only one call has them and the scratch at a time: it takes them off the
    storage of the cache it continues (one operation, whichever threads go on from that cache) and leaves them with the cache it
    returns.  Their launches are then in the order of their stream, which is also the one that the allocator gives them out again in.
    Inside a capture there are none: its launches run when and where the graph is replayed, beside whatever else counts by then
    (and the default stream, 0, cannot be captured)."""
    if stream and _capturing(dev):
        return None, 0
    if step_bytes > _STEP_BYTES:
        step_bytes = 0
    if past_k is not None:
        held = past_k.untyped_storage().__dict__.pop("_infllm_words", None)
        if held is not None and held[3] == stream and held[2] >= n and held[5] >= step_bytes:
            return held, 0
    head = -(-4 * n // 256) * 256
    t = torch.empty(((head + step_bytes + 3) // 4,), dtype=torch.int32, device=dev)
    ptr = t.data_ptr()
    return (t, ptr, n, stream, ptr + head, step_bytes), 1


def _ticket(words):
    return words[1] if words is not None else 0


def _cache_rows(t, dim):
    """(a cached tensor as the native call takes it: rows next to each other, its address, batch and head strides)"""
    sb, sh, sl, inner = t.stride()
    ptr = t.data_ptr()
    if inner != 1 or sl != dim or (sb | sh) & 7 or ptr & 15:
        t = t.clone(memory_format=torch.contiguous_format)
        sb, sh, _, _ = t.stride()
        ptr = t.data_ptr()
    return t, ptr, sb, sh


def _heads(x, batch, length, heads, dim):
    """(tensor that is kept alive, address, batch, head and row strides) of projected rows [batch, length, heads * dim]"""
    if x.shape != (batch, length, heads * dim):
        x = x.view(batch, length, heads * dim)
    x = rows16(x)
    sb, sl, _ = x.stride()
    return x, x.data_ptr(), sb, dim, sl


def _wide_heads(x, batch, length, heads, dim):
    x = widen(x.view(batch, length, heads, dim), dim)
    return x, x.data_ptr(), x.stride(0), x.stride(2), x.stride(1)


def _on_gpu(x):
    return x.is_cuda


def _check_rows(q, k, v):
    """projected rows: the native call takes them by address and reads bfloat16 on the GPU"""
    bf, dev = torch.bfloat16, q.device
    if q.dtype is not bf or k.dtype is not bf or v.dtype is not bf:
        raise TypeError(f"the HIP attention path computes in bfloat16, got {q.dtype}, {k.dtype}, {v.dtype}")
    if k.device != dev or v.device != dev or not _on_gpu(q):
        raise ValueError(f"q, k and v must be on one GPU, got {q.device}, {k.device}, {v.device}")


def _check_cached(k, v, raw, batch, heads, dim, device):
    """The rows of a cache that the call's rows can join.  The native call takes addresses and strides and cannot see how far a
    tensor reaches, so whatever joining the tensors would refuse - another batch, head count, width, type or device - is refused
    here."""
    bf, shape = torch.bfloat16, k.shape
    rows = shape[2] if len(shape) == 4 else -1
    if shape != (batch, heads, rows, dim) or v.shape != shape:
        raise ValueError(f"cached keys {tuple(shape)} and values {tuple(v.shape)} do not fit a call of batch {batch}, {heads} kv heads of {dim}")
    if k.dtype is not bf or v.dtype is not bf or k.device != device or v.device != device:
        raise ValueError(f"the cache must be bfloat16 on {device}, got {k.dtype} on {k.device} and {v.dtype} on {v.device}")
    if raw is not None and (raw.dim() != 4 or raw.shape != (batch, heads, raw.size(2), dim) or raw.dtype is not bf or raw.device != device):
        raise ValueError(f"un-rotated sinks {tuple(raw.shape)}, {raw.dtype} on {raw.device}, do not fit a call of batch {batch}, {heads} kv heads of {dim}")
    return rows


def _call(kind, n_local, n_init, query, key_value, position_bias, past, project_q, project_k, project_v, dim_head, num_heads, num_heads_kv):
    """Output rows [batch, len_q, heads * dim] and the new (keys, values, tokens seen, un-rotated sinks)."""
    (batch, len_q), n_new = query.shape[:2], key_value.size(1)
    xq, xk, xv = project_q(query), project_k(key_value), project_v(key_value)
    check_head_dim(dim_head)
    dev = xq.device
    # A step that goes on from a cache as the call before left it is csrc/host.cpp's: behind a short past it is bound by this code (causal
    # step behind 300 to 2,000 tokens 21.7 -> 12.4 us, sinks + window of 512 and 1,200 22.1 -> 13.5).
    if len_q == 1 and n_new == 1 and past is not None and dim_head in (64, HEAD_DIM) and _on_gpu(xq):
        stream = _stream()
        if not (stream and _capturing(dev)):
            done = _lib.host().step(kind, n_local, n_init, xq, xk, xv, past, position_bias.inv_freq, position_bias.distance_scale, batch, num_heads, num_heads_kv,
                                    dim_head, _step_bytes(kind, batch, num_heads, dim_head), stream, _lib.load().infllm_window_forward, _ticket)
            if done is not None:
                if type(done) is int:
                    _lib.check(done, "infllm_window_forward")
                return done
    _check_rows(xq, xk, xv)
    native = dim_head in (64, HEAD_DIM)                        # other widths travel in rows of 128
    dim = dim_head if native else HEAD_DIM
    split = _heads if native else _wide_heads
    q, q_ptr, q_sb, q_sh, q_sl = split(xq, batch, len_q, num_heads, dim_head)
    k, k_ptr, k_sb, k_sh, k_sl = split(xk, batch, n_new, num_heads_kv, dim_head)
    v, v_ptr, v_sb, v_sh, v_sl = split(xv, batch, n_new, num_heads_kv, dim_head)
    inv_freq = position_bias.inv_freq
    if inv_freq.device != dev or inv_freq.dtype != torch.float32 or inv_freq.numel() != dim // 2 or not inv_freq.is_contiguous():
        inv_freq = inv_freq.to(device=dev, dtype=torch.float32).contiguous() if native else wide_inv_freq(inv_freq, dev)
        if inv_freq.numel() != dim // 2:
            raise ValueError(f"the rotary embedding is built for head_dim {2 * position_bias.inv_freq.numel()}, the heads have {dim_head}")

    old_k = old_v = raw_old = None
    seen = rows_old = raw_rows = 0
    stream = _stream()
    if past is not None:
        old_k, old_v, seen, raw_old = past
        rows_old = _check_cached(old_k, old_v, raw_old, batch, num_heads_kv, dim_head, dev)
        if native:
            cached_k, cached_v = old_k, old_v
        else:
            cached_k, cached_v = widen(old_k, dim_head), widen(old_v, dim_head)
            raw_old = None if raw_old is None else widen(raw_old, dim_head)
        if raw_old is not None:
            if not raw_old.is_contiguous() or raw_old.data_ptr() & 15:
                raw_old = raw_old.clone(memory_format=torch.contiguous_format)
            raw_rows = raw_old.size(2)
    rows_all, len_k = rows_old + n_new, seen + n_new
    bf = torch.bfloat16
    cut = kind and len_k > n_local + n_init and rows_all > n_local + n_init
    raw, raw_new = raw_old, raw_rows
    if kind == 2 and raw_rows < n_init and seen == raw_rows:   # un-rotated copies of the first n_init keys
        raw_new = min(n_init, len_k)
        raw = torch.empty((batch, num_heads_kv, raw_new, dim), dtype=bf, device=dev)
    all_kv = None
    if cut:
        rows_new = n_init + n_local
        cache = torch.empty((2, batch, num_heads_kv, rows_new, dim), dtype=bf, device=dev)
        new_k, new_v = cache.unbind(0)
        if len_q > 1 or n_new > 1:
            all_kv = torch.empty((2, batch, num_heads_kv, rows_all, dim), dtype=bf, device=dev)
    else:
        rows_new = rows_all
        behind = _lib.host().claim(old_k, old_v, n_new, stream) if past is not None and native else None
        if behind is not None:
            new_k, new_v = behind
        else:
            cap = rows_all + max(256, rows_all // 4)
            if kind:
                cap = max(rows_all, min(cap, n_local + n_init))
            both = torch.empty((2, batch, num_heads_kv, cap, dim), dtype=bf, device=dev)
            _lib.host().make_room(both, rows_all, stream)
            new_k, new_v = both.narrow(3, 0, rows_all).unbind(0)

    step_bytes = _step_bytes(kind, batch, num_heads, dim)
    words, fresh = _take_words(old_k, batch * num_heads, step_bytes, dev, stream)
    work_bytes = step_bytes
    if len_q > 1:
        rows_q = batch * num_heads * len_q
        part_rows = 64 * rows_q if rows_q <= 2048 else _SPLIT_ROWS if 2 * rows_q <= _SPLIT_ROWS else 0
        work_bytes = (2 if kind else 1) * rows_q * dim * 2 + part_rows * (2 * dim + 4)
    # (a step's scratch comes with its words: one allocation of the three that its output, its cache and it take; words of a call that
    # needed less come with less)
    if len_q == 1 and words is not None and words[5] >= work_bytes:
        work_ptr = words[4]
    else:
        work = torch.empty((work_bytes,), dtype=torch.uint8, device=dev)
        work_ptr = work.data_ptr()
    out = torch.empty((batch, len_q, num_heads * dim), dtype=bf, device=dev)
    okp = ovp = 0
    ok_sb = ok_sh = ov_sb = ov_sh = 0
    if rows_old:
        cached_k, okp, ok_sb, ok_sh = _cache_rows(cached_k, dim)
        cached_v, ovp, ov_sb, ov_sh = _cache_rows(cached_v, dim)
    n_sb, n_sh, _, _ = new_k.stride()                          # (and new_v's: halves of one buffer)
    args = _ARGS.pack(q_ptr, k_ptr, v_ptr, q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, v_sb, v_sh, v_sl, batch, num_heads, num_heads_kv, dim,
                      len_q, n_new, kind, n_init, n_local, seen, inv_freq.data_ptr(), float(position_bias.distance_scale), okp, ovp, ok_sb, ok_sh, ov_sb,
                      ov_sh, new_k.data_ptr(), new_v.data_ptr(), n_sb, n_sh, n_sb, n_sh, rows_old, rows_new,
                      all_kv[0].data_ptr() if all_kv is not None else 0, all_kv[1].data_ptr() if all_kv is not None else 0,
                      raw_old.data_ptr() if raw_old is not None else 0, raw.data_ptr() if raw is not None else 0, raw_rows, raw_new, work_ptr,
                      work_bytes, out.data_ptr(), len_q * num_heads * dim, dim, num_heads * dim, _ticket(words),
                      1.0 / math.sqrt(dim_head), fresh)
    _lib.check(_lib.load().infllm_window_forward(args, stream), "infllm_window_forward")
    if not native:
        out = narrow(out.view(batch, len_q, num_heads, dim), dim_head).reshape(batch, len_q, num_heads * dim_head)
        new_k, new_v = narrow(new_k, dim_head), narrow(new_v, dim_head)
        raw = None if raw is None else narrow(raw, dim_head)
    if words is not None:
        new_k.untyped_storage()._infllm_words = words
    return out, (new_k, new_v, len_k, raw)


def sink_window_forward(kind, n_local, n_init, fattn=False):
    assert kind in ("stream-llm", "infinite-lm")
    code = _KINDS[kind]

    def forward(self, query, key_value, position_bias, use_cache, past_key_value, project_q, project_k, project_v,
                attention_out, dim_head, num_heads, num_heads_kv):
        out, cache = _call(code, n_local, n_init, query, key_value, position_bias, past_key_value, project_q, project_k, project_v, dim_head, num_heads,
                           num_heads_kv)
        out = attention_out(out)
        return (out, cache) if use_cache else out

    return forward


def causal_forward(fattn=False):
    def forward(self, query, key_value, position_bias, use_cache, past_key_value, project_q, project_k, project_v,
                attention_out, dim_head, num_heads, num_heads_kv):
        assert use_cache                                                           # origin.py:18
        past = None if past_key_value is None else (past_key_value[0], past_key_value[1], past_key_value[0].size(2), None)
        out, cache = _call(0, 0, 0, query, key_value, position_bias, past, project_q, project_k, project_v, dim_head, num_heads, num_heads_kv)
        return attention_out(out), cache[:2]

    return forward
