"""Python view of the reference's operator surface for the attention path, on torch device tensors.

torch is used for device memory and streams only; every computation is a call into libvsp_attn.so.  The operators'
host work (tensor descriptors, output allocation, workspaces) is native: one call each into _host.so
(csrc/py_host.cpp), which calls the library; what is not called per step goes through ctypes (_ffi.py).
Names and argument meaning follow the reference (paths relative to its tree):
  flash_attention(q,k,v,scale,is_causal,dropout_p,training)  include/vesper/ops/flash_attention.h:34-41
  scaled_dot_product_attention(q,k,v,is_causal,dropout_p)     include/vesper/nn/functional.h:132-136
  KVCache / GQAKVCache .update/.reset/.current_seq_len         include/vesper/nn/transformer.h:21-39,
                                                               include/vesper/nn/gqa_attention.h:110-163
  attention_core(q,k,v,cache,start_pos)                        steps 4-6 of GroupedQueryAttention::forward,
                                                               src/nn/gqa_attention.cpp:128-148
"""
import ctypes as C
import math

import torch

from . import _ffi
from . import _host
from ._ffi import VspError, VspKVCache, VspTensor, check, lib

_DT = {torch.float32: _ffi.F32, torch.bfloat16: _ffi.BF16, torch.float16: _ffi.F16, torch.int8: _ffi.I8,
       torch.int32: _ffi.I32}


def _desc(t):
    d = VspTensor()
    d.data = t.data_ptr() if t.numel() > 0 else (t.data_ptr() or 0)
    if t.dtype not in _DT:
        raise VspError(_ffi.ERR_UNSUPPORTED)
    d.dtype = _DT[t.dtype]
    d.ndim = min(t.dim(), 4)
    for i in range(min(t.dim(), 4)):
        d.shape[i] = t.shape[i]
        d.stride[i] = t.stride(i)
    if t.dim() > 4:
        d.ndim = t.dim()  # rejected by the library with the reference's message
    return d


def _stream(t):
    return C.c_void_p(torch.cuda.current_stream(t.device).cuda_stream)


def repeat_kv_is_fused():
    """ops::repeat_kv (src/ops/attention_ops.cpp:92-155) has no kernel here: query head h reads kv head
    h // n_rep inside the attention kernels."""
    return True


def flash_attention(q, k, v, scale, is_causal=True, dropout_p=0.0, training=False, return_lse=False):
    """ops::flash_attention; k, v may have fewer heads than q (GQA)."""
    return _host.flash(q, k, v, scale, is_causal, dropout_p, training, return_lse)


def flash_attention_split(q, k, v, scale, is_causal=True, return_lse=False, workspace=None):
    """ops::flash_attention for fp32 tensors through the bf16 matrix cores (vsp_attn_prefill_split): every operand as two
    bf16 terms, three MFMAs per product, fp32 accumulation; within the reference's 1e-4 of its fp32 result."""
    return _host.flash_split(q, k, v, scale, is_causal, return_lse, workspace)


def backward_workspace(q, fast=False):
    """Workspace of flash_attention_backward for tensors of q's shape; fast: the larger one that lets the bf16 path
    compute dS once (vsp_attn_backward_fast_workspace_bytes)."""
    f = lib.vsp_attn_backward_fast_workspace_bytes if fast else lib.vsp_attn_backward_workspace_bytes
    return torch.empty(max(f(q.shape[0], q.shape[1], q.shape[2]), 16), dtype=torch.uint8, device=q.device)


def flash_attention_backward(grad_output, q, k, v, output, lse, scale, is_causal=True, workspace=None):
    """ops::flash_attention_backward: (dq, dk, dv); k, v may have fewer heads than q (their gradients then sum over
    the query heads of each group).  workspace: from backward_workspace(); its size selects the bf16 path."""
    return _host.backward(grad_output, q, k, v, output, lse, scale, is_causal, workspace, False)


def flash_attention_backward_split(grad_output, q, k, v, output, lse, scale, is_causal=True, workspace=None):
    """ops::flash_attention_backward for fp32 tensors through the bf16 matrix cores (vsp_attn_prefill_backward_split):
    every operand as two bf16 terms, three MFMAs per product, fp32 accumulation and fp32 gradients."""
    return _host.backward(grad_output, q, k, v, output, lse, scale, is_causal, workspace, True)


class RopeTable:
    """{cos, sin} of the angles of functional::compute_rope_frequencies (src/nn/functional.cpp:424-443) for
    absolute positions [0, length): computed once on the host by the library, kept on the device."""

    def __init__(self, length, head_dim, theta=10000.0, device="cuda"):
        host = torch.empty((length, head_dim // 2, 2), dtype=torch.float32)
        lib.vsp_rope_fill_table(C.c_void_p(host.data_ptr()), 0, int(length), int(head_dim), float(theta))
        self.length, self.head_dim, self.theta = int(length), int(head_dim), float(theta)
        self.host = host
        self.table = host.to(device)


class KVCache:
    """nn::KVCache with selectable storage: fmt 'f32' (the reference's layout), 'bf16' or 'q8_0'."""

    _FMT = {"f32": _ffi.KV_F32, "bf16": _ffi.KV_BF16, "q8_0": _ffi.KV_Q8_0}

    def __init__(self, batch_size, num_heads, max_seq_len, head_dim, device="cuda", fmt="f32", paging=None):
        """paging=(page_tokens, n_pages): the planes hold n_pages pages of page_tokens tokens and `page_table`
        (device int32 [batch, max_seq_len / page_tokens], set by the caller) says which page holds which tokens."""
        self.fmt = fmt
        self.device = torch.device(device)
        c = VspKVCache()
        c.format = self._FMT[fmt]
        c.B, c.Hkv, c.S_max, c.D = batch_size, num_heads, max_seq_len, head_dim
        self.page_table = None
        if paging is not None:
            page_tokens, n_pages = paging
            c.page_tokens, c.n_pages = int(page_tokens), int(n_pages)
            c.pages_per_seq = max_seq_len // max(int(page_tokens), 1)
            self.page_table = torch.zeros((batch_size, max(c.pages_per_seq, 1)), dtype=torch.int32, device=self.device)
            c.page_table = self.page_table.data_ptr()
        self._planes = []
        for plane in range(4):
            if paging is not None:
                n = lib.vsp_kv_plane_bytes(c.format, c.n_pages, c.Hkv, c.page_tokens, c.D, plane)
            else:
                n = lib.vsp_kv_plane_bytes(c.format, c.B, c.Hkv, c.S_max, c.D, plane)
            self._planes.append(torch.empty(n, dtype=torch.uint8, device=self.device) if n else None)
        c.k, c.v, c.k_scale, c.v_scale = [p.data_ptr() if p is not None else None for p in self._planes]
        c.len = 0
        self._c = c
        self._addr = C.addressof(c)  # for the native host side; c lives as long as the cache
        check(lib.vsp_kv_cache_reset(C.byref(c), _stream(self._planes[0])))  # vesper::zeros, transformer.cpp:40-41

    # -- reference interface
    def current_seq_len(self):
        return int(self._c.len)

    def get_max_seq_len(self):
        return int(self._c.S_max)

    max_seq_len = get_max_seq_len

    def reset(self):
        check(lib.vsp_kv_cache_reset(C.byref(self._c), _stream(self._planes[0])))

    def update(self, new_k, new_v, start_pos, return_views=True, start_pos_dev=None):
        _host.update(self._addr, new_k, new_v, start_pos, start_pos_dev)
        if not return_views:
            return None
        return self.views()

    def rope_update(self, q, new_k, new_v, start_pos, rope, out_dtype=None, start_pos_dev=None, return_views=False,
                    out=None):
        """Steps 3-4 of the attention modules' cached forward in one launch (src/nn/gqa_attention.cpp:124-130):
        q and k rotated by `rope` (a RopeTable) at positions start_pos.., k and v written to the cache.
        Returns the rotated q (and the cache views when asked)."""
        q_out = _host.rope_update(self._addr, q, new_k, new_v, start_pos, rope.table, rope.length, out, out_dtype, start_pos_dev)
        return (q_out, self.views()) if return_views else q_out

    def prefill(self, q, seq_lens=None, is_causal=True, scale=None, return_lse=False, chunk_lens=None, split=True, max_len=0):
        """Attention of the last T tokens (q [B,Hq,T,D]) over the cached context, read in place from the planes:
        chunked prefill.  seq_lens: device int32[B] per-row context lengths (default: the cache's one length).
        split=False withholds the workspace that lets the library split a long context over workgroups.
        max_len: host-side bound of the device-side lengths (0: the cache's capacity), which the split is planned on."""
        sc = scale if scale is not None else 1.0 / math.sqrt(q.shape[-1])
        return _host.prefill(self._addr, q, seq_lens, max_len, chunk_lens, sc, is_causal, return_lse, split)

    # -- reads
    def views(self, dtype=None):
        """[:, :, 0:len, :] of K and V.  fp32 storage: true views (no copy), like the reference;
        other formats: materialised in `dtype` (default fp32)."""
        c = self._c
        if c.format == _ffi.KV_F32:
            shape = (c.B, c.Hkv, c.S_max, c.D)
            k = self._planes[0].view(torch.float32).view(shape)[:, :, :c.len, :]
            v = self._planes[1].view(torch.float32).view(shape)[:, :, :c.len, :]
            return k, v
        return self.read(0, c.len, dtype or torch.float32)

    def read(self, start, count, dtype=torch.float32):
        c = self._c
        k = torch.empty((c.B, c.Hkv, count, c.D), dtype=dtype, device=self.device)
        v = torch.empty_like(k)
        dk, dv = _desc(k), _desc(v)
        check(lib.vsp_kv_read(C.byref(c), int(start), int(count), C.byref(dk), C.byref(dv), _stream(k)))
        return k, v

    def read_q8_0(self, plane, start, count):
        c = self._c
        qs = torch.empty((c.B, c.Hkv, count, c.D), dtype=torch.int8, device=self.device)
        sc = torch.empty((c.B, c.Hkv, count, c.D // 32), dtype=torch.int16, device=self.device)
        check(lib.vsp_kv_read_q8_0(C.byref(c), plane, int(start), int(count), qs.data_ptr(), sc.data_ptr(), _stream(qs)))
        return qs, sc

    def raw_plane(self, plane):
        return self._planes[plane]

    def set_len(self, n):
        """Bench/test helper: declare `n` tokens valid without appending (planes filled directly)."""
        self._c.len = int(n)


class GQAKVCache(KVCache):
    """nn::GQAKVCache: same semantics, int64 bookkeeping in the reference."""


class RaggedKVCache(KVCache):
    """A cache whose rows have their own lengths, kept in a device int32[B] array (the reference's caches have
    one host-side length for the batch).  Every step is asynchronous: nothing is read back to the host.
    `upper` is a host-side upper bound of the longest row, used only to size work (grids, workspaces)."""

    def __init__(self, batch_size, num_heads, max_seq_len, head_dim, device="cuda", fmt="bf16", paging=None):
        super().__init__(batch_size, num_heads, max_seq_len, head_dim, device=device, fmt=fmt, paging=paging)
        self.seq_lens = torch.zeros(batch_size, dtype=torch.int32, device=self.device)
        self.upper = 0

    def reset_rows(self, rows):
        """Forget the given rows (a finished request leaves the batch); their tokens become stale, not zero."""
        self.seq_lens[torch.as_tensor(rows, device=self.device, dtype=torch.long)] = 0

    def _advance(self, n_new, T, ref):
        _host.advance(self.seq_lens, n_new, T, self._c.B, self._c.S_max)
        self.upper = min(self.upper + int(T), self._c.S_max)

    def append(self, new_k, new_v, n_new=None, q=None, rope=None, q_dtype=None):
        """Row b's first n_new[b] (default: all T) tokens go to positions seq_lens[b]..; with `rope`, q and k are
        rotated at those positions in the same launch and the rotated q is returned."""
        T = new_k.shape[2]
        if rope is not None:
            out = self.rope_update(q, new_k, new_v, 0, rope, out_dtype=q_dtype, start_pos_dev=self.seq_lens)
        else:
            self.update(new_k, new_v, 0, return_views=False, start_pos_dev=self.seq_lens)
            out = None
        self._advance(n_new, T, new_k)
        return out

    def decode(self, q, scale=None, out=None):
        return decode_attention(q, self, seq_lens=self.seq_lens, max_len=max(self.upper, 1), scale=scale, out=out)

    def prefill_chunk(self, q, n_new=None, scale=None):
        """Attention of the chunk just appended (q [B,Hq,T,D], row b valid for n_new[b] rows) over each row's context.
        A full chunk of a few tokens (T * query heads per kv head <= 16) goes through the decode kernels."""
        T, D = q.shape[2], q.shape[3]
        if n_new is None and T > 1 and T * (q.shape[1] // self._c.Hkv) <= 16 and D in (64, 128):
            return decode_attention_multi(q, self, seq_lens=self.seq_lens, max_len=max(self.upper, 1), scale=scale)
        return self.prefill(q, seq_lens=self.seq_lens, chunk_lens=n_new, scale=scale, max_len=max(self.upper, 1))


# What streams keep between calls, filled by the native host side; calls on different streams share none of it.
# ("cuda", device, stream) -> (grow-only split-K workspace, counters of the one-launch decode step).  A captured graph
# holds their addresses: growth during stream capture is refused (size the workspace with one eager call, or pass
# `workspace=`, before capturing; room that only makes a call faster is then done without), and a block that a capture was
# given is kept under ("held", device, address) when a later call needs a larger one.  clear() gives the memory back: not while a captured graph may be replayed.
_WS = {}
_host.bind(VspError, _WS)


def decode_attention(q, cache, seq_lens=None, max_len=0, scale=None, out=None, workspace=None):
    """One new token per sequence attending to the cache: q [B,Hq,1,D] -> [B,Hq,1,D].
    workspace: a caller-owned uint8 device tensor for the split-K partials (default: a cached one per stream)."""
    if scale is None:
        scale = 1.0 / math.sqrt(q.shape[-1])  # src/nn/functional.cpp:403
    return _host.decode(cache._addr, q, seq_lens, max_len, scale, out, workspace, 0)


def decode_attention_multi(q, cache, seq_lens=None, max_len=0, scale=None, out=None, workspace=None):
    """The last T tokens of each sequence (already appended) attending to the cache at the decode kernels' rate:
    q [B,Hq,T,D] -> [B,Hq,T,D], token t sees keys [0, L_b - T + t]; T * Hq/Hkv <= 16 (vsp_attn_decode_multi)."""
    if scale is None:
        scale = 1.0 / math.sqrt(q.shape[-1])
    return _host.decode(cache._addr, q, seq_lens, max_len, scale, out, workspace, 1)


def decode_attention_proj(q, cache, wo, bias=None, seq_lens=None, max_len=0, scale=None, out=None, workspace=None):
    """decode_attention followed by the module's output projection (src/nn/gqa_attention.cpp:151-152, Linear::forward
    src/nn/linear.cpp:41-49) in one call: q [B,Hq,1,D], wo [N, Hq*D], bias [N] or None -> y [B,1,N]."""
    if scale is None:
        scale = 1.0 / math.sqrt(q.shape[-1])
    return _host.decode_proj(cache._addr, q, wo, bias, seq_lens, max_len, scale, out, workspace)


def decode_attention_noalloc(q, cache, out, seq_lens=None, max_len=0, scale=None):
    """decode_attention through vsp_attn_decode_noalloc: the partials go to the library's fixed per-GPU array
    and the call allocates nothing (`out` is the caller's).  Calls overlapping on one GPU race."""
    if scale is None:
        scale = 1.0 / math.sqrt(q.shape[-1])
    return _host.decode(cache._addr, q, seq_lens, max_len, scale, out, None, 2)


def scaled_dot_product_attention(q, k, v, is_causal=False, dropout_p=0.0):
    """functional::scaled_dot_product_attention (src/nn/functional.cpp:370-422) on explicit tensors.
    The reference switches algorithm at T >= 512 for speed; here one kernel serves every T.
    Like the reference, a causal mask needs T == L (its [T,T] mask does not broadcast otherwise)
    unless T == 1."""
    if dropout_p > 0.0:
        raise VspError(_ffi.ERR_UNSUPPORTED)
    T, L = q.shape[2], k.shape[2]
    if is_causal and T != L and T != 1:
        raise VspError(_ffi.ERR_BROADCAST)
    scale = 1.0 / math.sqrt(q.shape[-1])
    return flash_attention(q, k, v, scale, is_causal=bool(is_causal) and T > 1)


def attention_core(q, new_k, new_v, cache=None, start_pos=0, rope=None, q_dtype=None):
    """Steps 4-6 of GroupedQueryAttention::forward(x, cache, start_pos), src/nn/gqa_attention.cpp:128-148
    (== MultiHeadAttention::forward, src/nn/transformer.cpp:190-205, with n_rep = 1):
    cache.update(k, v, start_pos); repeat_kv (fused); SDPA with use_causal = (T > 1).
    With `rope` (a RopeTable) step 3 (:124-127) is included: q and k are rotated at start_pos in the same
    launch that writes the cache; q continues in `q_dtype` (default: its own)."""
    T = q.shape[2]
    if cache is None:
        return scaled_dot_product_attention(q, new_k, new_v, is_causal=(T > 1))
    if T == 1 and q_dtype in (None, q.dtype):
        table, length = (rope.table, rope.length) if rope is not None else (None, 0)
        out = _host.token_step(cache._addr, q, new_k, new_v, start_pos, table, length, 1.0 / math.sqrt(q.shape[-1]))
        if out is not None:
            return out
    if T > 1 and rope is not None and q_dtype in (None, q.dtype):
        out = _host.prompt_step(cache._addr, q, new_k, new_v, start_pos, rope.table, rope.length, 1.0 / math.sqrt(q.shape[-1]))
        if out is not None:
            return out
    if rope is not None:
        q = cache.rope_update(q, new_k, new_v, start_pos, rope, out_dtype=q_dtype)
    else:
        cache.update(new_k, new_v, start_pos, return_views=False)
    if T == 1:
        return decode_attention(q, cache)
    if cache.current_seq_len() != T:
        raise VspError(_ffi.ERR_BROADCAST)  # the reference's [T,T] mask cannot be added to [T,L] scores
    if cache.fmt == "f32":
        k, v = cache.views()  # true views of the fp32 planes, as in the reference
        return flash_attention(q, k, v, 1.0 / math.sqrt(q.shape[-1]), is_causal=True)
    if q.dtype == torch.bfloat16:
        return cache.prefill(q, is_causal=True)  # bf16 / Q8_0 planes are read in place, nothing is materialised
    k, v = cache.views(dtype=q.dtype)  # fp32 queries over a narrower cache: the context is widened once
    return flash_attention(q, k, v, 1.0 / math.sqrt(q.shape[-1]), is_causal=True)
