"""torch-facing ops over the C ABI, registered under the reference's op names.

* ``torch.ops.turboquant_write.quantize_write_kv_cache`` — schema of
  csrc/src/quantize_write_binding.cu:285-286 (reference).
* ``torch.ops.turboquant_v5.decode_v5_from_cache_paged_splitkv_ws`` — schema of
  csrc/src/decode_v5_tc_binding.cu:966-973 (reference).
* ``torch.ops.turboquant_v5.decode_paged_balanced_ws`` — the same decode with
  the split plan made on the GPU from seq_lens (ragged batches); the
  backend's default.
* ``torch.ops.turboquant_v5.decode_v5_from_cache_ws`` and
  ``decode_v5_from_cache_splitkv_ws`` — schemas of decode_v5_tc_binding.cu:948-964,
  the non-split (graph-safe) and gather-then-split ops the reference backend
  and tests call; ``decode_v5_from_cache`` is the eager (allocating) form.

Both launch on the current torch stream, allocate nothing and never sync, so
they can be captured in a HIP graph.  They have a CUDA (= HIP on ROCm) kernel
only: CPU tensors raise.
"""
from __future__ import annotations

import ctypes

import torch

from . import _lib
from .geometry import entry_bytes

_DTYPES = {torch.float32: _lib.TQ_F32, torch.float16: _lib.TQ_F16, torch.bfloat16: _lib.TQ_BF16}


_nat = None


def _native():
    """The C++ forms of the calls below (_tq_torch.so, built beside the
    library by ``python -m turboquant_amd.build``); loading it also binds the
    registered ops.  Each takes the ordinary call and returns its result (True
    where the call has none); False or None means that it did nothing, and the
    checks here decide."""
    global _nat
    if _nat is None:
        _lib.load()
        try:
            from . import _tq_torch
        except ImportError as e:
            raise RuntimeError(f"turboquant_amd._tq_torch cannot be loaded ({e}). "
                               "Run `python -m turboquant_amd.build`.") from e
        abi = getattr(_tq_torch, "abi_version", None)
        if abi != _lib.ABI_VERSION:  # built against another header
            raise RuntimeError(f"turboquant_amd._tq_torch ABI {abi} != expected "
                               f"{_lib.ABI_VERSION}; rebuild it")
        _nat = _tq_torch
    return _nat


def _stream_ptr(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


def _require_gpu(*tensors: torch.Tensor) -> None:
    """Every tensor on a GPU, and all on the same one (the kernels launch on
    the first tensor's device and read the others' addresses there)."""
    dev = None
    for t in tensors:
        if not t.is_cuda:
            raise RuntimeError("TurboQuant ops run on the GPU only; got a CPU tensor")
        if dev is None:
            dev = t.device
        elif t.device != dev:
            raise RuntimeError(f"TurboQuant ops need all tensors on one GPU: {dev} and {t.device}")


def quantize_write_kv_cache(kv_cache: torch.Tensor, key: torch.Tensor, value: torch.Tensor,
                            signs: torch.Tensor, slot_mapping: torch.Tensor, head_dim: int,
                            padded_dim: int) -> None:
    """Quantize K/V [num_tokens, H, head_dim] and scatter into kv_cache in place.

    kv_cache: uint8-addressable [2, num_blocks, block_size, H, ebs].  Mirrors
    quantize_write_kv_cache (quantize_write_binding.cu:207-269) including its
    checks; key/value may be fp32 (as the reference requires), fp16 or bf16.
    """
    if (_nat or _native()).write_cache(kv_cache, key, value, signs, slot_mapping, head_dim,
                                       padded_dim):
        return
    if kv_cache.dim() != 5 or kv_cache.size(0) != 2:
        raise RuntimeError("kv_cache leading dim must be 2 (K,V)")
    if slot_mapping.dtype != torch.int32:
        raise RuntimeError("slot_mapping must be int32")
    if key.dtype not in _DTYPES or value.dtype != key.dtype:
        raise RuntimeError(f"key/value must share a float dtype, got {key.dtype}/{value.dtype}")
    if key.dim() != 3 or value.shape != key.shape:
        raise RuntimeError("key/value must be [num_tokens, num_heads, head_dim]")
    if key.size(2) < head_dim:
        # the kernel reads head_dim elements of every row
        raise RuntimeError(f"key/value rows hold {key.size(2)} elements, fewer than "
                           f"head_dim {head_dim}")
    _require_gpu(kv_cache, key, value, signs, slot_mapping)
    if key.stride(-1) != 1 or value.stride(-1) != 1:
        raise RuntimeError("key/value last dim must be contiguous")
    ebs = kv_cache.size(-1) * kv_cache.element_size()
    if ebs % 16 != 0:
        raise RuntimeError(f"kv_cache.size(-1) must be 16-byte aligned, got {ebs}")
    if not kv_cache.is_contiguous():
        raise RuntimeError("kv_cache must be contiguous")
    if signs.dtype != torch.float32 or signs.numel() < padded_dim:
        raise RuntimeError("signs must be fp32 [padded_dim]")
    num_tokens = min(key.size(0), slot_mapping.numel())
    if num_tokens == 0:
        return
    _, nb, bs, h, _ = kv_cache.shape
    if key.size(1) != h:
        raise RuntimeError(f"key has {key.size(1)} heads, cache has {h}")
    # the kernel reads both by address
    signs, slot_mapping = signs.contiguous(), slot_mapping.contiguous()
    lib = _lib.load()
    base = kv_cache.data_ptr()
    slab = nb * bs * h * ebs
    with torch.cuda.device(kv_cache.device):
        rc = lib.tq_quantize_write_kv_cache(
            base, base + slab, key.data_ptr(), value.data_ptr(), _DTYPES[key.dtype],
            key.stride(0), key.stride(1), value.stride(0), value.stride(1),
            signs.data_ptr(), slot_mapping.data_ptr(), num_tokens, h, int(head_dim),
            int(padded_dim), bs, ebs, nb, _stream_ptr(kv_cache.device))
    _lib.check(rc, "quantize_write_kv_cache")


def decode_paged_splitkv(q: torch.Tensor, kv_cache: torch.Tensor, indices: torch.Tensor,
                         indptr: torch.Tensor, seq_lens: torch.Tensor, num_kv_heads: int,
                         head_dim: int, padded_dim: int, sm_scale: float,
                         signs: torch.Tensor | None, o: torch.Tensor, partition_o: torch.Tensor,
                         partition_lse: torch.Tensor, num_splits: int,
                         kv_chunk_size: int) -> torch.Tensor:
    """Split-KV decode: q fp16 [B, Hq, pd] -> o fp16 [B, Hq, pd] (returned)."""
    _require_gpu(q, kv_cache, indices, indptr, seq_lens, o, partition_o, partition_lse)
    if q.dtype != torch.float16 or q.dim() != 3 or q.size(2) != padded_dim or q.stride(2) != 1:
        raise RuntimeError("q must be fp16 [B, Hq, padded_dim] with a contiguous last dim")
    b, hq, pd = q.shape
    for t, name in ((indices, "indices"), (indptr, "indptr"), (seq_lens, "seq_lens")):
        if t.dtype != torch.int32 or not t.is_contiguous():
            raise RuntimeError(f"{name} must be a contiguous int32 tensor")
    if seq_lens.numel() < b or indptr.numel() < b:
        raise RuntimeError("seq_lens / indptr shorter than the batch")
    if tuple(o.shape) != (b, hq, pd) or o.dtype != torch.float16 or not o.is_contiguous():
        raise RuntimeError("o_ws shape mismatch")
    if (partition_o.dtype != torch.float32 or partition_o.numel() < b * num_splits * hq * pd
            or not partition_o.is_contiguous()):
        raise RuntimeError("partition_o_ws shape/dtype mismatch")
    if (partition_lse.dtype != torch.float32 or partition_lse.numel() < b * num_splits * hq
            or not partition_lse.is_contiguous()):
        raise RuntimeError("partition_lse_ws shape/dtype mismatch")
    if kv_cache.dim() != 5 or kv_cache.size(0) != 2 or not kv_cache.is_contiguous():
        raise RuntimeError("kv_cache must be contiguous [2, num_blocks, block_size, H, ebs]")
    _, nb, bs, hk, _ = kv_cache.shape
    if hk != num_kv_heads:
        raise RuntimeError(f"kv_cache has {hk} kv heads, num_kv_heads={num_kv_heads}")
    ebs = kv_cache.size(-1) * kv_cache.element_size()
    sp = 0
    if signs is not None and signs.numel() > 0:
        if signs.dtype != torch.float32 or signs.numel() < pd:
            raise RuntimeError("hadamard_signs must be fp32 [padded_dim]")
        _require_gpu(q, signs)
        signs = signs.contiguous()
        sp = signs.data_ptr()
    lib = _lib.load()
    base = kv_cache.data_ptr()
    slab = nb * bs * hk * ebs
    with torch.cuda.device(q.device):
        rc = lib.tq_decode_paged_splitkv(
            q.data_ptr(), q.stride(0), q.stride(1), base, base + slab, indices.data_ptr(),
            indptr.data_ptr(), seq_lens.data_ptr(), b, hq, int(num_kv_heads), int(head_dim),
            int(padded_dim), bs, ebs, nb, float(sm_scale), sp, int(num_splits),
            int(kv_chunk_size), partition_o.data_ptr(), partition_lse.data_ptr(), o.data_ptr(),
            _stream_ptr(q.device))
    _lib.check(rc, "decode_paged_splitkv")
    return o


def balanced_rows(batch: int, num_qo_heads: int, num_kv_heads: int, padded_dim: int,
                  device: torch.device | None = None) -> int:
    """Partial rows a balanced decode of this geometry may use on `device`
    (the resident workgroup slots of the partials kernel, at least one per
    sequence): size partition_o [rows, Hq, pd] and partition_lse [rows, Hq]."""
    lib = _lib.load()
    with torch.cuda.device(device if device is not None else torch.cuda.current_device()):
        rows = lib.tq_decode_balanced_rows(int(batch), int(num_qo_heads), int(num_kv_heads),
                                           int(padded_dim))
    if rows < 0:
        _lib.check(rows, "decode_balanced_rows")
    return rows


def decode_paged_balanced(q: torch.Tensor, kv_cache: torch.Tensor, indices: torch.Tensor,
                          indptr: torch.Tensor, seq_lens: torch.Tensor, num_kv_heads: int,
                          head_dim: int, padded_dim: int, sm_scale: float,
                          signs: torch.Tensor | None, o: torch.Tensor,
                          partition_o: torch.Tensor, partition_lse: torch.Tensor,
                          split_indptr: torch.Tensor) -> torch.Tensor:
    """Split-KV decode with the split plan made on the GPU from seq_lens:
    every work unit covers about the same number of tokens whatever the
    length mix of the batch (the reference sizes splits from max_len,
    vllm_backend_fused.py:128-156).  split_indptr int32 [B + 2] receives the
    partial-row table (sequence b owns rows split_indptr[b] ..
    split_indptr[b + 1]) and, last, the unit size in tokens.  No host read,
    so it can be captured in a HIP graph whose seq_lens change per replay."""
    if (_nat or _native()).decode_balanced(q, kv_cache, indices, indptr, seq_lens, num_kv_heads,
                                           head_dim, padded_dim, sm_scale, signs, o, partition_o,
                                           partition_lse, split_indptr, False):
        return o
    _require_gpu(q, o)
    if q.dtype != torch.float16:
        raise RuntimeError("q must be fp16 [B, Hq, padded_dim] with a contiguous last dim")
    if o.dtype != torch.float16:
        raise RuntimeError("o_ws shape mismatch")
    return _decode_balanced(q, kv_cache, indices, indptr, seq_lens, num_kv_heads, head_dim,
                            padded_dim, sm_scale, signs, o, partition_o, partition_lse,
                            split_indptr, int(padded_dim))


def decode_paged_balanced_rows(q: torch.Tensor, kv_cache: torch.Tensor, indices: torch.Tensor,
                               indptr: torch.Tensor, seq_lens: torch.Tensor, num_kv_heads: int,
                               head_dim: int, padded_dim: int, sm_scale: float,
                               signs: torch.Tensor | None, o: torch.Tensor,
                               partition_o: torch.Tensor, partition_lse: torch.Tensor,
                               split_indptr: torch.Tensor) -> torch.Tensor:
    """decode_paged_balanced over the model's own rows: q and o [B, Hq,
    head_dim] (head_dim a multiple of 8), each fp16 or bf16, dims up to
    padded_dim counting as zero (tq_decode_paged_balanced_rows)."""
    if (_nat or _native()).decode_balanced(q, kv_cache, indices, indptr, seq_lens, num_kv_heads,
                                           head_dim, padded_dim, sm_scale, signs, o, partition_o,
                                           partition_lse, split_indptr, True):
        return o
    if q.dtype not in (torch.float16, torch.bfloat16) or \
            o.dtype not in (torch.float16, torch.bfloat16):
        raise RuntimeError("q and o must be fp16 or bf16 [B, Hq, head_dim]")
    return _decode_balanced(q, kv_cache, indices, indptr, seq_lens, num_kv_heads, head_dim,
                            padded_dim, sm_scale, signs, o, partition_o, partition_lse,
                            split_indptr, int(head_dim))


def _decode_balanced(q, kv_cache, indices, indptr, seq_lens, num_kv_heads, head_dim, padded_dim,
                     sm_scale, signs, o, partition_o, partition_lse, split_indptr, row_dim):
    _require_gpu(q, kv_cache, indices, indptr, seq_lens, o, partition_o, partition_lse,
                 split_indptr)
    if q.dim() != 3 or q.size(2) != row_dim or q.stride(2) != 1:
        raise RuntimeError("q must be fp16 [B, Hq, padded_dim] with a contiguous last dim"
                           if row_dim == padded_dim else
                           "q must be [B, Hq, head_dim] with a contiguous last dim")
    b, hq, _ = q.shape
    pd = int(padded_dim)
    rows_op = row_dim != pd or q.dtype != torch.float16 or o.dtype != torch.float16
    for t, name in ((indices, "indices"), (indptr, "indptr"), (seq_lens, "seq_lens"),
                    (split_indptr, "split_indptr")):
        if t.dtype != torch.int32 or not t.is_contiguous():
            raise RuntimeError(f"{name} must be a contiguous int32 tensor")
    if seq_lens.numel() < b or indptr.numel() < b:
        raise RuntimeError("seq_lens / indptr shorter than the batch")
    if split_indptr.numel() < b + 2:
        raise RuntimeError("split_indptr must hold batch + 2 entries")
    if tuple(o.shape) != (b, hq, row_dim) or not o.is_contiguous():
        raise RuntimeError("o_ws shape mismatch")
    if (partition_o.dtype != torch.float32 or partition_o.dim() != 3
            or tuple(partition_o.shape[1:]) != (hq, pd) or not partition_o.is_contiguous()):
        raise RuntimeError("partition_o_ws must be fp32 [rows, Hq, padded_dim]")
    rows = partition_o.size(0)
    if (partition_lse.dtype != torch.float32 or partition_lse.numel() < rows * hq
            or not partition_lse.is_contiguous()):
        raise RuntimeError("partition_lse_ws must be fp32 [rows, Hq]")
    if kv_cache.dim() != 5 or kv_cache.size(0) != 2 or not kv_cache.is_contiguous():
        raise RuntimeError("kv_cache must be contiguous [2, num_blocks, block_size, H, ebs]")
    _, nb, bs, hk, _ = kv_cache.shape
    if hk != num_kv_heads:
        raise RuntimeError(f"kv_cache has {hk} kv heads, num_kv_heads={num_kv_heads}")
    ebs = kv_cache.size(-1) * kv_cache.element_size()
    sp = 0
    if signs is not None and signs.numel() > 0:
        if signs.dtype != torch.float32 or signs.numel() < pd:
            raise RuntimeError("hadamard_signs must be fp32 [padded_dim]")
        _require_gpu(q, signs)
        signs = signs.contiguous()
        sp = signs.data_ptr()
    lib = _lib.load()
    base = kv_cache.data_ptr()
    slab = nb * bs * hk * ebs
    with torch.cuda.device(q.device):
        args = (base, base + slab, indices.data_ptr(), indptr.data_ptr(), seq_lens.data_ptr(), b,
                hq, int(num_kv_heads), int(head_dim), pd, bs, ebs, nb, float(sm_scale), sp, rows,
                partition_o.data_ptr(), partition_lse.data_ptr(), split_indptr.data_ptr(),
                o.data_ptr())
        st = _stream_ptr(q.device)
        if rows_op:
            rc = lib.tq_decode_paged_balanced_rows(q.data_ptr(), q.stride(0), q.stride(1),
                                                   _DTYPES[q.dtype], *args, _DTYPES[o.dtype], st)
        else:
            rc = lib.tq_decode_paged_balanced(q.data_ptr(), q.stride(0), q.stride(1), *args, st)
    _lib.check(rc, "decode_paged_balanced")
    return o


def prefill_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, o: torch.Tensor,
                      sm_scale: float) -> torch.Tensor:
    """Causal GQA attention of q [Lq, Hq, D] over k, v [Lk, Hkv, D] (fp16,
    D = 64, 128 or 256, Lq <= Lk), the queries aligned to the end of the keys
    (query i sees keys <= Lk - Lq + i), written into o [Lq, Hq, D] fp16.
    Heads and dims of every tensor contiguous; token strides free (multiples
    of 8)."""
    _require_gpu(q, k, v, o)
    for t, name in ((q, "q"), (k, "k"), (v, "v"), (o, "o")):
        if t.dtype != torch.float16 or t.dim() != 3 or t.stride(2) != 1:
            raise RuntimeError(f"{name} must be fp16 [tokens, heads, head_dim] with contiguous dims")
    lq, hq, d = q.shape
    lk, hkv, dk = k.shape
    if tuple(v.shape) != (lk, hkv, dk) or dk != d or tuple(o.shape) != (lq, hq, d):
        raise RuntimeError("prefill_attention: q/k/v/o shapes disagree")
    lib = _lib.load()
    with torch.cuda.device(q.device):
        # a short chunk over a long context splits its keys over workgroups;
        # the split's workspace comes from torch's allocator (graph-safe)
        nbytes = int(lib.tq_prefill_workspace_bytes(int(lq), int(lk), int(hq), int(hkv), int(d)))
        ws = torch.empty(nbytes, dtype=torch.uint8, device=q.device) if nbytes > 0 else None
        rc = lib.tq_prefill_attention_ws(q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(),
                                         k.stride(0), k.stride(1), v.data_ptr(), v.stride(0),
                                         v.stride(1), o.data_ptr(), o.stride(0), o.stride(1),
                                         int(lq), int(lk), int(hq), int(hkv), int(d),
                                         float(sm_scale),
                                         ws.data_ptr() if ws is not None else None, nbytes,
                                         _stream_ptr(q.device))
    _lib.check(rc, "prefill_attention")
    return o


def prefill_attention_batch(q: torch.Tensor, o: torch.Tensor, requests, num_kv_heads: int,
                            head_dim: int, padded_dim: int, sm_scale: float,
                            k: torch.Tensor | None = None, v: torch.Tensor | None = None,
                            k2: torch.Tensor | None = None,
                            v2: torch.Tensor | None = None) -> torch.Tensor:
    """prefill_attention for several requests in one launch: `requests` are
    (q_start, q_len, kv_start, kv_len, source) host integers, the request's
    rows of q / o and of k / v (source 0) or k2 / v2 (source 1).  q and o fp16
    or bf16 [tokens, Hq, head_dim]; K / V fp16 [tokens, Hkv, padded_dim], zero
    past head_dim; head_dim a multiple of 8."""
    if (_nat or _native()).prefill_batch(q, o, requests, num_kv_heads, head_dim, padded_dim,
                                         sm_scale, k, v, k2, v2):
        return o
    kvs = [t for t in (k, v, k2, v2) if t is not None]
    _require_gpu(q, o, *kvs)
    hq = q.size(1)
    if q.dim() != 3 or tuple(o.shape) != tuple(q.shape) or q.size(2) != head_dim:
        raise RuntimeError("prefill_attention_batch: q / o must be [tokens, heads, head_dim]")
    if q.dtype not in (torch.float16, torch.bfloat16) or \
            o.dtype not in (torch.float16, torch.bfloat16) or q.stride(2) != 1 or o.stride(2) != 1:
        raise RuntimeError("prefill_attention_batch: q / o must be fp16 or bf16 with contiguous "
                           "dims")
    for t in kvs:
        if t.dtype != torch.float16 or t.dim() != 3 or t.stride(2) != 1 or \
                tuple(t.shape[1:]) != (num_kv_heads, padded_dim):
            raise RuntimeError("prefill_attention_batch: k / v must be fp16 [tokens, Hkv, "
                               "padded_dim] with contiguous dims")
    for a, b in ((k, v), (k2, v2)):
        if (a is None) != (b is None) or (a is not None and a.size(0) != b.size(0)):
            raise RuntimeError("prefill_attention_batch: k and v must go together")
    if k2 is not None and k2.stride() != v2.stride():
        raise RuntimeError("prefill_attention_batch: k2 and v2 must share their strides")
    for qs, ql, ks, kl, src in requests:
        kv = k2 if src else k
        if qs < 0 or ql < 0 or qs + ql > q.size(0) or kv is None or ks < 0 or kl < ql \
                or ks + kl > kv.size(0):
            raise RuntimeError("prefill_attention_batch: a request is out of range")
    n = len(requests)
    cols = [(ctypes.c_int32 * max(1, n))(*c) for c in
            (zip(*requests) if n else ((),) * 5)]
    lib = _lib.load()
    st = lambda t: (0, 0) if t is None else (t.stride(0), t.stride(1))
    ptr = lambda t: None if t is None else t.data_ptr()
    with torch.cuda.device(q.device):
        nbytes = int(lib.tq_prefill_batch_workspace_bytes(cols[1], cols[3], n, hq,
                                                          int(padded_dim)))
        ws = torch.empty(nbytes, dtype=torch.uint8, device=q.device) if nbytes > 0 else None
        rc = lib.tq_prefill_attention_batch(
            q.data_ptr(), *st(q), _DTYPES[q.dtype], ptr(k), *st(k), ptr(v), *st(v), ptr(k2),
            ptr(v2), *st(k2), o.data_ptr(), *st(o), _DTYPES[o.dtype], *cols, n, hq,
            int(num_kv_heads), int(head_dim), int(padded_dim), float(sm_scale), ptr(ws), nbytes,
            _stream_ptr(q.device))
    _lib.check(rc, "prefill_attention_batch")
    return o


def dequant_paged(kv_cache: torch.Tensor, pages: torch.Tensor, num_tokens: int,
                  num_kv_heads: int, head_dim: int, padded_dim: int,
                  signs: torch.Tensor | None, out_k: torch.Tensor, out_v: torch.Tensor) -> None:
    """Cached K/V of tokens [0, num_tokens) of one sequence (its page-table
    row `pages`) as fp16 rows [num_tokens, H_kv, head_dim] in the original
    domain, written into out_k / out_v (rows may be strided, heads and dims
    contiguous)."""
    _require_gpu(kv_cache, pages, out_k, out_v)
    if kv_cache.dim() != 5 or kv_cache.size(0) != 2 or not kv_cache.is_contiguous():
        raise RuntimeError("kv_cache must be contiguous [2, num_blocks, block_size, H, ebs]")
    _, nb, bs, hk, _ = kv_cache.shape
    if hk != num_kv_heads:
        raise RuntimeError(f"kv_cache has {hk} kv heads, num_kv_heads={num_kv_heads}")
    if pages.dtype != torch.int32 or not pages.is_contiguous():
        raise RuntimeError("pages must be a contiguous int32 tensor")
    if num_tokens > pages.numel() * bs:
        raise RuntimeError("pages do not cover num_tokens")
    for t in (out_k, out_v):
        if (t.dtype != torch.float16 or t.dim() != 3 or t.size(0) < num_tokens
                or t.size(1) != num_kv_heads or t.size(2) != head_dim or t.stride(2) != 1
                or t.stride(1) != head_dim or t.stride(0) != out_k.stride(0)):
            raise RuntimeError("out_k / out_v must be fp16 [>= num_tokens, H_kv, head_dim] "
                               "with contiguous heads and one row stride")
    if num_tokens == 0:
        return
    ebs = kv_cache.size(-1) * kv_cache.element_size()
    sp = 0
    if signs is not None and signs.numel() > 0:
        if signs.dtype != torch.float32 or signs.numel() < padded_dim:
            raise RuntimeError("signs must be fp32 [padded_dim]")
        _require_gpu(kv_cache, signs)
        signs = signs.contiguous()
        sp = signs.data_ptr()
    lib = _lib.load()
    base = kv_cache.data_ptr()
    slab = nb * bs * hk * ebs
    with torch.cuda.device(kv_cache.device):
        rc = lib.tq_dequant_paged(base, base + slab, pages.data_ptr(), int(num_tokens),
                                  int(num_kv_heads), int(head_dim), int(padded_dim), bs, ebs, nb,
                                  sp, out_k.data_ptr(), out_v.data_ptr(), out_k.stride(0),
                                  _stream_ptr(kv_cache.device))
    _lib.check(rc, "dequant_paged")


def prefill_gather(kv_cache: torch.Tensor | None, block_table: torch.Tensor | None,
                   key: torch.Tensor, value: torch.Tensor, requests, head_dim: int,
                   padded_dim: int, signs: torch.Tensor | None, out_k: torch.Tensor,
                   out_v: torch.Tensor) -> None:
    """The keys and values of several prefill requests as fp16 rows
    [*, H_kv, padded_dim] in one launch (tq_prefill_gather): `requests` are
    (table_row, ctx, fresh_start, fresh_len, out_start) host integers; the ctx
    cached tokens of page-table row table_row are read back as dequant_paged
    does, the fresh rows of key / value (fp16, bf16 or fp32) converted, both
    zero-padded past head_dim.  kv_cache and block_table may be None when
    every ctx is 0."""
    if (_nat or _native()).prefill_gather(kv_cache, block_table, key, value, requests, head_dim,
                                          padded_dim, signs, out_k, out_v):
        return
    _require_gpu(key, value, out_k, out_v)
    if key.dtype not in _DTYPES or value.dtype != key.dtype:
        raise RuntimeError(f"key/value must share a float dtype, got {key.dtype}/{value.dtype}")
    if key.dim() != 3 or value.shape != key.shape or key.size(2) != head_dim \
            or key.stride(2) != 1 or value.stride(2) != 1:
        raise RuntimeError("prefill_gather: key/value must be [tokens, heads, head_dim] with "
                           "contiguous dims")
    h = key.size(1)
    for t in (out_k, out_v):
        if t.dtype != torch.float16 or t.dim() != 3 or tuple(t.shape[1:]) != (h, padded_dim) \
                or not t.is_contiguous():
            raise RuntimeError("prefill_gather: out_k / out_v must be contiguous fp16 "
                               "[rows, H_kv, padded_dim]")
    rows = min(out_k.size(0), out_v.size(0))
    bs, nb, ebs, base, slab, bt, bt_rows = 16, 0, entry_bytes(head_dim)[2], 0, 0, 0, 0
    if kv_cache is not None and block_table is not None:
        _require_gpu(key, kv_cache, block_table)
        if kv_cache.dim() != 5 or kv_cache.size(0) != 2 or not kv_cache.is_contiguous():
            raise RuntimeError("kv_cache must be contiguous [2, num_blocks, block_size, H, ebs]")
        _, nb, bs, hk, _ = kv_cache.shape
        if hk != h:
            raise RuntimeError(f"kv_cache has {hk} kv heads, num_kv_heads={h}")
        if block_table.dtype != torch.int32 or block_table.dim() != 2 \
                or block_table.stride(1) != 1:
            raise RuntimeError("block_table must be int32 [requests, pages] with contiguous rows")
        ebs = kv_cache.size(-1) * kv_cache.element_size()
        base, slab, bt, bt_rows = kv_cache.data_ptr(), nb * bs * h * ebs, block_table.data_ptr(), \
            block_table.size(0)
    for row, ctx, fs, fl, dst in requests:
        if ctx < 0 or fs < 0 or fl < 0 or dst < 0 or dst + ctx + fl > rows \
                or fs + fl > key.size(0):
            raise RuntimeError("prefill_gather: a request is out of range")
        if ctx > 0 and (not bt or not 0 <= row < bt_rows):
            raise RuntimeError("prefill_gather: cached context needs the cache and a table row")
        if ctx > 0 and ctx > block_table.size(1) * bs:
            raise RuntimeError("pages do not cover num_tokens")
    sp = 0
    if signs is not None and signs.numel() > 0:
        if signs.dtype != torch.float32 or signs.numel() < padded_dim:
            raise RuntimeError("signs must be fp32 [padded_dim]")
        _require_gpu(key, signs)
        signs = signs.contiguous()
        sp = signs.data_ptr()
    n = len(requests)
    if n == 0:
        return
    cols = [(ctypes.c_int32 * n)(*c) for c in zip(*requests)]
    lib = _lib.load()
    with torch.cuda.device(key.device):
        rc = lib.tq_prefill_gather(
            base, base + slab, bt, block_table.stride(0) if bt else 0, h, int(head_dim),
            int(padded_dim), bs, ebs, nb, sp, key.data_ptr(), value.data_ptr(),
            _DTYPES[key.dtype], key.stride(0), key.stride(1), value.stride(0), value.stride(1),
            *cols, n, out_k.data_ptr(), out_v.data_ptr(), _stream_ptr(key.device))
    _lib.check(rc, "prefill_gather")


def _floats(values) -> list | tuple:
    """A host table as the sequence that the native calls take."""
    return values if isinstance(values, (list, tuple)) else list(values)


def _host_f32(values) -> "ctypes.Array":
    vals = [float(v) for v in values]
    return (ctypes.c_float * max(1, len(vals)))(*vals)


def _aligned16(t: torch.Tensor) -> torch.Tensor:
    """t contiguous at a 16-byte aligned address (the kernels read it in
    16-byte pieces); a copy when it is not."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def qjl_halves(s: torch.Tensor, padded_dim: int):
    """(S hi, S lo, S^T hi, S^T lo): fp16 halves of the QJL matrix s fp32
    [dim, dim], zero-padded to [padded_dim, padded_dim] (tq_qjl_halves)."""
    r = (_nat or _native()).qjl_halves(s, padded_dim)
    if r is not None:
        return r
    _require_gpu(s)
    if s.dtype != torch.float32 or s.dim() != 2 or s.size(0) != s.size(1):
        raise RuntimeError("qjl_halves: S must be a square fp32 matrix")
    s = s.contiguous()
    out = torch.empty((4, padded_dim, padded_dim), dtype=torch.float16, device=s.device)
    lib = _lib.load()
    with torch.cuda.device(s.device):
        rc = lib.tq_qjl_halves(s.data_ptr(), s.size(0), int(padded_dim), out.data_ptr(),
                               _stream_ptr(s.device))
    _lib.check(rc, "qjl_halves")
    return out.unbind(0)


def qjl_operand(s: torch.Tensor, padded_dim: int, transposed: bool):
    """(hi, lo, scale) of the QJL matrix s fp32 [dim, dim], or of its transpose,
    for prod_quantize_qjl_ws / prod_dequantize_qjl_ws: fp16 halves [padded_dim,
    padded_dim] of the rows, each over its power of two scale[row]
    (tq_qjl_operand)."""
    r = (_nat or _native()).qjl_operand(s, padded_dim, transposed)
    if r is not None:
        return r
    _require_gpu(s)
    if s.dtype != torch.float32 or s.dim() != 2 or s.size(0) != s.size(1):
        raise RuntimeError("qjl_operand: S must be a square fp32 matrix")
    s = s.contiguous()
    out = torch.empty((2, padded_dim, padded_dim), dtype=torch.float16, device=s.device)
    scale = torch.empty((padded_dim,), dtype=torch.float32, device=s.device)
    lib = _lib.load()
    with torch.cuda.device(s.device):
        rc = lib.tq_qjl_operand(s.data_ptr(), s.size(0), int(padded_dim), int(transposed),
                                out.data_ptr(), scale.data_ptr(), _stream_ptr(s.device))
    _lib.check(rc, "qjl_operand")
    return out[0], out[1], scale


def mse_quantize(x: torch.Tensor, padded_dim: int, bit_width: int, signs: torch.Tensor,
                 boundaries) -> tuple[torch.Tensor, torch.Tensor]:
    """TurboQuantMSE.quantize on the GPU (tq_mse_quantize): x fp32
    [..., dim] -> (packed uint8 [..., padded_dim / per], norms fp32 [...]).
    `boundaries` are the codebook's 2^b - 1 scaled boundaries as host
    floats."""
    boundaries = _floats(boundaries)
    r = (_nat or _native()).mse_quantize(x, padded_dim, bit_width, signs, boundaries)
    if r is not None:
        return r
    _require_gpu(x, signs)
    if x.dtype != torch.float32:
        raise RuntimeError("mse_quantize: x must be fp32")
    if signs.dtype != torch.float32 or signs.numel() < padded_dim:
        raise RuntimeError("mse_quantize: signs must be fp32 [padded_dim]")
    x = x.contiguous()
    if x.data_ptr() % 16:
        x = x.clone()  # the kernel reads whole rows as float4
    dim = x.shape[-1]
    lead = x.shape[:-1]
    n = x.numel() // dim if dim else 0
    per = 2 if bit_width == 3 else 8 // bit_width
    packed = torch.empty((*lead, padded_dim // per), dtype=torch.uint8, device=x.device)
    norms = torch.empty(lead, dtype=torch.float32, device=x.device)
    signs = _aligned16(signs)
    lib = _lib.load()
    with torch.cuda.device(x.device):
        rc = lib.tq_mse_quantize(x.data_ptr(), n, dim, int(padded_dim), int(bit_width),
                                 signs.data_ptr(), _host_f32(boundaries), packed.data_ptr(),
                                 norms.data_ptr(), _stream_ptr(x.device))
    _lib.check(rc, "mse_quantize")
    return packed, norms


def mse_dequantize(packed: torch.Tensor, norms: torch.Tensor, dim: int, padded_dim: int,
                   bit_width: int, signs: torch.Tensor, centroids) -> torch.Tensor:
    """TurboQuantMSE.dequantize on the GPU (tq_mse_dequantize): packed uint8
    [..., padded_dim / per] and norms [...] -> fp32 [..., dim].  `centroids`
    are the codebook's 2^b scaled levels as host floats."""
    centroids = _floats(centroids)
    r = (_nat or _native()).mse_dequantize(packed, norms, dim, padded_dim, bit_width, signs,
                                           centroids)
    if r is not None:
        return r
    _require_gpu(packed, norms, signs)
    per = 2 if bit_width == 3 else 8 // bit_width
    if packed.dtype != torch.uint8 or packed.shape[-1] != padded_dim // per:
        raise RuntimeError("mse_dequantize: packed must be uint8 [..., padded_dim / per]")
    if tuple(norms.shape) != tuple(packed.shape[:-1]):
        raise RuntimeError("mse_dequantize: norms must match packed's leading dims")
    packed = packed.contiguous()
    if packed.data_ptr() % 16:
        packed = packed.clone()  # the kernel reads a lane's codes as dwords
    nf = norms.to(torch.float32).contiguous()
    lead = packed.shape[:-1]
    n = nf.numel()
    out = torch.empty((*lead, dim), dtype=torch.float32, device=packed.device)
    signs = _aligned16(signs)
    lib = _lib.load()
    with torch.cuda.device(packed.device):
        rc = lib.tq_mse_dequantize(packed.data_ptr(), nf.data_ptr(), n, int(dim),
                                   int(padded_dim), int(bit_width), signs.data_ptr(),
                                   _host_f32(centroids), out.data_ptr(),
                                   _stream_ptr(packed.device))
    _lib.check(rc, "mse_dequantize")
    return out


def prod_quantize(x: torch.Tensor, padded_dim: int, mse_bit_width: int, signs: torch.Tensor,
                  boundaries, centroids):
    """TurboQuantProd's MSE stage and residual on the GPU (tq_prod_quantize):
    x fp32 [..., dim] -> (packed, norms, residual_unit fp32 [..., dim],
    residual_norms fp32 [...]); packed and norms are mse_quantize's."""
    _require_gpu(x, signs)
    if x.dtype != torch.float32:
        raise RuntimeError("prod_quantize: x must be fp32")
    if signs.dtype != torch.float32 or signs.numel() < padded_dim:
        raise RuntimeError("prod_quantize: signs must be fp32 [padded_dim]")
    x = x.contiguous()
    if x.data_ptr() % 16:
        x = x.clone()
    dim = x.shape[-1]
    lead = x.shape[:-1]
    n = x.numel() // dim if dim else 0
    per = 2 if mse_bit_width == 3 else 8 // mse_bit_width
    packed = torch.empty((*lead, padded_dim // per), dtype=torch.uint8, device=x.device)
    norms = torch.empty(lead, dtype=torch.float32, device=x.device)
    resid = torch.empty((*lead, dim), dtype=torch.float32, device=x.device)
    rnorm = torch.empty(lead, dtype=torch.float32, device=x.device)
    signs = _aligned16(signs)
    lib = _lib.load()
    with torch.cuda.device(x.device):
        rc = lib.tq_prod_quantize(x.data_ptr(), n, dim, int(padded_dim), int(mse_bit_width),
                                  signs.data_ptr(), _host_f32(boundaries), _host_f32(centroids),
                                  packed.data_ptr(), norms.data_ptr(), resid.data_ptr(),
                                  rnorm.data_ptr(), _stream_ptr(x.device))
    _lib.check(rc, "prod_quantize")
    return packed, norms, resid, rnorm


def prod_dequantize(packed: torch.Tensor, norms: torch.Tensor, qjl_term: torch.Tensor,
                    residual_norms: torch.Tensor, dim: int, padded_dim: int, mse_bit_width: int,
                    signs: torch.Tensor, centroids) -> torch.Tensor:
    """TurboQuantProd.dequantize on the GPU (tq_prod_dequantize): the MSE
    read-back plus qjl_term * (sqrt(pi/2) / dim * residual_norms), qjl_term
    being z S (fp32 [..., dim])."""
    _require_gpu(packed, norms, qjl_term, residual_norms, signs)
    per = 2 if mse_bit_width == 3 else 8 // mse_bit_width
    if packed.dtype != torch.uint8 or packed.shape[-1] != padded_dim // per:
        raise RuntimeError("prod_dequantize: packed must be uint8 [..., padded_dim / per]")
    lead = tuple(packed.shape[:-1])
    if tuple(norms.shape) != lead or tuple(residual_norms.shape) != lead:
        raise RuntimeError("prod_dequantize: norms must match packed's leading dims")
    if tuple(qjl_term.shape) != (*lead, dim):
        raise RuntimeError("prod_dequantize: qjl_term must be [..., dim]")
    packed = packed.contiguous()
    if packed.data_ptr() % 16:
        packed = packed.clone()
    nf = norms.to(torch.float32).contiguous()
    rn = residual_norms.to(torch.float32).contiguous()
    qt = qjl_term.to(torch.float32).contiguous()
    out = torch.empty((*lead, dim), dtype=torch.float32, device=packed.device)
    signs = _aligned16(signs)
    lib = _lib.load()
    with torch.cuda.device(packed.device):
        rc = lib.tq_prod_dequantize(packed.data_ptr(), nf.data_ptr(), qt.data_ptr(),
                                    rn.data_ptr(), nf.numel(), int(dim), int(padded_dim),
                                    int(mse_bit_width), signs.data_ptr(), _host_f32(centroids),
                                    out.data_ptr(), _stream_ptr(packed.device))
    _lib.check(rc, "prod_dequantize")
    return out


def prod_quantize_qjl(x: torch.Tensor, padded_dim: int, mse_bit_width: int,
                      signs: torch.Tensor, boundaries, centroids, s_hi: torch.Tensor,
                      s_lo: torch.Tensor):
    """TurboQuantProd.quantize with the QJL product fused (tq_prod_quantize_qjl,
    padded_dim 64 or 128): x fp32 [..., dim] -> (packed, norms, qjl_signs int8
    [..., dim], residual_norms).  s_hi / s_lo: fp16 [padded_dim, padded_dim]
    halves of the QJL matrix."""
    return _prod_quantize_qjl(x, padded_dim, mse_bit_width, signs, boundaries, centroids, s_hi,
                              s_lo, False)


def prod_quantize_qjl_matrix(x: torch.Tensor, padded_dim: int, mse_bit_width: int,
                             signs: torch.Tensor, boundaries, centroids, s: torch.Tensor):
    """prod_quantize_qjl from the QJL matrix itself, fp32 [dim, dim]
    (tq_prod_quantize_qjl_matrix): nothing made from it to keep or go stale."""
    return _prod_quantize_qjl(x, padded_dim, mse_bit_width, signs, boundaries, centroids, s, None,
                              False)


def prod_quantize_qjl_ws(x: torch.Tensor, padded_dim: int, mse_bit_width: int,
                         signs: torch.Tensor, boundaries, centroids, s_hi: torch.Tensor,
                         s_lo: torch.Tensor):
    """prod_quantize_qjl at padded_dim 256, 512 or 1024: the row kernel and
    the QJL product on the matrix cores (tq_prod_quantize_qjl_ws), the unit
    residual between them in a workspace from torch's allocator."""
    return _prod_quantize_qjl(x, padded_dim, mse_bit_width, signs, boundaries, centroids, s_hi,
                              s_lo, True)


def _qjl_operands(hi, lo, dim, padded_dim, what):
    """The QJL operand as the library takes it: two halves, or (lo None) the
    matrix itself."""
    if lo is None:
        if hi.dtype != torch.float32 or tuple(hi.shape) != (dim, dim):
            raise RuntimeError(f"{what} must be fp32 [dim, dim]")
        return (_aligned16(hi),)
    _require_gpu(hi, lo)
    for t in (hi, lo):
        if t.dtype != torch.float16 or tuple(t.shape) != (padded_dim, padded_dim) \
                or not t.is_contiguous() or t.data_ptr() % 16:
            raise RuntimeError(f"{what} halves must be contiguous aligned fp16 "
                               "[padded_dim, padded_dim]")
    return hi, lo


def _prod_quantize_qjl(x, padded_dim, mse_bit_width, signs, boundaries, centroids, s_hi, s_lo,
                       large: bool):
    boundaries, centroids = _floats(boundaries), _floats(centroids)
    r = (_nat or _native()).prod_quantize_qjl(x, padded_dim, mse_bit_width, signs, boundaries,
                                              centroids, s_hi, s_lo, large)
    if r is not None:
        return r
    _require_gpu(x, signs, s_hi)
    if x.dtype != torch.float32:
        raise RuntimeError("prod_quantize_qjl: x must be fp32")
    operand = _qjl_operands(s_hi, s_lo, x.shape[-1], padded_dim, "prod_quantize_qjl: S")
    x = x.contiguous()
    if x.data_ptr() % 16:
        x = x.clone()
    dim = x.shape[-1]
    lead = x.shape[:-1]
    n = x.numel() // dim if dim else 0
    per = 2 if mse_bit_width == 3 else 8 // mse_bit_width
    packed = torch.empty((*lead, padded_dim // per), dtype=torch.uint8, device=x.device)
    norms = torch.empty(lead, dtype=torch.float32, device=x.device)
    z = torch.empty((*lead, dim), dtype=torch.int8, device=x.device)
    rnorm = torch.empty(lead, dtype=torch.float32, device=x.device)
    signs = _aligned16(signs)
    lib = _lib.load()
    args = (x.data_ptr(), n, dim, int(padded_dim), int(mse_bit_width), signs.data_ptr(),
            _host_f32(boundaries), _host_f32(centroids), *(t.data_ptr() for t in operand),
            packed.data_ptr(), norms.data_ptr(), z.data_ptr(), rnorm.data_ptr())
    with torch.cuda.device(x.device):
        if large:
            ws = torch.empty(int(lib.tq_prod_workspace_bytes(n, int(padded_dim))),
                             dtype=torch.uint8, device=x.device)
            rc = lib.tq_prod_quantize_qjl_ws(*args, ws.data_ptr(), ws.numel(),
                                             _stream_ptr(x.device))
        else:
            fn = lib.tq_prod_quantize_qjl_matrix if s_lo is None else lib.tq_prod_quantize_qjl
            rc = fn(*args, _stream_ptr(x.device))
    _lib.check(rc, "prod_quantize_qjl")
    return packed, norms, z, rnorm


def prod_dequantize_qjl(packed: torch.Tensor, norms: torch.Tensor, qjl_signs: torch.Tensor,
                        residual_norms: torch.Tensor, dim: int, padded_dim: int,
                        mse_bit_width: int, signs: torch.Tensor, centroids,
                        st_hi: torch.Tensor, st_lo: torch.Tensor) -> torch.Tensor:
    """TurboQuantProd.dequantize with z S formed in-kernel
    (tq_prod_dequantize_qjl, padded_dim 64 or 128).  st_hi / st_lo: fp16
    halves of S^T."""
    return _prod_dequantize_qjl(packed, norms, qjl_signs, residual_norms, dim, padded_dim,
                                mse_bit_width, signs, centroids, st_hi, st_lo, False)


def prod_dequantize_qjl_matrix(packed: torch.Tensor, norms: torch.Tensor, qjl_signs: torch.Tensor,
                               residual_norms: torch.Tensor, dim: int, padded_dim: int,
                               mse_bit_width: int, signs: torch.Tensor, centroids,
                               s: torch.Tensor) -> torch.Tensor:
    """prod_dequantize_qjl from the QJL matrix itself, S (not S^T) fp32
    [dim, dim] (tq_prod_dequantize_qjl_matrix)."""
    return _prod_dequantize_qjl(packed, norms, qjl_signs, residual_norms, dim, padded_dim,
                                mse_bit_width, signs, centroids, s, None, False)


def prod_dequantize_qjl_ws(packed: torch.Tensor, norms: torch.Tensor, qjl_signs: torch.Tensor,
                           residual_norms: torch.Tensor, dim: int, padded_dim: int,
                           mse_bit_width: int, signs: torch.Tensor, centroids,
                           st_hi: torch.Tensor, st_lo: torch.Tensor,
                           st_scale: torch.Tensor | None = None) -> torch.Tensor:
    """prod_dequantize_qjl at padded_dim 256, 512 or 1024
    (tq_prod_dequantize_qjl_ws); st_scale: fp32 [padded_dim], the row scales
    of the halves (qjl_operand), none for unscaled ones (qjl_halves)."""
    return _prod_dequantize_qjl(packed, norms, qjl_signs, residual_norms, dim, padded_dim,
                                mse_bit_width, signs, centroids, st_hi, st_lo, True, st_scale)


def _prod_dequantize_qjl(packed, norms, qjl_signs, residual_norms, dim, padded_dim, mse_bit_width,
                         signs, centroids, st_hi, st_lo, large: bool, st_scale=None):
    centroids = _floats(centroids)
    r = (_nat or _native()).prod_dequantize_qjl(packed, norms, qjl_signs, residual_norms, dim,
                                                padded_dim, mse_bit_width, signs, centroids, st_hi,
                                                st_lo, large, st_scale)
    if r is not None:
        return r
    _require_gpu(packed, norms, qjl_signs, residual_norms, signs, st_hi)
    per = 2 if mse_bit_width == 3 else 8 // mse_bit_width
    if packed.dtype != torch.uint8 or packed.shape[-1] != padded_dim // per:
        raise RuntimeError("prod_dequantize_qjl: packed must be uint8 [..., padded_dim / per]")
    lead = tuple(packed.shape[:-1])
    if tuple(norms.shape) != lead or tuple(residual_norms.shape) != lead:
        raise RuntimeError("prod_dequantize_qjl: norms must match packed's leading dims")
    if qjl_signs.dtype != torch.int8 or tuple(qjl_signs.shape) != (*lead, dim):
        raise RuntimeError("prod_dequantize_qjl: qjl_signs must be int8 [..., dim]")
    operand = _qjl_operands(st_hi, st_lo, dim, padded_dim,
                                "prod_dequantize_qjl: S" + ("" if st_lo is None else "^T"))
    if st_scale is not None:
        _require_gpu(packed, st_scale)
        if st_scale.dtype != torch.float32 or st_scale.numel() < padded_dim \
                or not st_scale.is_contiguous():
            raise RuntimeError("prod_dequantize_qjl: st_scale must be fp32 [padded_dim]")
    packed = packed.contiguous()
    if packed.data_ptr() % 16:
        packed = packed.clone()
    nf = norms.to(torch.float32).contiguous()
    rn = residual_norms.to(torch.float32).contiguous()
    z = _aligned16(qjl_signs)
    out = torch.empty((*lead, dim), dtype=torch.float32, device=packed.device)
    signs = _aligned16(signs)
    lib = _lib.load()
    with torch.cuda.device(packed.device):
        args = (packed.data_ptr(), nf.data_ptr(), z.data_ptr(), rn.data_ptr(), nf.numel(),
                int(dim), int(padded_dim), int(mse_bit_width), signs.data_ptr(),
                _host_f32(centroids), *(t.data_ptr() for t in operand))
        tail = (out.data_ptr(), _stream_ptr(packed.device))
        if large:
            rc = lib.tq_prod_dequantize_qjl_ws(
                *args, None if st_scale is None else st_scale.data_ptr(), *tail)
        else:
            fn = lib.tq_prod_dequantize_qjl_matrix if st_lo is None else lib.tq_prod_dequantize_qjl
            rc = fn(*args, *tail)
    _lib.check(rc, "prod_dequantize_qjl")
    return out


# --------------------------------------------------------------------------
# torch.library registration under the reference's namespaces and schemas
# --------------------------------------------------------------------------
_registered = False
_libs = []


def _reference_paged_splitkv(q, kv_cache, indices, indptr, last_page_len, seq_lens,
                             num_kv_heads, page_size, head_dim, padded_dim, sm_scale,
                             hadamard_signs, qbytes, nbytes, o_ws, max_len, partition_o_ws,
                             partition_lse_ws, request_indices, kv_tile_indices, split_indptr,
                             kv_chunk_size_t, num_splits):
    """Argument adapter for decode_v5_from_cache_paged_splitkv_ws.

    The chunk size is recomputed on the host as ceil(max_len / num_splits),
    the value the reference backend stores in kv_chunk_size_t
    (vllm_backend_fused.py:210-213), so no device tensor is read.
    request_indices / kv_tile_indices / split_indptr are implied by
    (batch, num_splits); last_page_len and nbytes are unused, as in the
    reference op.
    """
    if int(padded_dim) != q.size(-1):
        raise RuntimeError("padded_dim does not match q")
    exp_q, _, _ = entry_bytes(int(head_dim))
    if int(qbytes) != exp_q:
        raise RuntimeError(f"qbytes {qbytes} does not match head_dim {head_dim}")
    if int(max_len) <= 0:
        raise RuntimeError("max_len must be positive")
    if int(num_splits) < 1:
        raise RuntimeError("num_splits must be >= 1")
    cs = -(-int(max_len) // int(num_splits))
    return decode_paged_splitkv(q, kv_cache, indices, indptr, seq_lens, int(num_kv_heads),
                                int(head_dim), int(padded_dim), float(sm_scale), hadamard_signs,
                                o_ws, partition_o_ws, partition_lse_ws, int(num_splits), cs)


def _check_gather_ws(q, num_kv_heads, max_len, qbytes, padded_dim, k_quant_ws, v_quant_ws,
                     k_norms_ws, v_norms_ws, o_ws):
    """The workspace checks of decode_v5_from_cache_ws
    (decode_v5_tc_binding.cu:466-478), kept so that callers sized for the
    reference are accepted or refused alike."""
    b, hq = q.size(0), q.size(1)
    dc = int(padded_dim) // 64
    if int(max_len) <= 0:
        raise RuntimeError("max_len must be positive")
    if tuple(k_quant_ws.shape) != (b, int(num_kv_heads), int(max_len), int(qbytes)):
        raise RuntimeError("k_quant_ws shape mismatch")
    if tuple(v_quant_ws.shape) != tuple(k_quant_ws.shape):
        raise RuntimeError("v_quant_ws shape mismatch")
    if tuple(k_norms_ws.shape) != (b, int(num_kv_heads), int(max_len), dc):
        raise RuntimeError("k_norms_ws shape mismatch")
    if tuple(v_norms_ws.shape) != tuple(k_norms_ws.shape):
        raise RuntimeError("v_norms_ws shape mismatch")
    if tuple(o_ws.shape) != (b, hq, int(padded_dim)):
        raise RuntimeError("o_ws shape mismatch")


def _scratch_f32(t: torch.Tensor, n: int):
    """n fp32 elements at the start of a contiguous caller-owned buffer, or None."""
    if not t.is_contiguous() or t.numel() * t.element_size() < 4 * n or t.data_ptr() % 16:
        return None
    return t.view(-1).view(torch.uint8)[:4 * n].view(torch.float32)


def _from_cache_ws(q, kv_cache, indices, indptr, last_page_len, seq_lens, num_kv_heads,
                   page_size, head_dim, padded_dim, sm_scale, hadamard_signs, qbytes, nbytes,
                   k_quant_ws, v_quant_ws, k_norms_ws, v_norms_ws, o_ws, max_len):
    """decode_v5_from_cache_ws (decode_v5_tc_binding.cu:439-551): the reference
    gathers the pages into contiguous K/V workspaces and runs one unsplit
    kernel.  Here the paged kernel reads the pages directly, so the gather
    workspaces are free; they hold the split partials instead (the op owns
    their contents during the call, as the reference's gather does), which
    keeps the split-KV layout without any allocation.  Tokens are read up to
    min(seq_lens[b], num_splits * kv_chunk_size) with num_splits *
    kv_chunk_size >= max_len."""
    from .geometry import CHUNK_ALIGN, choose_splits
    _check_gather_ws(q, num_kv_heads, max_len, qbytes, padded_dim, k_quant_ws, v_quant_ws,
                     k_norms_ws, v_norms_ws, o_ws)
    b, hq, pd = q.size(0), q.size(1), int(padded_dim)
    splits, chunk = choose_splits(b, int(max_len), int(num_kv_heads), hq, pd)
    while True:
        po = _scratch_f32(k_quant_ws, b * splits * hq * pd)
        pl = _scratch_f32(v_quant_ws, b * splits * hq)
        if (po is not None and pl is not None) or splits == 1:
            break
        splits = max(1, splits // 2)
        chunk = -(-int(max_len) // splits)
        chunk = (chunk + CHUNK_ALIGN - 1) // CHUNK_ALIGN * CHUNK_ALIGN
        splits = -(-int(max_len) // chunk)
    if po is None or pl is None:
        raise RuntimeError("decode_v5_from_cache_ws: workspaces too small for the partials")
    return decode_paged_splitkv(q, kv_cache, indices, indptr, seq_lens, int(num_kv_heads),
                                int(head_dim), pd, float(sm_scale), hadamard_signs, o_ws, po,
                                pl, splits, chunk)


def _from_cache_splitkv_ws(q, kv_cache, indices, indptr, last_page_len, seq_lens, num_kv_heads,
                           page_size, head_dim, padded_dim, sm_scale, hadamard_signs, qbytes,
                           nbytes, k_quant_ws, v_quant_ws, k_norms_ws, v_norms_ws, o_ws, max_len,
                           partition_o_ws, partition_lse_ws, request_indices, kv_tile_indices,
                           split_indptr, kv_chunk_size_t, num_splits):
    """decode_v5_from_cache_splitkv_ws (decode_v5_tc_binding.cu:586-752): the
    gather-then-split variant.  The paged kernel needs no gather, so this is
    the paged split op with the caller's partition workspaces."""
    _check_gather_ws(q, num_kv_heads, max_len, qbytes, padded_dim, k_quant_ws, v_quant_ws,
                     k_norms_ws, v_norms_ws, o_ws)
    return _reference_paged_splitkv(q, kv_cache, indices, indptr, last_page_len, seq_lens,
                                    num_kv_heads, page_size, head_dim, padded_dim, sm_scale,
                                    hadamard_signs, qbytes, nbytes, o_ws, max_len, partition_o_ws,
                                    partition_lse_ws, request_indices, kv_tile_indices,
                                    split_indptr, kv_chunk_size_t, num_splits)


def decode_v5_from_cache(q, kv_cache, indices, indptr, last_page_len, seq_lens, num_kv_heads,
                         page_size, head_dim, padded_dim, sm_scale, hadamard_signs, qbytes,
                         nbytes):
    """The eager decode_v5_from_cache (decode_v5_tc_binding.cu:324-423): it
    allocates its own output and workspaces (not graph-capturable, as in the
    reference).  max_len is seq_lens.max(), as the reference computes it
    (decode_v5_tc_binding.cu:350); the op is eager, so this host read is
    allowed.  A CSR indptr whose later rows are longer than the first is
    covered."""
    from .geometry import choose_splits
    b, hq, pd = q.size(0), q.size(1), int(padded_dim)
    max_len = int(seq_lens[:b].max()) if b else 0
    max_len = max(max_len, int(page_size))
    splits, chunk = choose_splits(b, max_len, int(num_kv_heads), hq, pd)
    o = torch.empty((b, hq, pd), dtype=torch.float16, device=q.device)
    po = torch.empty((b * splits, hq, pd), dtype=torch.float32, device=q.device)
    pl = torch.empty((b * splits, hq), dtype=torch.float32, device=q.device)
    return decode_paged_splitkv(q, kv_cache, indices, indptr, seq_lens, int(num_kv_heads),
                                int(head_dim), pd, float(sm_scale), hadamard_signs, o, po, pl,
                                splits, chunk)


def _register_fakes() -> None:
    """Meta ("fake") kernels, so that torch.compile and vLLM's graph capture
    can trace the ops without running them: the write mutates its cache
    argument and returns nothing; the reference's decode ops return a tensor
    shaped like o_ws (fp16 [B, Hq, padded_dim]); the balanced op writes
    o_ws, which its schema marks, and returns nothing."""
    from torch.library import register_fake

    @register_fake("turboquant_write::quantize_write_kv_cache", lib=_libs[0])
    def _write_fake(kv_cache, key, value, signs, slot_mapping, head_dim, padded_dim):
        return None

    def _decode_fake(q, kv_cache, *args):
        return q.new_empty((q.size(0), q.size(1), q.size(2)), dtype=torch.float16)

    for name in ("decode_v5_from_cache_paged_splitkv_ws", "decode_v5_from_cache_ws",
                 "decode_v5_from_cache_splitkv_ws"):
        register_fake(f"turboquant_v5::{name}", _decode_fake, lib=_libs[1])

    def _balanced_fake(q, kv_cache, indices, indptr, seq_lens, num_kv_heads, head_dim,
                       padded_dim, sm_scale, hadamard_signs, o_ws, partition_o_ws,
                       partition_lse_ws, split_indptr):
        return None

    for name in ("decode_paged_balanced_ws", "decode_paged_balanced_rows_ws"):
        register_fake(f"turboquant_v5::{name}", _balanced_fake, lib=_libs[1])


def register_ops() -> None:
    """Define turboquant_write::* and turboquant_v5::* with the reference
    schemas and bind the HIP implementations to the CUDA dispatch key (the
    write and the balanced decodes in C++, tq_torch.cpp; the others here)."""
    global _registered
    if _registered:
        return
    from torch.library import Library
    w = Library("turboquant_write", "DEF")
    w.define("quantize_write_kv_cache(Tensor(a!) kv_cache, Tensor key, Tensor value, "
             "Tensor signs, Tensor slot_mapping, int head_dim, int padded_dim) -> ()")
    d = Library("turboquant_v5", "DEF")
    d.define("decode_v5_from_cache_paged_splitkv_ws(Tensor q, Tensor kv_cache, "
             "Tensor indices, Tensor indptr, Tensor last_page_len, Tensor seq_lens, "
             "int num_kv_heads, int page_size, int head_dim, int padded_dim, "
             "float sm_scale, Tensor hadamard_signs, int qbytes, int nbytes, "
             "Tensor o_ws, int max_len, "
             "Tensor partition_o_ws, Tensor partition_lse_ws, "
             "Tensor request_indices, Tensor kv_tile_indices, "
             "Tensor split_indptr, Tensor kv_chunk_size_t, int num_splits) -> Tensor")
    d.impl("decode_v5_from_cache_paged_splitkv_ws", _reference_paged_splitkv, "CUDA")
    d.define("decode_v5_from_cache_ws(Tensor q, Tensor kv_cache, Tensor indices, "
             "Tensor indptr, Tensor last_page_len, Tensor seq_lens, "
             "int num_kv_heads, int page_size, int head_dim, int padded_dim, "
             "float sm_scale, Tensor hadamard_signs, int qbytes, int nbytes, "
             "Tensor k_quant_ws, Tensor v_quant_ws, Tensor k_norms_ws, "
             "Tensor v_norms_ws, Tensor o_ws, int max_len) -> Tensor")
    d.impl("decode_v5_from_cache_ws", _from_cache_ws, "CUDA")
    d.define("decode_v5_from_cache_splitkv_ws(Tensor q, Tensor kv_cache, Tensor indices, "
             "Tensor indptr, Tensor last_page_len, Tensor seq_lens, "
             "int num_kv_heads, int page_size, int head_dim, int padded_dim, "
             "float sm_scale, Tensor hadamard_signs, int qbytes, int nbytes, "
             "Tensor k_quant_ws, Tensor v_quant_ws, Tensor k_norms_ws, "
             "Tensor v_norms_ws, Tensor o_ws, int max_len, "
             "Tensor partition_o_ws, Tensor partition_lse_ws, "
             "Tensor request_indices, Tensor kv_tile_indices, "
             "Tensor split_indptr, Tensor kv_chunk_size_t, int num_splits) -> Tensor")
    d.impl("decode_v5_from_cache_splitkv_ws", _from_cache_splitkv_ws, "CUDA")
    # this build's balanced-split decode (no reference counterpart: the
    # reference plans splits on the host from max_len)
    # it writes its result into o_ws, and the partial rows, LSEs and row table
    # into the other workspaces, and says so in its schema (returning
    # nothing: functionalization refuses aliased outputs of custom ops), so
    # functionalization and torch.compile keep the call and its writes
    for name in ("decode_paged_balanced_ws", "decode_paged_balanced_rows_ws"):
        d.define(f"{name}(Tensor q, Tensor kv_cache, Tensor indices, "
                 "Tensor indptr, Tensor seq_lens, int num_kv_heads, int head_dim, "
                 "int padded_dim, float sm_scale, Tensor hadamard_signs, Tensor(a!) o_ws, "
                 "Tensor(b!) partition_o_ws, Tensor(c!) partition_lse_ws, "
                 "Tensor(d!) split_indptr) -> ()")
    _native()  # binds the write and the two balanced ops
    _libs.extend([w, d])
    _register_fakes()
    _registered = True
