"""Drop-in attention boundary of the paged KV-cache path, backed by libkvpath.so.

Mirrors kavor/layers/attention/flash_attention_kvcache.py:
  store_kvcache(key, value, k_cache, v_cache, slot_mapping)      (:37-46)
  Attention(num_heads, head_dim, scale, num_kv_heads, num_kv_slots=1)
      .forward(q, k, v, slot=0)                                   (:49-84)
and replaces the two flash-attn calls it makes with
  paged_decode(...)    for flash_attn_with_kvcache(...)           (:80-83)
  varlen_prefill(...)  for flash_attn_varlen_func(...)            (:76-79)
which keep flash-attn's argument names and meaning.  Every function here only
validates layouts and forwards raw pointers and strides to the C ABI (include/kvpath.h)
on the current stream; nothing computes on the host and there is no fallback.
"""

from __future__ import annotations

from functools import lru_cache

import torch
from torch import nn

from kavor_amd._lib import check, lib
from kavor_amd.layers.workspace import Workspaces, retired
from kavor_amd.utils.context import get_context

__all__ = [
    "store_kvcache", "paged_decode", "paged_decode_fused", "varlen_prefill", "Attention",
    "reserve_decode_workspace", "decode_workspace_bytes",
    "reserve_prefill_workspace", "prefill_workspace_bytes",
    "flash_attn_with_kvcache", "flash_attn_varlen_func",
]


def _stream(t: torch.Tensor) -> int:
    """The current stream's handle (building a torch.cuda.Stream for it takes 3.5 us)."""
    return torch._C._cuda_getCurrentRawStream(t.get_device())


def _require_cuda_bf16(name: str, t: torch.Tensor) -> None:
    if not t.is_cuda:
        raise ValueError(f"{name} must be a CUDA (HIP) tensor, got device {t.device}")
    if t.dtype != torch.bfloat16:
        raise ValueError(f"{name} must be bfloat16, got {t.dtype}")


def _require_int32(name: str, t: torch.Tensor, device: torch.device) -> None:
    if t.dtype != torch.int32:
        raise ValueError(f"{name} must be int32, got {t.dtype}")
    if t.device != device:
        raise ValueError(f"{name} must live on {device}, got {t.device}")
    if not t.is_contiguous():
        raise ValueError(f"{name} must be contiguous")


# ----------------------------------------------------------------------------- append

def store_kvcache(key: torch.Tensor, value: torch.Tensor, k_cache: torch.Tensor,
                  v_cache: torch.Tensor, slot_mapping: torch.Tensor) -> None:
    """Writes key[i] / value[i] into slot slot_mapping[i] of k_cache / v_cache.

    Same contract and layout assertions as store_kvcache in
    kavor/layers/attention/flash_attention_kvcache.py:37-46: key/value are
    [N, num_kv_heads, head_dim] with contiguous heads (row strides may differ), the
    caches are [num_blocks, block_size, num_kv_heads, head_dim] views whose block
    stride may exceed block_size*num_kv_heads*head_dim (K/V interleaved pages), and
    slot -1 is skipped.  Bit-exact copy on the device.
    """
    N, num_heads, head_dim = key.shape
    D = num_heads * head_dim
    key_str, value_str, cache_str = key.stride(), value.stride(), k_cache.stride()
    assert key_str[-1] == 1 and value_str[-1] == 1
    assert key_str[1] == head_dim and value_str[1] == head_dim
    assert slot_mapping.numel() == N
    assert value.shape == key.shape
    assert k_cache.shape == v_cache.shape and cache_str == v_cache.stride()
    assert cache_str[1] == D
    assert k_cache.dim() == 4
    num_blocks, block_size, cache_heads, cache_dim = k_cache.shape
    assert (cache_heads, cache_dim) == (num_heads, head_dim)
    _require_cuda_bf16("key", key)
    _require_cuda_bf16("value", value)
    _require_cuda_bf16("k_cache", k_cache)
    _require_cuda_bf16("v_cache", v_cache)
    _require_int32("slot_mapping", slot_mapping, key.device)
    rc = lib().kvp_append_bf16(
        key.data_ptr(), key_str[0], key_str[1],
        value.data_ptr(), value_str[0], value_str[1],
        k_cache.data_ptr(), v_cache.data_ptr(),
        cache_str[0], cache_str[1], cache_str[2], num_blocks * block_size,
        slot_mapping.data_ptr(), N, num_heads, head_dim, block_size, _stream(key))
    check("kvp_append_bf16", rc)


# ----------------------------------------------------------------------------- decode

_decode_workspaces = Workspaces("paged-decode", "reserve_decode_workspace")
_workspaces = _decode_workspaces.default
_retired_workspaces = retired


@lru_cache(maxsize=1024)  # arithmetic on the sizes
def decode_workspace_bytes(max_num_seqs: int, num_q_heads: int, head_dim: int,
                           max_blocks_per_seq: int, block_size: int) -> int:
    return int(lib().kvp_decode_workspace_bytes(max_num_seqs, num_q_heads, head_dim,
                                                 max_blocks_per_seq, block_size))


def reserve_decode_workspace(max_num_seqs: int, num_q_heads: int, head_dim: int,
                             max_blocks_per_seq: int, block_size: int,
                             device: torch.device | str | int) -> torch.Tensor:
    """Allocates (or grows) the current stream's decode workspace on a device.  Call before graph
    capture with the largest batch a captured graph will use: the capture takes the buffer over,
    and eager calls, which need no reservation, go on in another.  It holds the states of
    one-step (32-token) ranges, four times as many as kvp_decode_workspace_bytes counts for the
    same block table: the one-launch step runs a small batch faster in them."""
    return _decode_workspaces.get(
        device, decode_workspace_bytes(max_num_seqs, num_q_heads, head_dim, 4 * max_blocks_per_seq, block_size),
        decode_workspace_bytes(max_num_seqs, num_q_heads, head_dim, max_blocks_per_seq, block_size))


def _decode_workspace(index, stream, num_seqs, num_q_heads, head_dim, max_blocks, block_size) -> torch.Tensor:
    nbytes = decode_workspace_bytes(num_seqs, num_q_heads, head_dim, 4 * max_blocks, block_size)
    ws = _decode_workspaces.ready(index, stream, nbytes)
    if ws is None:
        ws = reserve_decode_workspace(num_seqs, num_q_heads, head_dim, max_blocks, block_size, index)
    return ws


# ----------------------------------------------------------------------------- prefill workspace

_prefill_pool = Workspaces("prefill", "reserve_prefill_workspace")
_prefill_workspaces = _prefill_pool.default
_split_pool = Workspaces("split prefill", "reserve_prefill_workspace")


@lru_cache(maxsize=1024)
def prefill_workspace_bytes(num_seqs: int, max_seqlen_q: int, num_q_heads: int, num_kv_heads: int) -> int:
    return int(lib().kvp_prefill_workspace_bytes(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads))


@lru_cache(maxsize=1024)
def _prefill_split_bytes(num_seqs: int, max_seqlen_q: int, num_q_heads: int, num_kv_heads: int) -> int:
    nbytes = int(lib().kvp_prefill_split_workspace_bytes(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads))
    return -(-nbytes // (1 << 20)) << 20  # one size for all launches that can be split: their work lists are small


# Query tiles x kv heads of a launch that may be split, at most, and keys from which one may be.
_SPLIT_TILES, _SPLIT_MIN_KEYS = 512, 1024


def _may_split(num_seqs: int, max_seqlen_q: int, max_keys: int, num_q_heads: int, num_kv_heads: int) -> bool:
    """Whether the kernel may cut the keys of such a batch, given room for the partial states."""
    group = num_q_heads // num_kv_heads if num_kv_heads else 0
    if max_keys < _SPLIT_MIN_KEYS or group not in (1, 2, 4, 5, 8):
        return False
    return 0 < num_seqs * -(-max_seqlen_q // (128 // group)) * num_kv_heads <= _SPLIT_TILES


def _split_pays(num_seqs: int, total_q: int, max_seqlen_q: int, max_keys: int, num_q_heads: int,
                num_kv_heads: int) -> bool:
    """Whether cutting the keys of a batch that may be split is likely to gain, from what the host
    knows of its lengths.

    The plan kernel decides by the lengths themselves, but a split launch in which it cuts nothing
    costs 3 to 5 us over an uncut one (its plan, and a merge that finds no work): 4 prompts of
    1024 tokens (16q/8kv) 45.6 -> 48.7 us, 4 of 700 on 2048 cached 84.8 -> 88.2, 2 of 750 on
    15000 (32q/8kv) 408 -> 411.  So the plan's cost model runs here on an average tile first.  A
    batch of about equal new lengths is taken to have equal cached ones, a ragged batch to have
    0.6 of the longest on average; averages and thresholds are fitted over 900 shapes.  17 of them
    are slower than uncut, by 4 us each (174 where every batch that may be split takes the split
    launch); 50 of the 689 that would gain stay uncut, above all equal turns on very unequal
    histories (4 of 509 tokens on 0 to 16384: 425 us against 301)."""
    tok = 128 // (num_q_heads // num_kv_heads)
    slots = _SPLIT_TILES / num_kv_heads
    even = total_q >= 0.95 * num_seqs * max_seqlen_q
    longest = -(-max_keys // 64)  # all in key tiles
    own = max_seqlen_q / 64
    cached = max(0.0, longest - own)
    tiles = num_seqs * -(-max_seqlen_q // tok)
    if not even:
        tiles = min(tiles, total_q / tok + 0.5 * num_seqs)
        cached, own = 0.6 * cached, 0.7 * own
    mean = cached + own / 2
    arrive = num_seqs * (cached + own) * num_kv_heads / 300
    least = (1.0 if num_seqs == 1 else 0.95 if even else 0.9) * max(longest, arrive)
    for parts in (2, 3, 4, 6, 8, 12, 16):
        chunk = -(-longest // parts)
        if chunk < 8:
            break
        units = tiles * min(parts, mean / chunk + 0.5)
        busy = chunk if units <= slots else tiles * mean / slots + chunk / 2
        whole = tiles * min(1.0, max(0.0, chunk - cached) / own)
        if max(arrive, busy) + (units - whole) * num_kv_heads / 48 + 4 < least:
            return True
    return False


def reserve_prefill_workspace(num_seqs: int, max_seqlen_q: int, num_q_heads: int, num_kv_heads: int,
                              device: torch.device | str | int) -> torch.Tensor:
    """Allocates (or grows) the current stream's prefill workspaces on a device: the work list of a
    launch, which is returned, and the partial states of a batch whose keys are split
    (kvp_prefill_split_workspace_bytes, 69 MB).  A caller that captures prefill into a graph
    reserves the largest batch first: the capture takes the buffers over.  Eager calls need no
    reservation, and hold partial states only once a batch may be split."""
    _split_pool.get(device, _prefill_split_bytes(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads))
    return _work_list(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads, device)


@lru_cache(maxsize=1024)
def _work_list_bytes(num_seqs: int, max_seqlen_q: int, num_q_heads: int, num_kv_heads: int) -> int:
    nbytes = prefill_workspace_bytes(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads)
    return 1 << max(4095, nbytes - 1).bit_length()  # so that batches of growing size allocate few buffers


def _work_list(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads, device) -> torch.Tensor:
    return _prefill_pool.get(device, _work_list_bytes(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads),
                             prefill_workspace_bytes(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads))


@lru_cache(maxsize=4096)  # the layers of a step share one answer
def _split_room(num_seqs, total_q, max_seqlen_q, max_keys, num_q_heads, num_kv_heads) -> int:
    """Bytes of the workspace that a split launch of such a batch takes; 0 for an uncut one."""
    if _may_split(num_seqs, max_seqlen_q, max_keys, num_q_heads, num_kv_heads) and \
            _split_pays(num_seqs, total_q, max_seqlen_q, max_keys, num_q_heads, num_kv_heads):
        return _prefill_split_bytes(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads)
    return 0


def _prefill_workspace(index, stream, num_seqs, total_q, max_seqlen_q, max_keys, num_q_heads,
                       num_kv_heads) -> torch.Tensor:
    room = _split_room(num_seqs, total_q, max_seqlen_q, max_keys, num_q_heads, num_kv_heads)
    if room:
        ws = _split_pool.ready(index, stream, room)
        if ws is None:
            ws = _split_pool.get(index, room, optional=True)
        if ws is not None:  # inside a capture without it the launch is not split
            return ws
    ws = _prefill_pool.ready(index, stream, _work_list_bytes(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads))
    return ws if ws is not None else _work_list(num_seqs, max_seqlen_q, num_q_heads, num_kv_heads, index)


def paged_decode(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                 cache_seqlens: torch.Tensor, block_table: torch.Tensor, softmax_scale: float,
                 causal: bool = True, out: torch.Tensor | None = None) -> torch.Tensor:
    """Paged decode attention, one query token per sequence.

    Argument meaning follows flash_attn_with_kvcache as called at
    kavor/layers/attention/flash_attention_kvcache.py:81-83: q is [B, 1, Hq, D] (or
    [B, Hq, D]), the caches are [num_blocks, block_size, Hkv, D], cache_seqlens int32 [B]
    counts the cached tokens including the one just appended, block_table int32
    [B, max_blocks] (entries past ceil(len/block_size) are never read).  Returns
    [B, 1, Hq, D] (or [B, Hq, D]) in bf16.  `causal` is accepted for signature
    compatibility; with one query token it changes nothing.
    """
    del causal
    if q.dim() == 4 and q.shape[1] == 1:
        q3, four_d = q[:, 0], True
    elif q.dim() == 3:
        q3, four_d = q, False
    else:
        raise ValueError(f"paged_decode takes one query token per sequence, got q of shape {tuple(q.shape)}")
    B, Hq, D = q3.shape
    _require_cuda_bf16("q", q3)
    _require_cuda_bf16("k_cache", k_cache)
    _require_cuda_bf16("v_cache", v_cache)
    cache_str, q_str = k_cache.stride(), q3.stride()
    if k_cache.shape != v_cache.shape or cache_str != v_cache.stride():
        raise ValueError("k_cache and v_cache must share shape and strides")
    num_blocks, block_size, Hkv, Dk = k_cache.shape
    if Dk != D or cache_str[3] != 1 or q_str[2] != 1:
        raise ValueError("head_dim mismatch or non-contiguous head_dim")
    _require_int32("cache_seqlens", cache_seqlens, q3.device)
    if block_table.dtype != torch.int32 or block_table.dim() != 2 or block_table.stride(1) != 1:
        raise ValueError("block_table must be an int32 [B, max_blocks] tensor with contiguous rows")
    if cache_seqlens.numel() < B or block_table.shape[0] < B:
        raise ValueError("cache_seqlens / block_table have fewer rows than q")
    if out is None:
        out3 = torch.empty(B, Hq, D, dtype=torch.bfloat16, device=q3.device)
        out = out3.unsqueeze(1) if four_d else out3
    else:
        out3 = out[:, 0] if out.dim() == 4 else out
        if out3.shape != (B, Hq, D) or out3.dtype != torch.bfloat16 or out3.stride(2) != 1:
            raise ValueError("out must be bf16 [B, 1, Hq, D] or [B, Hq, D] with contiguous head_dim")
    max_blocks = block_table.shape[1]
    stream = _stream(q3)
    ws = _decode_workspace(q3.get_device(), stream, B, Hq, D, max_blocks, block_size)
    rc = lib().kvp_paged_decode_bf16(
        q3.data_ptr(), q_str[0], q_str[1],
        k_cache.data_ptr(), v_cache.data_ptr(),
        cache_str[0], cache_str[1], cache_str[2], num_blocks,
        block_table.data_ptr(), block_table.stride(0),
        cache_seqlens.data_ptr(), B, Hq, Hkv, D, block_size, max_blocks,
        float(softmax_scale),
        out3.data_ptr(), out3.stride(0), out3.stride(1),
        ws.data_ptr(), ws.numel(), stream)
    check("kvp_paged_decode_bf16", rc)
    return out


def paged_decode_fused(qkv: torch.Tensor, cos_sin: torch.Tensor,
                       q_norm_weight: torch.Tensor, k_norm_weight: torch.Tensor, eps: float,
                       num_q_heads: int, num_kv_heads: int, k_cache: torch.Tensor,
                       v_cache: torch.Tensor, slot_mapping: torch.Tensor, cache_seqlens: torch.Tensor,
                       block_table: torch.Tensor, softmax_scale: float,
                       out: torch.Tensor | None = None) -> torch.Tensor:
    """A Qwen3 decode step of one attention layer in one launch: q/k RMSNorm + RoPE of
    each sequence's new token from its qkv row, the append of its k / v at slot_mapping,
    and paged decode attention over cache_seqlens tokens (the last one being the new
    token).  Returns [B, Hq, 128] bf16.  The token's position is cache_seqlens - 1 and
    slot_mapping must hold the slot of that position, as the engine's decode metadata
    has them."""
    B = qkv.shape[0]
    D = k_cache.shape[-1]
    for name, t in (("qkv", qkv), ("k_cache", k_cache), ("v_cache", v_cache)):
        _require_cuda_bf16(name, t)
    if qkv.dim() != 2 or qkv.stride(1) != 1 or qkv.shape[1] != (num_q_heads + 2 * num_kv_heads) * D:
        raise ValueError("qkv must be [B, (Hq + 2 Hkv) * head_dim] with contiguous rows")
    if k_cache.shape != v_cache.shape or k_cache.stride() != v_cache.stride():
        raise ValueError("k_cache and v_cache must share shape and strides")
    num_blocks, block_size, Hkv, _ = k_cache.shape
    if Hkv != num_kv_heads:
        raise ValueError("cache heads do not match num_kv_heads")
    for name, t in (("slot_mapping", slot_mapping), ("cache_seqlens", cache_seqlens)):
        _require_int32(name, t, qkv.device)
        if t.numel() < B:
            raise ValueError(f"{name} has fewer rows than qkv")
    if cos_sin.dtype != torch.float32 or not cos_sin.is_contiguous() or cos_sin.shape[1] != D:
        raise ValueError("cos_sin must be a contiguous fp32 [max_position, head_dim] table")
    if block_table.dtype != torch.int32 or block_table.dim() != 2 or block_table.stride(1) != 1:
        raise ValueError("block_table must be an int32 [B, max_blocks] tensor with contiguous rows")
    if out is None:
        out = torch.empty(B, num_q_heads, D, dtype=torch.bfloat16, device=qkv.device)
    max_blocks = block_table.shape[1]
    stream = _stream(qkv)
    ws = _decode_workspace(qkv.get_device(), stream, B, num_q_heads, D, max_blocks, block_size)
    rc = lib().kvp_paged_decode_fused_bf16(
        qkv.data_ptr(), qkv.stride(0), cos_sin.data_ptr(), cos_sin.shape[0],
        q_norm_weight.data_ptr(), k_norm_weight.data_ptr(), float(eps),
        k_cache.data_ptr(), v_cache.data_ptr(), k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
        num_blocks, slot_mapping.data_ptr(), block_table.data_ptr(), block_table.stride(0),
        cache_seqlens.data_ptr(), B, num_q_heads, num_kv_heads, D, block_size, max_blocks,
        float(softmax_scale), out.data_ptr(), out.stride(0), out.stride(1),
        ws.data_ptr(), ws.numel(), stream)
    check("kvp_paged_decode_fused_bf16", rc)
    return out


# ----------------------------------------------------------------------------- prefill

def varlen_prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, max_seqlen_q: int,
                   cu_seqlens_q: torch.Tensor, max_seqlen_k: int, cu_seqlens_k: torch.Tensor,
                   softmax_scale: float, causal: bool = True,
                   block_table: torch.Tensor | None = None,
                   out: torch.Tensor | None = None) -> torch.Tensor:
    """Packed variable-length attention over dense or paged K/V (bf16 MFMA).

    Argument meaning follows flash_attn_varlen_func as called at
    kavor/layers/attention/flash_attention_kvcache.py:76-79: q is [Tq, Hq, D]; with
    block_table None, k / v are [Tk, Hkv, D] rows addressed through cu_seqlens_k; with
    a block_table they are the paged caches [num_blocks, block_size, Hkv, D].  The
    causal mask is bottom-right aligned.  Returns [Tq, Hq, D] bf16.  The kernel reads lengths
    on the device; max_seqlen_k (0 or no int: unknown) only helps to choose the launch.
    """
    Tq, Hq, D = q.shape
    _require_cuda_bf16("q", q)
    _require_cuda_bf16("k", k)
    _require_cuda_bf16("v", v)
    _require_int32("cu_seqlens_q", cu_seqlens_q, q.device)
    _require_int32("cu_seqlens_k", cu_seqlens_k, q.device)
    num_seqs = cu_seqlens_q.numel() - 1
    if cu_seqlens_k.numel() != num_seqs + 1:
        raise ValueError("cu_seqlens_q and cu_seqlens_k must have the same length")
    if q.stride(2) != 1 or k.stride(-1) != 1 or v.stride(-1) != 1:
        raise ValueError("head_dim must be contiguous in q, k and v")
    if out is None:
        out = torch.empty(Tq, Hq, D, dtype=torch.bfloat16, device=q.device)
    if block_table is None:
        if k.dim() != 3 or v.shape != k.shape:
            raise ValueError("dense k / v must be [Tk, Hkv, D] of equal shape")
        Hkv = k.shape[1]
        kstr = (0, k.stride(0), k.stride(1))
        vstr = (0, v.stride(0), v.stride(1))
        bt_ptr, bt_stride, num_blocks, block_size, max_blocks = 0, 0, 0, 0, 0
    else:
        if k.dim() != 4 or v.shape != k.shape:
            raise ValueError("paged k / v must be [num_blocks, block_size, Hkv, D] of equal shape")
        if block_table.dtype != torch.int32 or block_table.dim() != 2 or block_table.stride(1) != 1:
            raise ValueError("block_table must be an int32 [B, max_blocks] tensor with contiguous rows")
        if block_table.shape[0] < num_seqs:
            raise ValueError("block_table has fewer rows than sequences")
        num_blocks, block_size, Hkv = k.shape[0], k.shape[1], k.shape[2]
        kstr = (k.stride(0), k.stride(1), k.stride(2))
        vstr = (v.stride(0), v.stride(1), v.stride(2))
        bt_ptr, bt_stride, max_blocks = block_table.data_ptr(), block_table.stride(0), block_table.shape[1]
    if k.shape[-1] != D:
        raise ValueError("head_dim mismatch between q and k")
    ws, stream = None, _stream(q)
    if num_seqs:
        max_keys = max_blocks * block_size if block_table is not None else int(max_seqlen_q)
        if isinstance(max_seqlen_k, int) and 0 < max_seqlen_k < max_keys:
            max_keys = max_seqlen_k
        ws = _prefill_workspace(q.get_device(), stream, num_seqs, Tq, int(max_seqlen_q), max_keys if causal else 0, Hq,
                                Hkv)
    rc = lib().kvp_varlen_prefill_bf16(
        q.data_ptr(), q.stride(0), q.stride(1),
        k.data_ptr(), *kstr,
        v.data_ptr(), *vstr,
        bt_ptr, bt_stride, num_blocks, block_size, max_blocks,
        cu_seqlens_q.data_ptr(), cu_seqlens_k.data_ptr(), num_seqs, int(max_seqlen_q),
        Hq, Hkv, D, float(softmax_scale), 1 if causal else 0,
        out.data_ptr(), out.stride(0), out.stride(1),
        ws.data_ptr() if ws is not None else 0, ws.numel() if ws is not None else 0, stream)
    check("kvp_varlen_prefill_bf16", rc)
    return out


# flash-attn spellings, so call sites written against flash_attn keep working.
flash_attn_with_kvcache = paged_decode
flash_attn_varlen_func = varlen_prefill


# ----------------------------------------------------------------------------- module

class Attention(nn.Module):
    """Paged-KV attention layer; same constructor, attributes and forward as
    kavor/layers/attention/flash_attention_kvcache.py:49-84.

    k_cache / v_cache are lists with one entry per KV slot (num_kv_slots); a page pool
    binds them by duck typing (kavor/engine/cache_pool.py:98-101, 311-322).  forward
    appends k / v when a cache is bound, then runs varlen prefill (paged when the
    context carries block tables) or paged decode, reading the global Context.
    """

    def __init__(self, num_heads, head_dim, scale, num_kv_heads, num_kv_slots: int = 1):
        super().__init__()
        self.num_heads = num_heads
        self.head_dim = head_dim
        self.scale = scale
        self.num_kv_heads = num_kv_heads
        self.num_kv_slots = num_kv_slots
        self.k_cache = [torch.tensor([]) for _ in range(num_kv_slots)]
        self.v_cache = [torch.tensor([]) for _ in range(num_kv_slots)]

    def forward(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, slot: int = 0):
        context = get_context()
        k_cache, v_cache = self.k_cache[slot], self.v_cache[slot]
        if k_cache.numel() and v_cache.numel():
            store_kvcache(k, v, k_cache, v_cache, context.slot_mapping)
        if context.is_prefill:
            if context.block_tables is not None:  # prefix cache: attend over the pages
                k, v = k_cache, v_cache
            return self._prefill(q, k, v, context)
        return self._decode(q, k_cache, v_cache, context)

    def forward_cached(self, q: torch.Tensor, slot: int = 0):
        """Attention over the pages when the caller has already appended this step's k / v
        (the fused q/k-norm + RoPE + append kernel).  Prefill then always reads the pages,
        so the context must carry block tables."""
        context = get_context()
        k_cache, v_cache = self.k_cache[slot], self.v_cache[slot]
        if context.is_prefill:
            if context.block_tables is None:
                raise ValueError("forward_cached prefill reads the pages: the context needs block tables")
            return self._prefill(q, k_cache, v_cache, context)
        return self._decode(q, k_cache, v_cache, context)

    def _prefill(self, q, k, v, context):
        return varlen_prefill(q, k, v, max_seqlen_q=context.max_seqlen_q,
                              cu_seqlens_q=context.cu_seqlens_q,
                              max_seqlen_k=context.max_seqlen_k,
                              cu_seqlens_k=context.cu_seqlens_k,
                              softmax_scale=self.scale, causal=True,
                              block_table=context.block_tables)

    def _decode(self, q, k_cache, v_cache, context):
        return paged_decode(q.unsqueeze(1), k_cache, v_cache,
                            cache_seqlens=context.context_lens,
                            block_table=context.block_tables,
                            softmax_scale=self.scale, causal=True)
