"""Tensor-level wrappers over the C ABI: argument checks, output allocation, workspaces, streams.

Every op launches on the current HIP stream of its tensors' device and never synchronizes. Bad
arguments raise ``RuntimeError`` before anything is launched (the convention of a TORCH_CHECK).
Workspaces are device scratch buffers owned here (one per kind, device and stream, grown on
demand and reserved before any graph capture); kernels never need them zeroed.
"""

from __future__ import annotations

import contextlib
import functools

import torch
from torch import Tensor

from miniserve_amd import _native

EPI_NONE, EPI_SILU_MUL, EPI_RESIDUAL = 0, 1, 2


def _check(cond: bool, msg: str) -> None:
    if not cond:
        raise RuntimeError(msg)


# Pointer and stream arguments go to ctypes as plain ints (None for NULL): every C-ABI signature
# declares them c_void_p, so ctypes converts them itself.
def _ptr(t: Tensor | None) -> int | None:
    return t.data_ptr() if t is not None else None


# The current HIP stream of a device as a raw handle (what ``torch.cuda.current_stream(d).cuda_stream``
# returns, without building a Stream object: a few microseconds less host time per launch).
_raw_stream = torch._C._cuda_getCurrentRawStream


def _stream(t: Tensor) -> int:
    return _raw_stream(t.device.index)


def _on_gpu(*ts: Tensor) -> None:
    dev = ts[0].get_device()  # -1 for a CPU tensor
    for t in ts:
        d = t.get_device()
        if d != dev or d < 0:
            _check(t.is_cuda, "miniserve_amd ops run on the GPU only (got a CPU tensor)")
            _check(False, "all tensors of an op must be on one device")


class _Workspaces:
    """Device scratch per (kind, device, stream): calls on one stream are ordered by it, so they
    share a buffer; calls on different streams (concurrent graph branches) never do."""

    def __init__(self) -> None:
        self._bufs: dict[tuple[str, int, int], Tensor] = {}

    def get(
        self, kind: str, device: torch.device, nbytes: int, stream: torch.cuda.Stream | None = None,
        need: int | None = None,
    ) -> Tensor | None:
        """The buffer of ``kind`` for the device's current stream (or for ``stream``: allocated on
        it, so that the allocator recycles it only behind that stream's work). ``need``: during a graph
        capture what is already there will do if it holds that many bytes (None if 0 and nothing is)."""
        if nbytes == 0:
            return None
        idx = device.index if device.index is not None else torch.cuda.current_device()
        key = (kind, idx, stream.cuda_stream if stream is not None else _raw_stream(idx))
        buf = self._bufs.get(key)
        if buf is None or buf.numel() < nbytes:
            if need is not None and (buf.numel() if buf is not None else 0) >= need:
                if torch.cuda.is_current_stream_capturing():
                    return buf
            _check(
                not torch.cuda.is_current_stream_capturing(),
                f"workspace '{kind}' must be reserved before graph capture (need {nbytes} bytes)",
            )
            size = max(nbytes, 2 * (buf.numel() if buf is not None else 0), 1 << 20)
            with torch.cuda.stream(stream) if stream is not None else contextlib.nullcontext():
                buf = torch.empty(size, dtype=torch.uint8, device=device)
            self._bufs[key] = buf
        return buf

    def reserve(self, kind: str, device: torch.device, nbytes: int) -> None:
        self.get(kind, device, nbytes)

    def linear(self, call: str, device: torch.device, m: int, n: int, k: int) -> tuple[int | None, int]:
        """(pointer, bytes) of the linears' scratch for ``call`` on an [m, k] x [n, k] product."""
        nbytes = _native.query(call + "_workspace_size", m, n, k)
        if not nbytes:
            return None, 0
        ws = self.get("linear", device, nbytes, None, _native.query("msa_int8_linear_min_workspace_size", m, n, k))
        return (ws.data_ptr(), ws.numel()) if ws is not None else (None, 0)


workspaces = _Workspaces()


# ---- int8 linears ---------------------------------------------------------------------------------


def int8_quantize(weight: Tensor) -> tuple[Tensor, Tensor]:
    """(qweight int8 [out, in], scale bf16 [out]) -- quant/int8.py:25-33 on the GPU."""
    _on_gpu(weight)
    _check(weight.dim() == 2, "int8_quantize expects a 2-D weight")
    _check(weight.dtype in (torch.bfloat16, torch.float32), "int8_quantize supports bf16 or float32 weights")
    w = weight.detach().contiguous()
    rows, cols = w.shape
    q = torch.empty(rows, cols, dtype=torch.int8, device=w.device)
    s = torch.empty(rows, dtype=torch.bfloat16, device=w.device)
    dtype_code = 0 if w.dtype == torch.bfloat16 else 1
    _native.call("msa_int8_quantize", _ptr(w), dtype_code, rows, cols, _ptr(q), _ptr(s), _stream(w))
    return q, s


def int8_linear(
    x: Tensor,
    qweight: Tensor,
    scale: Tensor,
    epilogue: int = EPI_NONE,
    residual: Tensor | None = None,
    out: Tensor | None = None,
) -> Tensor:
    """y = x @ bf16(qweight * scale)^T (quant/int8.py:35-37) with an optional fused epilogue.

    x [..., in] bf16. EPI_SILU_MUL treats the rows as [gate | up] and returns silu(g) * u
    [..., out/2]; EPI_RESIDUAL returns residual + y.
    """
    dev = x.get_device()  # -1 for a CPU tensor
    if dev < 0 or qweight.get_device() != dev or scale.get_device() != dev:
        _on_gpu(x, qweight, scale)
    if x.dtype != torch.bfloat16:
        raise RuntimeError("int8_linear: activations must be bf16")
    wshape, xshape = qweight.shape, x.shape
    if qweight.dtype != torch.int8 or len(wshape) != 2 or not qweight.is_contiguous():
        raise RuntimeError("int8_linear: bad qweight")
    n, k = wshape
    if scale.dtype != torch.bfloat16 or scale.numel() != n:
        raise RuntimeError("int8_linear: bad scale")
    if xshape[-1] != k:
        raise RuntimeError(f"int8_linear: x has {xshape[-1]} features, weight expects {k}")
    x2 = x if len(xshape) == 2 else x.reshape(-1, k)
    m = x2.shape[0]
    ldx, unit = x2.stride()
    if m == 1:
        ldx = k  # one row has no pitch, whatever stride its view carries
    px = x2.data_ptr()
    if unit != 1 or ldx % 8 != 0 or px % 16 != 0:
        x2 = x2.contiguous()
        ldx, px = k, x2.data_ptr()
    cols = n // 2 if epilogue == EPI_SILU_MUL else n
    if out is None:
        out = torch.empty((*xshape[:-1], cols), dtype=torch.bfloat16, device=x.device)
    elif out.shape[-1] != cols or not out.is_contiguous():
        raise RuntimeError("int8_linear: bad out")
    pr, ldr = None, 0
    if epilogue == EPI_RESIDUAL:
        _check(residual is not None and residual.shape[-1] == n, "int8_linear: residual epilogue needs residual")
        r2 = residual.reshape(-1, n)
        _check(r2.stride(-1) == 1 and r2.dtype == torch.bfloat16, "int8_linear: residual must be row-major bf16")
        pr, ldr = r2.data_ptr(), r2.stride(0)
    pw, nw = None, 0
    if _native.query("msa_int8_linear_workspace_size", m, n, k):
        pw, nw = workspaces.linear("msa_int8_linear", x.device, m, n, k)
    _native.call("msa_int8_linear", px, m, k, ldx, qweight.data_ptr(), scale.data_ptr(), n, out.data_ptr(), cols,
                 epilogue, pr, ldr, pw, nw, _raw_stream(dev))
    return out


def int8_linear_add_rmsnorm(
    x: Tensor, qweight: Tensor, scale: Tensor, residual: Tensor, norm_w: Tensor, eps: float, out: Tensor | None = None
) -> Tensor:
    """residual += x @ bf16(qweight * scale)^T (bf16 rounding of the product and the sum, in place),
    then returns RMSNorm(residual) with norm_w: the o / down projection with the next norm
    (model/qwen3.py:121-122). A GEMM that splits K merges its partials, adds and normalizes in one
    kernel (msa_int8_linear_add_rmsnorm)."""
    _on_gpu(x, qweight, scale, residual, norm_w)
    _check(x.dtype == torch.bfloat16 and x.dim() == 2 and x.stride(-1) == 1, "int8_linear_add_rmsnorm: x [m, k] bf16")
    _check(qweight.dtype == torch.int8 and qweight.is_contiguous(), "int8_linear_add_rmsnorm: bad qweight")
    n, k = qweight.shape
    m = x.shape[0]
    _check(x.shape[1] == k, "int8_linear_add_rmsnorm: x / weight feature mismatch")
    _check(residual.shape == (m, n) and residual.is_contiguous() and residual.dtype == torch.bfloat16,
           "int8_linear_add_rmsnorm: residual [m, n] contiguous bf16")
    _check(norm_w.dtype == torch.bfloat16 and norm_w.numel() == n, "int8_linear_add_rmsnorm: norm weight")
    if out is None:
        out = torch.empty_like(residual)
    _check(out.shape == (m, n) and out.is_contiguous(), "int8_linear_add_rmsnorm: bad out")
    pw, nw = workspaces.linear("msa_int8_linear_add_rmsnorm", x.device, m, n, k)
    _native.call(
        "msa_int8_linear_add_rmsnorm", _ptr(x), m, k, x.stride(0), _ptr(qweight), _ptr(scale), n, _ptr(residual),
        _ptr(norm_w), float(eps), _ptr(out), pw, nw, _stream(x),
    )
    return out


def default_split(m: int, n: int, k: int) -> int:
    """K splits for a split-K linear: none when the 32-row x 64-row output tiles give 128+
    workgroups, else about 256 workgroups, each split a whole multiple of four 64-wide K chunks
    (one per wavefront). The C ABI's default plan for msa_int8_linear makes the same choice."""
    chunks = -(-k // 64)
    blocks = -(-n // 32) * -(-m // 64)
    if blocks >= 128:
        return 1
    split = max(1, min(-(-256 // blocks), max(1, chunks // 4)))
    per = -(-chunks // split)
    per = -(-per // 4) * 4
    return max(1, -(-chunks // per))


def int8_linear_splitk(x: Tensor, qweight: Tensor, scale: Tensor, k_split: int) -> Tensor:
    """float32 partials [k_split, m, n] of x @ bf16(qweight * scale)^T over k_split ranges of K;
    bf16(partials.sum(0)) is the linear's output. Consumers sum them inside their own kernel."""
    _on_gpu(x, qweight, scale)
    _check(x.dtype == torch.bfloat16 and x.dim() == 2 and x.stride(-1) == 1, "int8_linear_splitk: x [m, k] bf16")
    _check(qweight.dtype == torch.int8 and qweight.is_contiguous(), "int8_linear_splitk: bad qweight")
    n, k = qweight.shape
    m = x.shape[0]
    part = torch.empty(k_split, m, n, dtype=torch.float32, device=x.device)
    _native.call("msa_int8_linear_splitk", _ptr(x), m, k, x.stride(0), _ptr(qweight), _ptr(scale), n, k_split,
                 _ptr(part), _stream(x))
    return part


def splitk_add_rmsnorm(
    partials: Tensor, residual: Tensor, weight: Tensor, eps: float, residual_out: Tensor | None = None
) -> tuple[Tensor, Tensor]:
    """(bf16(residual + bf16(sum of partials)), RMSNorm of it) in one kernel."""
    _on_gpu(partials, residual, weight)
    k_split, rows, dim = partials.shape
    _check(partials.dtype == torch.float32 and partials.is_contiguous(), "splitk_add_rmsnorm: partials")
    _check(residual.shape == (rows, dim) and residual.is_contiguous(), "splitk_add_rmsnorm: residual")
    if residual_out is None:
        residual_out = torch.empty_like(residual)
    out = torch.empty_like(residual)
    _native.call("msa_splitk_add_rmsnorm", _ptr(partials), k_split, _ptr(residual), _ptr(residual_out),
                 _ptr(weight), _ptr(out), rows, dim, float(eps), _stream(partials))
    return residual_out, out


def qk_norm_rope_cache_splitk(
    partials: Tensor,
    heads: int,
    kv_heads: int,
    head_dim: int,
    q_norm_w: Tensor,
    k_norm_w: Tensor,
    eps: float,
    cos: Tensor,
    sin: Tensor,
    slot_mapping: Tensor,
    k_cache: Tensor,
    v_cache: Tensor,
) -> Tensor:
    """qk_norm_rope_cache whose qkv rows arrive as split-K partials [k_split, T, (H+2KVH)*D]."""
    _on_gpu(partials, q_norm_w, k_norm_w, cos, sin, slot_mapping, k_cache, v_cache)
    k_split, t, cols = partials.shape
    _check(cols == (heads + 2 * kv_heads) * head_dim and partials.is_contiguous(), "qkv partials shape")
    _check(cos.shape == (t, head_dim) and sin.shape == (t, head_dim) and cos.dtype == torch.float32, "cos/sin")
    _check(slot_mapping.dtype == torch.int64 and slot_mapping.numel() == t, "slot_mapping")
    _check(k_cache.shape[-2:] == (kv_heads, head_dim) and k_cache.is_contiguous() and v_cache.is_contiguous(), "caches")
    q = torch.empty(t, heads, head_dim, dtype=torch.bfloat16, device=partials.device)
    _native.call(
        "msa_qk_norm_rope_cache_splitk", _ptr(partials), k_split, t, heads, kv_heads, head_dim, _ptr(q_norm_w),
        _ptr(k_norm_w), float(eps), _ptr(cos), _ptr(sin), _ptr(slot_mapping), _ptr(q), _ptr(k_cache), _ptr(v_cache),
        k_cache.shape[0], _stream(partials),
    )
    return q


# ---- norms / RoPE / cache -------------------------------------------------------------------------


def embed_rope_rows(
    ids: Tensor, positions: Tensor, weight: Tensor, cos_table: Tensor, sin_table: Tensor
) -> tuple[Tensor, Tensor, Tensor]:
    """(weight[ids] [T, hidden], cos_table[positions], sin_table[positions] [T, 128]) in one launch
    (model/qwen3.py:147-148); ids and positions out of range abort, as indexing on the GPU does."""
    _on_gpu(ids, positions, weight, cos_table, sin_table)
    for t in (ids, positions):
        _check(t.dtype == torch.int64 and t.dim() == 1 and t.is_contiguous() and t.numel() == ids.numel(),
               "embed_rope_rows: int64 [T] ids and positions")
    _check(weight.dtype == torch.bfloat16 and weight.dim() == 2 and weight.is_contiguous(), "embed_rope_rows: weight bf16")
    for c in (cos_table, sin_table):
        _check(c.dtype == torch.float32 and c.is_contiguous() and c.shape == (cos_table.shape[0], 128),
               "embed_rope_rows: float32 [positions, 128] tables")
    t, (vocab, hidden) = ids.numel(), weight.shape
    x = torch.empty(t, hidden, dtype=torch.bfloat16, device=ids.device)
    rows = torch.empty(2, t, 128, dtype=torch.float32, device=ids.device)
    _native.call("msa_embed_rope_rows", _ptr(ids), _ptr(positions), t, _ptr(weight), vocab, hidden, _ptr(cos_table),
                 _ptr(sin_table), cos_table.shape[0], _ptr(x), rows.data_ptr(), rows[1].data_ptr(), _stream(ids))
    return x, rows[0], rows[1]


def rmsnorm(x: Tensor, weight: Tensor, eps: float, out: Tensor | None = None) -> Tensor:
    """RMSNorm over the last dim (model/layers.py:18-22)."""
    _on_gpu(x, weight)
    _check(x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16, "rmsnorm: bf16 only")
    dim = x.shape[-1]
    _check(weight.numel() == dim, "rmsnorm: weight size mismatch")
    x2 = x.reshape(-1, dim)
    if x2.stride(-1) != 1:
        x2 = x2.contiguous()
    if out is None:
        out = torch.empty(x.shape, dtype=torch.bfloat16, device=x.device)
    o2 = out.view(-1, dim)
    _native.call("msa_rmsnorm", _ptr(x2), x2.stride(0), _ptr(weight), _ptr(o2), o2.stride(0), x2.shape[0], dim,
                 float(eps), _stream(x))
    return out


def add_rmsnorm(
    residual: Tensor, delta: Tensor, weight: Tensor, eps: float, residual_out: Tensor | None = None
) -> tuple[Tensor, Tensor]:
    """(bf16(residual + delta), RMSNorm of it) -- model/qwen3.py:121-122 fused."""
    _on_gpu(residual, delta, weight)
    _check(residual.shape == delta.shape and residual.is_contiguous() and delta.is_contiguous(), "add_rmsnorm: shapes")
    dim = residual.shape[-1]
    if residual_out is None:
        residual_out = torch.empty_like(residual)
    out = torch.empty_like(residual)
    _native.call("msa_add_rmsnorm", _ptr(residual), _ptr(delta), _ptr(residual_out), _ptr(weight), _ptr(out),
                 residual.numel() // dim, dim, float(eps), _stream(residual))
    return residual_out, out


def qk_norm_rope_cache(
    qkv: Tensor,
    heads: int,
    kv_heads: int,
    head_dim: int,
    q_norm_w: Tensor,
    k_norm_w: Tensor,
    eps: float,
    cos: Tensor,
    sin: Tensor,
    slot_mapping: Tensor,
    k_cache: Tensor,
    v_cache: Tensor,
) -> Tensor:
    """q/k-norm + RoPE of the fused qkv rows, k/v written to the cache; returns q [T, H, D]."""
    _on_gpu(qkv, q_norm_w, k_norm_w, cos, sin, slot_mapping, k_cache, v_cache)
    t = qkv.shape[0]
    _check(qkv.shape[-1] == (heads + 2 * kv_heads) * head_dim and qkv.stride(-1) == 1, "qk_norm_rope_cache: qkv shape")
    _check(cos.dtype == torch.float32 and cos.shape == (t, head_dim) and cos.is_contiguous(), "qk_norm_rope_cache: cos")
    _check(sin.dtype == torch.float32 and sin.shape == (t, head_dim) and sin.is_contiguous(), "qk_norm_rope_cache: sin")
    _check(slot_mapping.dtype == torch.int64 and slot_mapping.numel() == t, "qk_norm_rope_cache: slot_mapping")
    _check(k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape == v_cache.shape, "caches")
    _check(k_cache.shape[-2:] == (kv_heads, head_dim), "qk_norm_rope_cache: cache layout [slots, KVH, D]")
    q = torch.empty(t, heads, head_dim, dtype=torch.bfloat16, device=qkv.device)
    _native.call(
        "msa_qk_norm_rope_cache", _ptr(qkv), qkv.stride(0), t, heads, kv_heads, head_dim, _ptr(q_norm_w),
        _ptr(k_norm_w), float(eps), _ptr(cos), _ptr(sin), _ptr(slot_mapping), _ptr(q), _ptr(k_cache),
        _ptr(v_cache), k_cache.shape[0], _stream(qkv),
    )
    return q


def qkv_gemm_fuses_norm(m: int, heads: int, kv_heads: int, head_dim: int, k: int) -> bool:
    """Whether the qkv projection of ``m`` tokens takes the prefill GEMM with the q/k-norm, RoPE and
    cache write fused after it (``int8_linear_qk_norm_rope_cache``): in its epilogue, or in the
    kernel that merges its split-K partials."""
    return head_dim == 128 and m >= 128 and k % 64 == 0


def int8_linear_qk_norm_rope_cache(
    x: Tensor,
    qweight: Tensor,
    scale: Tensor,
    heads: int,
    kv_heads: int,
    head_dim: int,
    q_norm_w: Tensor,
    k_norm_w: Tensor,
    eps: float,
    cos: Tensor,
    sin: Tensor,
    slot_mapping: Tensor,
    k_cache: Tensor,
    v_cache: Tensor,
) -> Tensor:
    """``qk_norm_rope_cache(int8_linear(x, qweight, scale), ...)`` in one GEMM whose epilogue norms and
    rotates q and k and writes k / v to the cache -- the same values bit for bit; returns q [T, H, D]."""
    _on_gpu(x, qweight, scale, q_norm_w, k_norm_w, cos, sin, slot_mapping, k_cache, v_cache)
    t, k = x.shape
    _check(x.dtype == torch.bfloat16 and x.stride(-1) == 1, "int8_linear_qk_norm_rope_cache: x bf16 rows")
    _check(qweight.dtype == torch.int8 and qweight.is_contiguous()
           and qweight.shape == ((heads + 2 * kv_heads) * head_dim, k), "int8_linear_qk_norm_rope_cache: qweight")
    _check(scale.dtype == torch.bfloat16 and scale.numel() == qweight.shape[0], "int8_linear_qk_norm_rope_cache: scale")
    _check(cos.dtype == torch.float32 and cos.shape == (t, head_dim) and cos.is_contiguous(), "cos [T, D] float32")
    _check(sin.dtype == torch.float32 and sin.shape == (t, head_dim) and sin.is_contiguous(), "sin [T, D] float32")
    _check(slot_mapping.dtype == torch.int64 and slot_mapping.numel() == t, "slot_mapping [T] int64")
    _check(k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape == v_cache.shape, "caches")
    _check(k_cache.shape[-2:] == (kv_heads, head_dim), "cache layout [slots, KVH, D]")
    q = torch.empty(t, heads, head_dim, dtype=torch.bfloat16, device=x.device)
    pw, nw = workspaces.linear("msa_int8_gemm_qk_norm_rope_cache", x.device, t, qweight.shape[0], k)
    _native.call(
        "msa_int8_gemm_qk_norm_rope_cache", _ptr(x), t, k, x.stride(0), _ptr(qweight), _ptr(scale), heads, kv_heads,
        head_dim, _ptr(q_norm_w), _ptr(k_norm_w), float(eps), _ptr(cos), _ptr(sin), _ptr(slot_mapping), _ptr(q),
        _ptr(k_cache), _ptr(v_cache), k_cache.shape[0], pw, nw, _stream(x),
    )
    return q


def reshape_and_cache(k: Tensor, v: Tensor, k_cache: Tensor, v_cache: Tensor, slot_mapping: Tensor) -> None:
    """k_cache[slot_mapping] = k; v_cache[slot_mapping] = v (attention/backends.py:159-160)."""
    _on_gpu(k, v, k_cache, v_cache, slot_mapping)
    t, kvh, d = k.shape
    if v.shape != k.shape or k_cache.shape[-2:] != (kvh, d):
        raise RuntimeError("reshape_and_cache: shapes")
    if slot_mapping.dtype != torch.int64 or slot_mapping.numel() != t:
        raise RuntimeError("reshape_and_cache: slot_mapping")
    ks, vs = k.stride(), v.stride()
    k2 = k if ks[2] == 1 and ks[1] == d else k.contiguous()
    v2 = v if vs[2] == 1 and vs[1] == d else v.contiguous()
    _native.call("msa_reshape_and_cache", _ptr(k2), k2.stride(0), _ptr(v2), v2.stride(0), t, kvh, d,
                 _ptr(slot_mapping), _ptr(k_cache), _ptr(v_cache), k_cache.shape[0], _stream(k))


# ---- paged attention ------------------------------------------------------------------------------


DECODE_MAX_PART_TOKENS = 4096  # keys per decode split: 64 blocks per wavefront of a four-wavefront workgroup
DECODE_MAX_SPLITS = 32  # splits per sequence at most, at the longest context a plan is keyed on
DECODE_SPLIT_FILL_MAX_TOKENS = 2048  # longest split the workgroup-fill target picks below 256 pairs


def decode_splits(
    num_seqs: int, kv_heads: int, max_blocks: int, group: int, split_context: int | None = None
) -> tuple[int, int]:
    """(partition_tokens, partitions) for the decode kernel (``group`` = query heads per KV head).

    The keys per split depend only on the batch's shape -- its (sequence, KV head) count and the
    group size -- and on ``split_context``, the longest context the caller plans for (the runner's
    max_model_len, the same for a step captured in a graph and the same step run eagerly; by
    default the block-table width), never on the contexts themselves, so a captured step (tables
    padded to the longest context the graph accepts) and the eager step split every sequence at
    the same keys and sum in the same order. When the pairs alone give 256+ workgroups: one split
    per sequence up to 4096 keys (256 sequences x 8 KV heads at G = 4, contexts U[512, 4096]:
    408 us against 419 with 2048-key splits). Otherwise splits sized so the planned context fills
    about 256 workgroups (one per CU), a power of two from 64 to 2048 keys, and at least
    split_context / 32 keys, so a sequence at the planned maximum has no more than 32 splits to
    merge. Measured on 16 q / 8 KV heads against the former ~512-workgroup target (us per launch):
    4 x U[2048, 4096] 24.0 -> 15.7, 2 x 8192 24.7 -> 19.5, 8 x U[4096, 8192] 45.9 -> 38.3,
    16 x U[128, 1024] 14.8 -> 12.8, 4 x 32768 99.6 -> 93.9, 16 x U[16384, 32768] 298.5 -> 286.0;
    batch 1 at 4096 and at 32768 keys unchanged (128- and 1024-key splits). ``partitions`` only
    sizes the grid to cover the table width; a sequence uses ceil(context / partition_tokens)."""
    wgs = max(1, num_seqs * kv_heads)
    if wgs >= 256:
        part = DECODE_MAX_PART_TOKENS
    else:
        ctx = split_context if split_context else max_blocks * 16
        fill = -(-ctx * wgs // (256 * 16))  # blocks per split for ~256 workgroups at the planned context
        blocks = max(4, min(fill, DECODE_SPLIT_FILL_MAX_TOKENS // 16), -(-ctx // (16 * DECODE_MAX_SPLITS)))
        part = 16 * min(1 << (blocks - 1).bit_length(), DECODE_MAX_PART_TOKENS // 16)
    return part, max(1, -(-max_blocks * 16 // part))


@functools.lru_cache(maxsize=1024)  # plain arithmetic of five whole numbers, asked once a layer
def decode_plan(
    num_seqs: int, kv_heads: int, max_blocks: int, group: int, split_context: int | None = None
) -> tuple[int, int]:
    """``decode_splits`` as the attention calls use it: a plan of more than 2048 keys per CU runs in
    rounds of 2048-key workgroups, and where those leave much of the last round empty the splits are
    halved, when that wastes less and still gives at most 32 of them. Like decode_splits it depends on
    the batch's shape and the planned context alone. Measured at 32 q / 8 KV heads (us with the merge):
    3 x U[20000, 32768], a round and a half, 77.3 -> 66.6; 6 x U[8000, 16000] 73.8 -> 66.0. Whole rounds
    keep 2048 keys (31 x U[500, 4096] at 16 q heads 53.3 against 60.5 with 1024)."""
    part, partitions = decode_splits(num_seqs, kv_heads, max_blocks, group, split_context)
    ctx = split_context if split_context else max_blocks * 16
    keys = -(-ctx * num_seqs * kv_heads // 256)  # per CU
    half = DECODE_SPLIT_FILL_MAX_TOKENS // 2
    if (
        num_seqs * kv_heads < 256
        and part == 2 * half < keys
        and max(ctx, max_blocks * 16) <= DECODE_MAX_SPLITS * half
        and -(-keys // half) * half < -(-keys // part) * part
    ):
        return half, max(1, -(-max_blocks * 16 // half))
    return part, partitions


def paged_attention_decode(
    q: Tensor,
    k_cache: Tensor,
    v_cache: Tensor,
    block_tables: Tensor,
    context_lens: Tensor,
    q_rows: Tensor,
    partition_tokens: int,
    max_partitions: int,
    scale: float,
    out: Tensor,
    block_size: int = 16,
    narrow: bool = False,
    stream: torch.cuda.Stream | None = None,
) -> Tensor:
    """Decode attention through the block table; (partition_tokens, max_partitions) as from
    ``decode_splits``; partition_tokens * max_partitions must cover the block-table width.
    ``narrow``: four-wavefront workgroups at every partition size (msa_paged_attention_decode_narrow),
    for decode rows attended beside another kernel running on another stream. ``stream``: launch on
    this stream instead of the current one (its own workspace)."""
    _on_gpu(q, k_cache, v_cache, block_tables, context_lens, q_rows, out)
    _, heads, d = q.shape
    kvh = k_cache.shape[1]
    num = context_lens.numel()
    _check(block_tables.dtype == torch.int32 and block_tables.is_contiguous() and block_tables.shape[0] == num,
           "paged_attention_decode: block_tables")
    _check(context_lens.dtype == torch.int32 and q_rows.dtype == torch.int32, "paged_attention_decode: int32 metadata")
    ws_bytes = _native.query("msa_paged_attention_decode_workspace_size", num, heads, d, max_partitions)
    ws = workspaces.get("attention", q.device, ws_bytes, stream)
    _native.call(
        "msa_paged_attention_decode_narrow" if narrow else "msa_paged_attention_decode", _ptr(q), q.stride(0),
        _ptr(k_cache), _ptr(v_cache), k_cache.shape[0], heads,
        kvh, d, block_size, _ptr(block_tables), block_tables.shape[1], _ptr(context_lens), _ptr(q_rows), num,
        partition_tokens, max_partitions, float(scale), _ptr(out), out.stride(0), _ptr(ws),
        ws.numel() if ws is not None else 0, stream.cuda_stream if stream is not None else _stream(q),
    )
    return out


def paged_attention_decode_qkv(
    qkv: Tensor,
    heads: int,
    q_norm_w: Tensor,
    k_norm_w: Tensor,
    qk_eps: float,
    cos_table: Tensor,
    sin_table: Tensor,
    slot_mapping: Tensor,
    k_cache: Tensor,
    v_cache: Tensor,
    block_tables: Tensor,
    context_lens: Tensor,
    q_rows: Tensor,
    partition_tokens: int,
    max_partitions: int,
    scale: float,
    out: Tensor,
    block_size: int = 16,
    rope_rows: bool = False,
) -> Tensor:
    """Decode attention from the qkv projection rows [q | k | v] (msa_paged_attention_decode_qkv):
    per-head q/k RMSNorm and RoPE at position context_len - 1, the new key and value written into
    the caches at slot_mapping (negative slots are skipped), attention over the cached keys plus
    the new one. out [T, heads, head_dim]. ``rope_rows``: cos_table / sin_table hold one row per row
    of qkv, gathered by the caller (msa_paged_attention_decode_qkv_rows)."""
    _on_gpu(qkv, q_norm_w, k_norm_w, cos_table, sin_table, slot_mapping, k_cache, v_cache, block_tables, context_lens,
            q_rows, out)
    _check(slot_mapping.dtype == torch.int64 and slot_mapping.numel() == qkv.shape[0], "paged_attention_decode_qkv: slots")
    _, kvh, d = k_cache.shape
    _check(qkv.dtype == torch.bfloat16 and qkv.dim() == 2 and qkv.stride(-1) == 1
           and qkv.shape[1] == (heads + 2 * kvh) * d, "paged_attention_decode_qkv: qkv [T, (H + 2 KVH) * D]")
    _check(cos_table.dtype == torch.float32 and cos_table.is_contiguous() and cos_table.shape[-1] == d
           and sin_table.shape == cos_table.shape and sin_table.is_contiguous(), "paged_attention_decode_qkv: rotary")
    _check(not rope_rows or cos_table.shape[0] == qkv.shape[0], "paged_attention_decode_qkv: a rotary row per qkv row")
    _check(k_cache.is_contiguous() and v_cache.is_contiguous(), "paged_attention_decode_qkv: caches")
    num = context_lens.numel()
    _check(block_tables.dtype == torch.int32 and block_tables.is_contiguous() and block_tables.shape[0] == num,
           "paged_attention_decode_qkv: block_tables")
    _check(context_lens.dtype == torch.int32 and q_rows.dtype == torch.int32, "paged_attention_decode_qkv: metadata")
    ws_bytes = _native.query("msa_paged_attention_decode_workspace_size", num, heads, d, max_partitions)
    ws = workspaces.get("attention", qkv.device, ws_bytes)
    o2 = out.view(out.shape[0], -1)
    _native.call(
        "msa_paged_attention_decode_qkv_rows" if rope_rows else "msa_paged_attention_decode_qkv", _ptr(qkv),
        qkv.stride(0), _ptr(q_norm_w), _ptr(k_norm_w), float(qk_eps),
        _ptr(cos_table), _ptr(sin_table), cos_table.shape[0], _ptr(slot_mapping), _ptr(k_cache), _ptr(v_cache),
        k_cache.shape[0], heads,
        kvh, d, block_size, _ptr(block_tables), block_tables.shape[1], _ptr(context_lens), _ptr(q_rows), num,
        partition_tokens, max_partitions, float(scale), _ptr(o2), o2.stride(0), _ptr(ws),
        ws.numel() if ws is not None else 0, _stream(qkv),
    )
    return out


def paged_attention_prefill(
    q: Tensor,
    k_cache: Tensor,
    v_cache: Tensor,
    block_tables: Tensor,
    seq_info: Tensor,
    work: Tensor,
    scale: float,
    out: Tensor,
    block_size: int = 16,
    wide: bool = False,
) -> Tensor:
    """``work`` lists query tiles of 64 / (H / KVH) tokens (``wide``: of 128 / (H / KVH))."""
    _on_gpu(q, k_cache, v_cache, block_tables, seq_info, work, out)
    _, heads, d = q.shape
    kvh = k_cache.shape[1]
    _check(seq_info.dtype == torch.int32 and work.dtype == torch.int32 and block_tables.dtype == torch.int32,
           "paged_attention_prefill: int32 metadata")
    _native.call(
        "msa_paged_attention_prefill_wide" if wide else "msa_paged_attention_prefill", _ptr(q), q.stride(0), _ptr(k_cache), _ptr(v_cache), k_cache.shape[0], heads,
        kvh, d, block_size, _ptr(block_tables), block_tables.shape[1], _ptr(seq_info), _ptr(work), work.shape[0],
        float(scale), _ptr(out), out.stride(0), _stream(q),
    )
    return out


# ---- token-split int8 linears with fused prologues / epilogues ------------------------------------

ROWS_MAX_TOKENS = 256  # above this the split-K kernels (or a prefill GEMM) serve the shape


def rows_supported(k: int) -> bool:
    """Whether msa_int8_linear_rows / msa_qkv_rope_cache_rows take this in_features (the [16, k]
    activation tile has to fit in LDS next to the kernel's other scratch)."""
    return k % 64 == 0 and 16 * (k + 8) * 2 + 16 * 1024 <= 160 * 1024


def int8_linear_rows(
    x: Tensor,
    qweight: Tensor,
    scale: Tensor,
    epilogue: int = EPI_NONE,
    residual: Tensor | None = None,
    out: Tensor | None = None,
    norm_w: Tensor | None = None,
    eps: float = 0.0,
) -> Tensor:
    """y = [RMSNorm](x) @ bf16(qweight * scale)^T with the epilogue fused (token-split kernel).

    x [m, k] bf16. ``norm_w`` applies RMSNorm(x) (model/layers.py:18-22) before the product
    (SILU_MUL only). EPI_RESIDUAL returns residual + y and may write in place (out=residual).
    """
    _on_gpu(x, qweight, scale)
    _check(x.dtype == torch.bfloat16 and x.dim() == 2 and x.stride(-1) == 1, "int8_linear_rows: x [m, k] bf16")
    _check(qweight.dtype == torch.int8 and qweight.is_contiguous(), "int8_linear_rows: bad qweight")
    n, k = qweight.shape
    m = x.shape[0]
    _check(x.shape[1] == k, "int8_linear_rows: x / weight feature mismatch")
    cols = n // 2 if epilogue == EPI_SILU_MUL else n
    if out is None:
        out = torch.empty(m, cols, dtype=torch.bfloat16, device=x.device)
    _check(out.shape == (m, cols) and out.stride(-1) == 1, "int8_linear_rows: bad out")
    r2 = None
    if epilogue == EPI_RESIDUAL:
        _check(residual is not None and residual.shape == (m, n) and residual.stride(-1) == 1, "int8_linear_rows: residual")
        r2 = residual
    if norm_w is not None:
        _check(norm_w.dtype == torch.bfloat16 and norm_w.numel() == k, "int8_linear_rows: norm weight")
    _native.call(
        "msa_int8_linear_rows", _ptr(x), x.stride(0), m, k, _ptr(norm_w), float(eps), _ptr(qweight), _ptr(scale), n,
        epilogue, _ptr(out), out.stride(0), _ptr(r2), r2.stride(0) if r2 is not None else 0, _stream(x),
    )
    return out


DEC_MAX_TOKENS = 128  # decode-sized batches the pipeline sends to msa_int8_linear_dec


WIDE_MIN_WEIGHTS = 12 << 20  # int8 weights of this many bytes: one launch streams for longer than it takes to start
STREAM_MAX_TOKENS = 16  # tokens the streaming decode linear (RMSNorm prologue included) serves


def dec_supported(k: int) -> bool:
    """Whether msa_int8_linear_dec takes this in_features (K split over 4-16 wavefronts of four
    64-wide chunks each)."""
    return k in (1024, 2048, 3072, 4096)


def int8_linear_dec(
    x: Tensor,
    qweight: Tensor,
    scale: Tensor,
    epilogue: int = EPI_NONE,
    residual: Tensor | None = None,
    out: Tensor | None = None,
    norm_w: Tensor | None = None,
    eps: float = 0.0,
    gather: Tensor | None = None,
    x_copy: Tensor | None = None,
) -> Tensor:
    """y = [RMSNorm]([x[gather]]) @ bf16(qweight * scale)^T with the epilogue fused, for
    decode-sized batches (msa_int8_linear_dec).

    x [rows, k] bf16. ``gather`` (int64 [m]) takes the activation rows x[gather] (the embedding
    lookup) and, with ``x_copy`` [m, k], also writes them there (the residual stream); it needs
    ``norm_w`` and EPI_NONE. ``norm_w`` applies RMSNorm (model/layers.py:18-22) before the product.
    EPI_RESIDUAL returns residual + y and may write in place (out=residual).
    """
    _on_gpu(x, qweight, scale)
    _check(x.dtype == torch.bfloat16 and x.dim() == 2 and x.stride(-1) == 1, "int8_linear_dec: x [rows, k] bf16")
    _check(qweight.dtype == torch.int8 and qweight.is_contiguous(), "int8_linear_dec: bad qweight")
    n, k = qweight.shape
    _check(x.shape[1] == k, "int8_linear_dec: x / weight feature mismatch")
    if gather is not None:
        _check(gather.dtype == torch.int64 and gather.dim() == 1 and gather.is_contiguous(), "int8_linear_dec: gather")
        m = gather.numel()
    else:
        m = x.shape[0]
    cols = n // 2 if epilogue == EPI_SILU_MUL else n
    if out is None:
        out = torch.empty(m, cols, dtype=torch.bfloat16, device=x.device)
    _check(out.shape == (m, cols) and out.stride(-1) == 1, "int8_linear_dec: bad out")
    r2 = None
    if epilogue == EPI_RESIDUAL:
        _check(residual is not None and residual.shape == (m, n) and residual.stride(-1) == 1, "int8_linear_dec: residual")
        r2 = residual
    if norm_w is not None:
        _check(norm_w.dtype == torch.bfloat16 and norm_w.numel() == k, "int8_linear_dec: norm weight")
    if x_copy is not None:
        _check(x_copy.shape == (m, k) and x_copy.stride(-1) == 1, "int8_linear_dec: x_copy")
    _native.call(
        "msa_int8_linear_dec", _ptr(x), x.stride(0), x.shape[0], _ptr(gather), _ptr(x_copy),
        x_copy.stride(0) if x_copy is not None else 0, m, k, _ptr(norm_w), float(eps), _ptr(qweight), _ptr(scale), n,
        epilogue, _ptr(out), out.stride(0), _ptr(r2), r2.stride(0) if r2 is not None else 0, _stream(x),
    )
    return out


def qkv_rope_cache_rows(
    x: Tensor,
    qweight: Tensor,
    scale: Tensor,
    heads: int,
    kv_heads: int,
    head_dim: int,
    q_norm_w: Tensor,
    k_norm_w: Tensor,
    qk_eps: float,
    positions: Tensor,
    cos_table: Tensor,
    sin_table: Tensor,
    slot_mapping: Tensor,
    k_cache: Tensor,
    v_cache: Tensor,
    norm_w: Tensor | None = None,
    eps: float = 0.0,
    gather: Tensor | None = None,
    x_copy: Tensor | None = None,
) -> Tensor:
    """The attention block's front half in one kernel: [gather rows] -> [RMSNorm] -> int8 qkv
    projection -> per-head q/k RMSNorm -> RoPE -> k/v written at slot_mapping; returns q [T, H, D].

    With ``gather`` (int64 [T]) the activation rows are x[gather] (the embedding lookup) and are
    also written to ``x_copy`` [T, k] (the residual stream) when given. cos/sin tables are the
    rotary's float32 [max_positions, D] tables, indexed by ``positions`` inside the kernel.
    """
    _on_gpu(x, qweight, scale, q_norm_w, k_norm_w, positions, cos_table, sin_table, slot_mapping, k_cache, v_cache)
    _check(x.dtype == torch.bfloat16 and x.dim() == 2 and x.stride(-1) == 1, "qkv_rope_cache_rows: x")
    n, k = qweight.shape
    _check(n == (heads + 2 * kv_heads) * head_dim and x.shape[1] == k, "qkv_rope_cache_rows: qkv weight shape")
    t = gather.numel() if gather is not None else x.shape[0]
    _check(positions.dtype == torch.int64 and positions.numel() == t, "qkv_rope_cache_rows: positions")
    _check(slot_mapping.dtype == torch.int64 and slot_mapping.numel() == t, "qkv_rope_cache_rows: slot_mapping")
    _check(cos_table.dtype == torch.float32 and cos_table.is_contiguous() and cos_table.shape[-1] == head_dim, "cos")
    _check(sin_table.shape == cos_table.shape and sin_table.is_contiguous(), "sin")
    _check(k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape[-2:] == (kv_heads, head_dim), "caches")
    if gather is not None:
        _check(gather.dtype == torch.int64 and gather.is_contiguous(), "qkv_rope_cache_rows: gather")
        _check(norm_w is not None, "qkv_rope_cache_rows: gathered rows need norm_w")
    if x_copy is not None:
        _check(x_copy.shape == (t, k) and x_copy.stride(-1) == 1, "qkv_rope_cache_rows: x_copy")
    q = torch.empty(t, heads, head_dim, dtype=torch.bfloat16, device=x.device)
    _native.call(
        "msa_qkv_rope_cache_rows", _ptr(x), x.stride(0), x.shape[0], _ptr(gather), _ptr(norm_w), float(eps), _ptr(x_copy),
        x_copy.stride(0) if x_copy is not None else 0, t, k, _ptr(qweight), _ptr(scale), heads, kv_heads, head_dim,
        _ptr(q_norm_w), _ptr(k_norm_w), float(qk_eps), _ptr(positions), _ptr(cos_table), _ptr(sin_table),
        cos_table.shape[0], _ptr(slot_mapping), _ptr(q), _ptr(k_cache), _ptr(v_cache), k_cache.shape[0], _stream(x),
    )
    return q


def lm_head_argmax(
    hidden: Tensor, rows: Tensor, norm_w: Tensor, eps: float, weight: Tensor, prenormed: bool = False
) -> Tensor:
    """Greedy next tokens of the sampled rows: argmax over bf16(RMSNorm(hidden[rows]) @ weight^T)
    with the first index winning ties (model/qwen3.py:152-158 + runner/sampler.py:59); int64 [R].
    ``prenormed``: hidden already holds the final norm's output (no RMSNorm is applied)."""
    _on_gpu(hidden, rows, norm_w, weight)
    _check(hidden.dtype == torch.bfloat16 and hidden.dim() == 2 and hidden.stride(-1) == 1, "lm_head_argmax: hidden")
    _check(rows.dtype == torch.int64 and rows.is_contiguous(), "lm_head_argmax: rows must be int64")
    _check(weight.dtype == torch.bfloat16 and weight.is_contiguous() and weight.shape[1] == hidden.shape[1],
           "lm_head_argmax: weight [vocab, hidden] bf16")
    r = rows.numel()
    vocab, k = weight.shape
    out = torch.empty(r, dtype=torch.int64, device=hidden.device)
    ws_bytes = _native.query("msa_lm_head_argmax_workspace_size", r, k, vocab) if r else 0
    ws = workspaces.get("lm_head", hidden.device, ws_bytes)
    _native.call(
        "msa_lm_head_argmax", _ptr(hidden), hidden.stride(0), hidden.shape[0], _ptr(rows), r, k,
        _ptr(None if prenormed else norm_w),
        float(eps), _ptr(weight),
        vocab, _ptr(out), _ptr(ws), ws.numel() if ws is not None else 0, _stream(hidden),
    )
    return out


def lm_head_logits(
    hidden: Tensor, rows: Tensor, norm_w: Tensor | None, eps: float, weight: Tensor, prenormed: bool = False
) -> Tensor:
    """Logits of the sampled rows: float32(bf16(RMSNorm(hidden[rows]) @ weight^T)) -- the reference's
    ``compute_logits`` on the final norm's rows (model/qwen3.py:152-158); float32 [R, vocab].
    ``prenormed``: hidden already holds the final norm's output (no RMSNorm is applied)."""
    _on_gpu(hidden, rows, weight)
    _check(hidden.dtype == torch.bfloat16 and hidden.dim() == 2 and hidden.stride(-1) == 1, "lm_head_logits: hidden")
    _check(rows.dtype == torch.int64 and rows.is_contiguous(), "lm_head_logits: rows must be int64")
    _check(weight.dtype == torch.bfloat16 and weight.is_contiguous() and weight.shape[1] == hidden.shape[1],
           "lm_head_logits: weight [vocab, hidden] bf16")
    _check(prenormed or norm_w is not None, "lm_head_logits: norm_w required unless prenormed")
    r = rows.numel()
    vocab, k = weight.shape
    out = torch.empty(r, vocab, dtype=torch.float32, device=hidden.device)
    ws_bytes = _native.query("msa_lm_head_logits_workspace_size", r, k, vocab) if r else 0
    ws = workspaces.get("lm_head", hidden.device, ws_bytes)
    _native.call(
        "msa_lm_head_logits", _ptr(hidden), hidden.stride(0), hidden.shape[0], _ptr(rows), r, k,
        _ptr(None if prenormed else norm_w), float(eps), _ptr(weight), vocab, _ptr(out), out.stride(0),
        _ptr(ws), ws.numel() if ws is not None else 0, _stream(hidden),
    )
    return out


# ---- sampling ---------------------------------------------------------------------------------------

# Rows without top-k or top-p take the two launches that spread them over vocabulary chunks from this
# vocabulary on (64 rows of 3072: 17.9 us by a workgroup each, 19.1 spread; of 4096: 20.5, 19.5); with
# top-p from the smallest (1 x 64: 34, 24).
SAMPLE_WIDE_MIN_VOCAB = 4096


def _rows_f32(logits: Tensor, name: str) -> Tensor:
    _check(logits.dtype == torch.float32 and logits.dim() == 2 and logits.stride(-1) == 1, f"{name}: float32 [R, V] logits")
    return logits


def _opt_param(t: Tensor | None, dtype: torch.dtype, rows: int, name: str) -> Tensor | None:
    if t is None:
        return None
    _check(t.dtype == dtype and t.is_contiguous() and t.numel() == rows and t.is_cuda, f"{name}: [{rows}] {dtype}")
    return t


def top_k_top_p_mask(logits: Tensor, top_k: Tensor | None, top_p: Tensor | None) -> Tensor:
    """logits where inside each row's top-k and top-p nucleus, -inf elsewhere (runner/sampler.py:12-27)."""
    _on_gpu(logits)
    _rows_f32(logits, "top_k_top_p_mask")
    r, v = logits.shape
    out = torch.empty_like(logits, memory_format=torch.contiguous_format)
    _native.call("msa_top_k_top_p_mask", _ptr(logits), logits.stride(0), r, v,
                 _ptr(_opt_param(top_k, torch.int32, r, "top_k")), _ptr(_opt_param(top_p, torch.float32, r, "top_p")),
                 _ptr(out), out.stride(0), _stream(logits))
    return out


def sampling_probs(logits: Tensor, temperature: Tensor | None, top_k: Tensor | None, top_p: Tensor | None) -> Tensor:
    """softmax(top-k / top-p of logits / temperature) per row (runner/sampler.py:30-40)."""
    _on_gpu(logits)
    _rows_f32(logits, "sampling_probs")
    r, v = logits.shape
    out = torch.empty_like(logits, memory_format=torch.contiguous_format)
    _native.call("msa_sampling_probs", _ptr(logits), logits.stride(0), r, v,
                 _ptr(_opt_param(temperature, torch.float32, r, "temperature")),
                 _ptr(_opt_param(top_k, torch.int32, r, "top_k")), _ptr(_opt_param(top_p, torch.float32, r, "top_p")),
                 _ptr(out), out.stride(0), _stream(logits))
    return out


def sample_ids(
    logits: Tensor,
    temperature: Tensor | None,
    top_k: Tensor | None,
    top_p: Tensor | None,
    greedy: Tensor | None,
    noise: Tensor | None,
    wide: bool | None = None,
) -> Tensor:
    """Token id per row: the greedy argmax where ``greedy``, else argmax(probs / noise) with the
    probabilities of ``sampling_probs`` (runner/sampler.py:55-69). ``noise`` [R, V] float32 ~ Exp(1);
    it may be None only when every row is greedy. ``wide``: spread the rows without top-k over vocabulary
    chunks, in two more launches; else such a row is served by one workgroup (the same ids either way).
    By default only where ``top_k`` is None, so that no row has it."""
    _on_gpu(logits)
    _rows_f32(logits, "sample_ids")
    r, v = logits.shape
    if noise is None:
        _check(greedy is not None, "sample_ids: noise is required for sampled rows")
        noise = logits  # never read: every row is greedy
        wide = False
    if wide is None:
        wide = top_k is None and (top_p is not None or v >= SAMPLE_WIDE_MIN_VOCAB)
    _check(noise.dtype == torch.float32 and noise.dim() == 2 and noise.shape == (r, v) and noise.stride(-1) == 1,
           "sample_ids: noise [R, V] float32")
    out = torch.empty(r, dtype=torch.int64, device=logits.device)
    temps = _opt_param(temperature, torch.float32, r, "temperature")
    tk = _opt_param(top_k, torch.int32, r, "top_k")
    tp = _opt_param(top_p, torch.float32, r, "top_p")
    gr = _opt_param(greedy, torch.uint8, r, "greedy")
    # Greedy rows, rows with 0 < top_k <= 256 and, with wide, rows without top-k run over vocabulary chunks
    # (the workspace holds each chunk's candidates); the others take a workgroup per row in the same call.
    ws_bytes = _native.query("msa_sample_workspace_size", r, v)
    ws = workspaces.get("sample", logits.device, ws_bytes)
    _native.call("msa_sample_wide" if wide else "msa_sample", _ptr(logits), logits.stride(0), r, v, _ptr(temps),
                 _ptr(tk), _ptr(tp), _ptr(gr), _ptr(noise), noise.stride(0), _ptr(out), _ptr(ws),
                 ws.numel() if ws is not None else 0, _stream(logits))
    return out


# ---- speculative-decoding verification --------------------------------------------------------------


def _i64(t: Tensor, shape: tuple[int, ...], name: str) -> Tensor:
    _check(t.is_cuda and t.dtype == torch.int64 and tuple(t.shape) == shape, f"{name}: int64 {list(shape)}")
    return t.contiguous()


def verify_greedy_ids(target_ids: Tensor, drafts: Tensor, num_drafts: Tensor) -> tuple[Tensor, Tensor]:
    """(accepted [B], next_token [B]) from the target's argmax ids [B, K+1] (spec/rejection.py:27-40)."""
    _on_gpu(target_ids, drafts, num_drafts)
    b, k1 = target_ids.shape
    ids = _i64(target_ids, (b, k1), "target_ids")
    dr = _i64(drafts, (b, k1 - 1), "drafts")
    nd = _i64(num_drafts, (b,), "num_drafts")
    accepted = torch.empty(b, dtype=torch.int64, device=ids.device)
    nxt = torch.empty_like(accepted)
    _native.call("msa_verify_greedy", _ptr(ids), b, k1 - 1, _ptr(dr), _ptr(nd), _ptr(accepted), _ptr(nxt), _stream(ids))
    return accepted, nxt


def verify_sampled(
    target_probs: Tensor, drafts: Tensor, num_drafts: Tensor, draft_probs: Tensor | None, uniform: Tensor, noise: Tensor
) -> tuple[Tensor, Tensor]:
    """(accepted [B], next_token [B]) by rejection sampling (spec/rejection.py:43-79)."""
    _on_gpu(target_probs, drafts, num_drafts, uniform, noise)
    b, k1, v = target_probs.shape
    k = k1 - 1
    _check(k >= 1, "verify_sampled: at least one draft position")
    tp = target_probs.float().contiguous()
    dp = None
    if draft_probs is not None:
        _check(tuple(draft_probs.shape) == (b, k, v), "verify_sampled: draft_probs [B, K, V]")
        dp = draft_probs.float().contiguous()
    _check(tuple(uniform.shape) == (b, k) and tuple(noise.shape) == (b, v), "verify_sampled: uniform [B, K], noise [B, V]")
    # Every converted operand is held by a local until the launch is queued: a temporary passed
    # straight to _ptr would return its memory to the caching allocator first, and the next
    # conversion could be given (and overwrite) that block before the kernel reads it.
    dr = _i64(drafts, (b, k), "drafts")
    nd = _i64(num_drafts, (b,), "num_drafts")
    un = uniform.float().contiguous()
    nz = noise.float().contiguous()
    accepted = torch.empty(b, dtype=torch.int64, device=tp.device)
    nxt = torch.empty_like(accepted)
    _native.call("msa_verify_sampled", _ptr(tp), b, k, v, _ptr(dr), _ptr(nd), _ptr(dp), _ptr(un), _ptr(nz),
                 _ptr(accepted), _ptr(nxt), _stream(tp))
    return accepted, nxt
