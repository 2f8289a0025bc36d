"""Operator-level mirror of the reference's kernel entry points, backed by the HIP library.

Same names, argument meaning and error behaviour as
``fourier_attn_triton/fourier_triton_valid4_v2.py``:

* ``mat_fourier_triton``            (lines 81-102)
* ``mat_avg_std_triton``            (lines 433-461)
* ``mat_fourier_avg_std_triton``    (lines 285-326)
* ``triton_fourier_attn``           (lines 684-779)  - also exported as ``fourier_attn``
* ``mat_fourier_inv_torch``         (lines 782-791)  - as ``mat_fourier_inv``
* ``MultiDimHiPPO2``                (lines 840-865)

The names keep the reference's ``_triton`` suffix so call sites need no edit; nothing
here uses Triton.  Tensors must live on the GPU; PyTorch only provides the memory and
the current stream.
"""
from __future__ import annotations

from typing import Dict, Optional, Tuple

import torch
from torch.autograd.forward_ad import unpack_dual

from . import _lib
from ._lib import FA_BF16, FA_FP16, FA_FP32, check

_DTYPE_CODE = {torch.bfloat16: FA_BF16, torch.float16: FA_FP16, torch.float32: FA_FP32}


def dtype_code(dt: torch.dtype) -> int:
    try:
        return _DTYPE_CODE[dt]
    except KeyError:
        raise TypeError(f"unsupported dtype {dt}; expected bfloat16, float16 or float32") from None


def _current_raw_stream(index: int) -> int:
    return torch.cuda.current_stream(index).cuda_stream


# device index -> handle of torch's current stream there (the bare handle where torch offers it, without building a
# torch.cuda.Stream object around it)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or _current_raw_stream


def _stream(device) -> int:
    """Handle of the stream the caller's tensor work is queued on (torch's current stream of ``device``).  Looked up
    on every call: the caller may switch streams, or capture into a graph, between two operators."""
    idx = device.index
    return _raw_stream(torch.cuda.current_device() if idx is None else idx)


def _require_gpu(t: torch.Tensor, name: str) -> None:
    if not t.is_cuda:
        raise RuntimeError(f"{name} must be a GPU tensor: the HIP kernels are the only implementation")


_workspaces: Dict[Tuple[int, str], torch.Tensor] = {}


def workspace(device: torch.device, nbytes: int, tag: str = "default") -> torch.Tensor:
    """A per-device scratch buffer that only grows.  Work that shares a tag must be issued on
    one stream (kernels of consecutive calls then run in order and may reuse it)."""
    key = (device.index if device.index is not None else torch.cuda.current_device(), tag)
    buf = _workspaces.get(key)
    if buf is None or buf.numel() < nbytes:
        buf = torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=device)
        _workspaces[key] = buf
    return buf


def _ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None or t.numel() == 0 else t.data_ptr()


def as_i32(t: torch.Tensor) -> torch.Tensor:
    return t if t.dtype == torch.int32 else t.to(torch.int32)


# --------------------------------------------------------------------------- K1
def mat_fourier(a: torch.Tensor, N: int, T: int, K_start: int = 0, cols: Optional[torch.Tensor] = None,
                out: Optional[torch.Tensor] = None, accumulate: bool = False, K: Optional[int] = None,
                matrix_cores: bool = True) -> torch.Tensor:
    """``c[b, n, m] (+)= sum_k cos(2 pi (k + K_start) n / T) a[b, k, cols[m]]`` and the sin rows.

    ``a (B, K, width)`` may be a strided view as long as its last dim is contiguous; ``cols``
    (int32, GPU) selects columns; ``K`` limits the rows read.  Long 16-bit inputs run on the matrix
    cores (fp16 basis, fp32 accumulation) unless ``matrix_cores`` is false."""
    _require_gpu(a, "a")
    assert a.dim() == 3 and a.stride(2) == 1, "a must be (B, K, M) with a contiguous last dim"
    B, rows, width = a.shape
    K = rows if K is None else min(int(K), rows)
    Mc = width if cols is None else cols.numel()
    if out is None:
        assert not accumulate
        out = torch.empty((B, 2 * N, Mc), device=a.device, dtype=torch.float32)
    assert out.is_contiguous() and out.dtype == torch.float32 and tuple(out.shape) == (B, 2 * N, Mc)
    if Mc == 0 or B == 0:
        return out
    lib = _lib.load()
    ws_bytes = int(lib.fa_mat_fourier_workspace_bytes(dtype_code(a.dtype), B, K, Mc, N)) if matrix_cores else 0
    ws = workspace(a.device, ws_bytes, "spectral") if ws_bytes else None
    check(lib.fa_mat_fourier(a.data_ptr(), dtype_code(a.dtype), a.stride(0), a.stride(1), _ptr(cols), out.data_ptr(), B, K,
                             Mc, N, int(T), int(K_start), int(accumulate), _ptr(ws), ws_bytes, _stream(a.device)))
    return out


def mat_fourier_triton(a: torch.Tensor, N: int, T: int, K_start: int = 0) -> torch.Tensor:
    assert a.is_contiguous(), "Matrix A must be contiguous"  # TRI:82
    return mat_fourier(a, N, T, K_start)


# --------------------------------------------------------------------------- K2
def mat_avg_std(a: torch.Tensor, cols: Optional[torch.Tensor] = None, round_dtype: Optional[torch.dtype] = None):
    """fp32 ``(avg, max_dev)`` of the columns of ``a (B, K, width)``, each rounded through
    ``round_dtype`` when given."""
    _require_gpu(a, "a")
    assert a.dim() == 3 and a.stride(2) == 1
    B, K, width = a.shape
    Mc = width if cols is None else cols.numel()
    avg = torch.empty((B, Mc), device=a.device, dtype=torch.float32)
    dev = torch.empty((B, Mc), device=a.device, dtype=torch.float32)
    if Mc == 0 or B == 0:
        return avg, dev
    lib = _lib.load()
    nbytes = lib.fa_stats_workspace_bytes(B, Mc, K)
    ws = workspace(a.device, nbytes)
    rd = FA_FP32 if round_dtype is None else dtype_code(round_dtype)
    check(lib.fa_mat_avg_std(a.data_ptr(), dtype_code(a.dtype), a.stride(0), a.stride(1), _ptr(cols), avg.data_ptr(),
                             dev.data_ptr(), B, K, Mc, rd, ws.data_ptr(), ws.numel(), _stream(a.device)))
    return avg, dev


def mat_avg_std_triton(a: torch.Tensor):
    assert a.is_cuda and a.is_contiguous(), "Input tensor must be a contiguous CUDA tensor"  # TRI:438
    assert a.dim() == 3, "Input tensor must be 3-dimensional"
    return _cast_pair(mat_avg_std(a, round_dtype=a.dtype), a.dtype)  # TRI:461


def _cast_pair(pair, dtype: torch.dtype):
    """Both tensors in ``dtype``, each in memory of its own, in one launch."""
    if dtype == torch.float32:
        return pair
    out = tuple(torch.empty_like(t, dtype=dtype) for t in pair)
    torch._foreach_copy_(out, pair)
    return out


# --------------------------------------------------------------------------- K3
def mat_fourier_avg_std(c: torch.Tensor, K: int, T: int, round_dtype: Optional[torch.dtype] = torch.float16,
                        matrix_cores: bool = True):
    """Mean and maximum deviation, per column, of the signal reconstructed from ``c`` at positions 0..K-1.
    Long reconstructions run on the matrix cores (fp16 operands, fp32 accumulation) unless
    ``matrix_cores`` is false."""
    _require_gpu(c, "c")
    assert c.is_contiguous() and c.dtype == torch.float32 and c.dim() == 3
    B, N2, Mc = c.shape
    avg = torch.empty((B, Mc), device=c.device, dtype=torch.float32)
    dev = torch.empty((B, Mc), device=c.device, dtype=torch.float32)
    if Mc == 0 or B == 0:
        return avg, dev
    lib = _lib.load()
    if matrix_cores:
        nbytes = lib.fa_mat_fourier_avg_std_workspace_bytes(B, N2 // 2, Mc, int(K))
    else:
        nbytes = lib.fa_stats_workspace_bytes(B, Mc, int(K))
    ws = workspace(c.device, nbytes, "spectral")
    rd = FA_FP32 if round_dtype is None else dtype_code(round_dtype)
    check(lib.fa_mat_fourier_avg_std(c.data_ptr(), avg.data_ptr(), dev.data_ptr(), B, N2 // 2, Mc, int(K), int(T), rd,
                                     ws.data_ptr(), int(nbytes), _stream(c.device)))
    return avg, dev


def mat_fourier_avg_std_triton(c: torch.Tensor, K: int, T: int):
    assert c.is_contiguous(), "Matrix C must be contiguous"  # TRI:286
    return _cast_pair(mat_fourier_avg_std(c.float() if c.dtype != torch.float32 else c, K, T, torch.float16), torch.float16)  # TRI:326


def recon_scale(c: torch.Tensor, K: int, T: int, u_avg: torch.Tensor, u_dev: torch.Tensor, dtype: torch.dtype):
    """What a cache of a ``dtype`` model keeps of a compressed tensor's statistics (cache_utils_fourier.py:567, 590), without
    launches of its own: ``(scale, u_avg, avg_d)`` in the types the reference leaves them in - the quotient of the two
    deviations promoted, the mean of the original in ``dtype``, that of the reconstruction in float16 - and the same three as
    the kernels take them, float32 ``(u_avg, avg_d, scale)``.  ``u_avg, u_dev``: ``mat_avg_std(..., round_dtype=dtype)``."""
    _require_gpu(c, "c")
    assert c.is_contiguous() and c.dtype == torch.float32 and c.dim() == 3
    B, N2, Mc = c.shape
    assert all(t.is_contiguous() and t.dtype == torch.float32 and tuple(t.shape) == (B, Mc) for t in (u_avg, u_dev))
    new = lambda dt: torch.empty((B, Mc), device=c.device, dtype=dt)
    avg, scale, avg_h = new(torch.float32), new(torch.float32), new(torch.float16)
    u_avg_m = u_avg if dtype == torch.float32 else new(dtype)
    scale_m = new(torch.float16) if dtype == torch.float16 else scale
    if Mc and B:
        lib = _lib.load()
        nbytes = lib.fa_mat_fourier_avg_std_workspace_bytes(B, N2 // 2, Mc, int(K))
        ws = workspace(c.device, nbytes, "spectral")
        check(lib.fa_recon_scale(c.data_ptr(), u_avg.data_ptr(), u_dev.data_ptr(), avg.data_ptr(), scale.data_ptr(), avg_h.data_ptr(),
                                 u_avg_m.data_ptr(), scale_m.data_ptr(), dtype_code(dtype), B, N2 // 2, Mc, int(K), int(T),
                                 ws.data_ptr(), int(nbytes), _stream(c.device)))
    return scale_m, u_avg_m, avg_h, (u_avg, avg, scale)


# ------------------------------------------------------------------ reconstruction
def mat_fourier_inv(c: torch.Tensor, K: int, T: int, avg_u=None, avg_d=None, scale=None) -> torch.Tensor:
    """``(B, K, Mc)`` fp32 reconstruction (TRI:782-791), optionally through the affine statistics."""
    _require_gpu(c, "c")
    assert c.is_contiguous() and c.dtype == torch.float32 and c.dim() == 3
    B, N2, Mc = c.shape
    r = torch.empty((B, int(K), Mc), device=c.device, dtype=torch.float32)
    if r.numel() == 0:
        return r
    f = lambda t: None if t is None else t.float().contiguous()
    au, ad, sc = f(avg_u), f(avg_d), f(scale)
    check(_lib.load().fa_reconstruct(c.data_ptr(), _ptr(au), _ptr(ad), _ptr(sc), r.data_ptr(), B, N2 // 2, Mc, int(K), int(T),
                                     _stream(c.device)))
    return r


# -------------------------------------------------------------------- rank-1 update
def coeff_update_(c: torch.Tensor, row: torch.Tensor, cols: Optional[torch.Tensor], p: int, T: int) -> torch.Tensor:
    """In place ``c[b, n, j] += cos(2 pi p n / T) row[b, cols[j]]`` (+ sin rows).  ``row (B, width)``
    may be a strided view with a contiguous last dim."""
    _require_gpu(c, "c")
    assert c.is_contiguous() and c.dtype == torch.float32 and c.dim() == 3
    assert row.dim() == 2 and row.stride(1) == 1
    B, N2, Mc = c.shape
    if Mc == 0 or B == 0:
        return c
    check(_lib.load().fa_coeff_update(c.data_ptr(), row.data_ptr(), dtype_code(row.dtype), row.stride(0), _ptr(cols), B,
                                      N2 // 2, Mc, int(p), int(T), _stream(c.device)))
    return c


def stream_update(k_new: torch.Tensor, v_new: torch.Tensor, k_ring: torch.Tensor, v_ring: torch.Tensor, evict_slot: int,
                  write_slot: int, k_coef: torch.Tensor, v_coef: torch.Tensor, kc_list: torch.Tensor, vc_list: torch.Tensor,
                  phase: int, T: int, k_mid, v_mid, mid_pos: int, skip_coef: bool = False) -> None:
    """One streaming step of one layer in one launch (the body of cache_utils_fourier.py:731-748 for K and V):
    the rows in window slot ``evict_slot`` enter the coefficients (rank-1 update at ``phase``) and the page
    stores (at token ``mid_pos``); ``k_new, v_new (B, width)`` are written to window slot ``write_slot``.
    ``k_ring, v_ring (B, slots, width)`` share their strides; ``k_mid, v_mid`` are ``MidStore`` objects.  The new rows
    may also come as the token itself, ``(B, heads, 1, D)`` with the heads side by side.
    ``skip_coef``: leave the coefficients alone; the caller owes them the update (``coeff_update_``, or the
    ``pending`` argument of the layer's next ``decode_attn_raw``) before that window slot is written again."""
    _lib.load_host().stream_update(k_new, v_new, k_ring, v_ring, evict_slot, write_slot, k_coef, v_coef, kc_list, vc_list,
                                   phase, T, k_mid, v_mid, mid_pos, skip_coef)


def append_rows(k: torch.Tensor, v: torch.Tensor, k_dst: torch.Tensor, v_dst: torch.Tensor, pos: int) -> None:
    """Rows of K and V ``(B, rows, width)`` to rows ``pos ..`` of two buffers, in one launch."""
    _lib.load_host().append_rows(k, v, k_dst, v_dst, pos)


def recorded() -> bool:
    """Whether the operations of this thread are recorded or transformed: tracing, a dispatch mode (``make_fx``, fake tensors), a
    ``torch.func`` transform.  What a kernel reads and writes by address is not seen there."""
    return (torch.jit.is_tracing() or torch._C._len_torch_dispatch_stack() > 0
            or torch._C._functorch.peek_interpreter_stack() is not None)


def prompt_rows(k: torch.Tensor, v: torch.Tensor, near: Optional[Tuple[torch.Tensor, torch.Tensor]] = None, first: int = 0,
                last: int = 0, spare: int = 0):
    """The rows of a prompt, ``k, v (B, heads, S, D)``, as token-major ``(B, S, heads*D)`` tensors (the source's own memory
    where its heads lie side by side, else copies) and, in the same launch, into ``near = (k, v)``, ``(B, slots, heads*D)``:
    the first ``first`` rows, the last ``last``, then ``spare`` rows of zeros.  ``None`` where the layout is for tensor
    operations: rows that are no multiples of 16 bytes, other devices, tensors that take part in a graph of gradients or carry a
    tangent, calls that are recorded."""
    B, heads, S, D = k.shape
    es = k.element_size()
    if recorded() or type(k) is not torch.Tensor or type(v) is not torch.Tensor:
        return None
    if (not k.is_cuda or k.device != v.device or k.shape != v.shape or k.dtype != v.dtype or k.dtype not in _DTYPE_CODE
            or k.stride() != v.stride() or k.stride(3) != 1 or k.requires_grad or v.requires_grad or not 0 < B <= 65535 or S == 0
            or any((s * es) % 16 for s in (*k.stride()[:3], D)) or k.data_ptr() % 16 or v.data_ptr() % 16
            or first + last > S or any(unpack_dual(t).tangent is not None for t in (k, v))):
        return None
    if near is not None and any(t.dtype != k.dtype or t.device != k.device or t.stride(2) != 1 or t.stride(1) != heads * D
                                or t.stride(0) != near[0].stride(0) or t.shape[1] < first + last + spare or t.data_ptr() % 16
                                for t in near):
        return None
    out, tok = (k, v), (None, None)
    if heads == 1 or k.stride(1) == D:
        out = tuple(t.permute(0, 2, 1, 3).reshape(B, S, heads * D) for t in (k, v))
        if near is None:
            return out
    else:
        out = tok = tuple(torch.empty((B, S, heads * D), dtype=k.dtype, device=k.device) for _ in (k, v))
    n = (None, None) if near is None else near
    check(_lib.load().fa_prompt_rows(k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(1), k.stride(2), _ptr(tok[0]), _ptr(tok[1]),
                                     _ptr(n[0]), _ptr(n[1]), 0 if near is None else near[0].stride(0), first, last, spare,
                                     dtype_code(k.dtype), B, S, heads, D, _stream(k.device)))
    return out


def add_rmsnorm(h: torch.Tensor, delta: Optional[torch.Tensor], weight: torch.Tensor, eps: float) -> torch.Tensor:
    """``h += delta`` (when given, in place) and ``LlamaRMSNorm`` of the result in one launch
    (modeling_llama_fourier.py:735-750, 87-92).  ``h, delta (..., hidden)`` contiguous."""
    return _lib.load_host().add_rmsnorm(h, delta, weight, eps)


def _rotary_tables(cos: torch.Tensor, sin: torch.Tensor, x: torch.Tensor):
    if cos.shape[0] != x.shape[0]:
        cos, sin = cos.expand(x.shape[0], -1, -1), sin.expand(x.shape[0], -1, -1)
    if cos.dtype != x.dtype or sin.dtype != x.dtype or not (cos.is_contiguous() and sin.is_contiguous()):
        cos, sin = cos.to(x.dtype).contiguous(), sin.to(x.dtype).contiguous()
    return cos, sin


def rope_qk(q: torch.Tensor, k: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, head_dim: int) -> torch.Tensor:
    """Rotary embedding of ``q (B, q_len, Hq*D)`` and ``k (B, q_len, Hkv*D)`` (the projection outputs, possibly
    column slices of one fused projection output); ``cos, sin (B or 1, q_len, D)`` (modeling_llama_fourier.py:213-244).
    ``k`` is rotated in place; the rotated ``q`` is returned densely packed (``q`` itself when it was dense)."""
    cos, sin = _rotary_tables(cos, sin, q)
    return _lib.load_host().rope_qk(q, k, cos, sin, head_dim)


def rope_qk_(q: torch.Tensor, k: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, head_dim: int) -> None:
    """``rope_qk`` in place on densely packed ``q`` and ``k``."""
    assert q.is_contiguous() and k.is_contiguous()
    rope_qk(q, k, cos, sin, head_dim)


def silu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """``silu(gate) * up`` in one launch (modeling_llama_fourier.py:277); ``gate, up (..., cols)`` dense or column
    slices of one fused projection output (rows evenly spaced, the same spacing for both); the result is dense."""
    return _lib.load_host().silu_mul(gate, up)


class WeightStamp:
    """Identity and version of the tensors a derived copy was made from: ``changed()`` once any of them has been
    written in place (``load_state_dict``, an optimizer step) or replaced (``.to()``, re-assignment of ``.data``)."""

    def __init__(self, tensors):
        self._refs = list(tensors)
        self._seen = [(t.data_ptr(), t._version) for t in self._refs]

    def changed(self) -> bool:
        return any((t.data_ptr(), t._version) != s for t, s in zip(self._refs, self._seen))


class PackedLinearWeight:
    """A bias-free ``nn.Linear`` weight ``(n_out, K)`` re-laid for ``linear_packed``: the order in which the matrix
    cores take it, so that a decode step (a handful of rows) streams it in contiguous KiB pieces.  ``sources``: the
    parameters the weight was assembled from; ``stale()`` tells when the copy no longer matches them."""

    def __init__(self, weight: torch.Tensor, sources=None):
        self.stamp = WeightStamp(sources if sources is not None else [weight])
        _require_gpu(weight, "weight")
        assert weight.dim() == 2 and weight.is_contiguous() and weight.dtype in (torch.bfloat16, torch.float16)
        self.n_out, self.k = int(weight.shape[0]), int(weight.shape[1])
        self.dtype = weight.dtype
        self._rows_ok = {}     # row count -> whether the kernel takes it (asked once per count)
        self._norm_ok = {}     # ... and an RMSNorm in front of it
        self.data = torch.empty_like(weight)
        check(_lib.load().fa_linear_pack(weight.data_ptr(), self.data.data_ptr(), self.n_out, self.k, dtype_code(weight.dtype),
                                         _stream(weight.device)))

    def stale(self) -> bool:
        return self.stamp.changed()

    def covers(self, x: torch.Tensor) -> bool:
        if not (x.is_cuda and x.dtype == self.dtype and x.shape[-1] == self.k and x.stride(-1) == 1):
            return False
        rows = x.numel() // max(self.k, 1)
        ok = self._rows_ok.get(rows)
        if ok is None:
            ok = self._rows_ok[rows] = bool(_lib.load().fa_linear_packed_ok(rows, self.k, self.n_out))
        return ok

    def normalises(self, x: torch.Tensor, norm: torch.Tensor) -> bool:
        """Whether ``linear_packed_step`` takes an RMSNorm of the rows of ``x`` into its launch: rows that a workgroup
        normalises for itself, 16-byte aligned like the norm's weight."""
        if (x.data_ptr() | norm.data_ptr()) % 16:
            return False
        rows = x.numel() // max(self.k, 1)
        ok = self._norm_ok.get(rows)
        if ok is None:
            ok = self._norm_ok[rows] = bool(_lib.load().fa_linear_packed_norm_ok(rows, self.k))
        return ok


def linear_packed_step(x: torch.Tensor, w: PackedLinearWeight, norm: Optional[torch.Tensor] = None, eps: float = 0.0,
                       residual: Optional[torch.Tensor] = None, gated: bool = False) -> torch.Tensor:
    """``linear_packed`` with the decoder's elementwise steps in the same launch, rounded where ``add_rmsnorm`` and
    ``silu_mul`` round: ``norm``, the weight of an RMSNorm of the rows of ``x`` in front (``w.normalises(x, norm)``);
    ``residual (..., n_out)``, which the product is added to in place (and which is returned); ``gated``, a weight of gate
    and then up rows (``n_out`` a multiple of 32), ``silu(gate) * up`` is returned (modeling_llama_fourier.py:87-92, 277, 735-750)."""
    return _lib.load_host().linear_packed(x, w.data, w.k, w.n_out, norm, eps, residual, gated)


def rotary_pairs(rows: int, heads: int, head_dim: int, device) -> torch.Tensor:
    """The order of a q/k/v weight's rows that ``linear_packed_qkv`` takes: in the first ``heads`` heads (q and k) eight rows of
    the first half of the head and the eight they turn with side by side, the rest as they are."""
    turned = torch.arange(heads * head_dim, device=device).view(heads, 2, head_dim // 16, 8).transpose(1, 2).reshape(-1)
    return torch.cat([turned, torch.arange(heads * head_dim, rows, device=device)])


def linear_packed_qkv(x: torch.Tensor, w: PackedLinearWeight, norm: Optional[torch.Tensor], eps: float, cos: torch.Tensor,
                      sin: torch.Tensor, num_heads: int, num_kv_heads: int, head_dim: int):
    """q, k and v of a decode step, ``(B, heads, q_len, head_dim)`` views, from ``x (B, q_len, hidden)``: RMSNorm in front
    (``norm``, if given), one pass over the weight (its rows in the order of ``rotary_pairs``), rotary embedding of q and k - what
    ``linear_packed_step`` and ``rope_qk`` do in two launches, with the same results.  ``cos, sin``: as for ``rope_qk``."""
    # (the launch reads the tables in vectors; ``rope_qk`` takes them wherever they lie)
    cos, sin = (t if t.data_ptr() % 16 == 0 else t.clone() for t in _rotary_tables(cos, sin, x))
    return _lib.load_host().linear_packed_qkv(x, w.data, norm, eps, cos, sin, num_heads, num_kv_heads, head_dim)


def linear_packed(x: torch.Tensor, w: PackedLinearWeight) -> torch.Tensor:
    """``F.linear(x, weight)`` for ``x (..., K)`` of at most 16 rows (fp32 accumulation, result in the storage type)
    on the packed weight; rows must be evenly spaced (dense, or slices of wider rows)."""
    return _lib.load_host().linear_packed(x, w.data, w.k, w.n_out)


def prefill_attention_supported(q: torch.Tensor, k: torch.Tensor, head_dim: int) -> bool:
    """Shapes the matrix-core prompt attention covers: 16-bit GPU tensors, heads of 64 or 128 dims, 16-byte rows."""
    return (q.is_cuda and q.dtype in (torch.bfloat16, torch.float16) and k.dtype == q.dtype and head_dim in (64, 128)
            and q.stride(-1) == 1 and k.stride(-1) == 1 and all(s % 8 == 0 for s in q.stride()[:-1])
            and all(s % 8 == 0 for s in k.stride()[:-1]) and q.data_ptr() % 16 == 0 and k.data_ptr() % 16 == 0)


def prefill_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, num_kv_heads: int, sm_scale: float = -1.0,
                      out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Exact causal attention of the prompt pass (modeling_llama_fourier.py:623-633, ``flash_attn_func(q, k, v,
    causal=True)``).  ``q (B, Hq, q_len, D)`` (any strides with a contiguous last dim), ``k, v (B, S, Hkv*D)``
    token-major with common strides; returns ``(B, q_len, Hq, D)`` in the dtype of ``q``.  Query row ``i`` sees keys
    ``0 .. i + S - q_len``."""
    _require_gpu(q, "q")
    B, Hq, q_len, D = q.shape
    S = k.shape[1]
    assert k.shape == v.shape and k.stride() == v.stride() and k.shape[0] == B and k.shape[2] == num_kv_heads * D
    assert prefill_attention_supported(q, k, D) and v.dtype == q.dtype and v.data_ptr() % 16 == 0, \
        "prefill_attention: 16-bit GPU tensors, head_dim 64 or 128, 16-byte aligned rows"
    if out is None:
        out = torch.empty((B, q_len, Hq, D), dtype=q.dtype, device=q.device)
    assert out.is_contiguous() and tuple(out.shape) == (B, q_len, Hq, D) and out.dtype == q.dtype
    lib = _lib.load()
    nbytes = lib.fa_prefill_attn_workspace_bytes(B, num_kv_heads, D, S)
    ws = workspace(q.device, nbytes, "prefill")
    check(lib.fa_prefill_attn(q.data_ptr(), q.stride(0), q.stride(1), q.stride(2), k.data_ptr(), v.data_ptr(), k.stride(0),
                              k.stride(1), out.data_ptr(), dtype_code(q.dtype), B, Hq, num_kv_heads, D, S, q_len,
                              float(sm_scale), ws.data_ptr(), ws.numel(), _stream(q.device)))
    return out


class MultiDimHiPPO2(torch.nn.Module):
    """Same call contract as the reference class (TRI:840-865): without ``slice_input`` the
    whole ``base_input (B, L, C)`` is projected (period and length ``int(1/dt)``: longer inputs
    are cut, shorter ones behave as zero-padded); with ``slice_input (B, 1, C)`` the result is
    ``base_input + transform(slice_input)`` entering at phase ``token_num``."""

    def __init__(self, N, input_dim, method="legt", dt=1.0, T=1.0, discretization="bilinear", scale=False, c=0.0):
        super().__init__()
        self.method, self.N, self.input_dim, self.dt, self.T, self.c = method, N, input_dim, dt, T, c
        self.base_N = N // input_dim

    def forward(self, base_input, token_num, slice_input=None, fast=False):
        base_N = self.N // self.input_dim // 2
        period = int(1 / self.dt)
        if slice_input is not None:
            out = base_input.clone()
            return coeff_update_(out, slice_input[:, 0, :], None, token_num, period)
        return mat_fourier(base_input, base_N, period, 0, K=period)


# ------------------------------------------------------------------ decode attention
def decode_tables(n_f: int, period: int, device) -> Optional[torch.Tensor]:
    """Constant operand tables of the MFMA decode path for ``(N, T)``; ``None`` when that path
    does not cover ``N`` (the call then takes the generic kernels)."""
    lib = _lib.load()
    nbytes = lib.fa_decode_tables_bytes(int(n_f))
    if nbytes == 0 or n_f not in (128, 256, 512, 1024):
        return None
    buf = torch.empty(nbytes, dtype=torch.uint8, device=device)
    check(lib.fa_decode_tables_build(buf.data_ptr(), nbytes, int(n_f), int(period), _stream(torch.device(device))))
    return buf


def decode_attn_raw(q, il_segments, k_mc, v_mc, k_mn, v_mn, stats_k, stats_v, lists, num_head_q, num_head_kv, seq_len_m,
                    T, sm_scale=-1.0, out=None, tables=None, force_generic=False, timings=None, out_dtype=None,
                    no_alloc=False, balance_heads=True, no_fuse=0, pending=None, step=None):
    """Thin call into ``fa_decode_attn``.  The result is float32 like the reference's (TRI:779) unless ``out_dtype``
    names the dtype of ``q``: then the merge launch rounds it to that type itself (the caller's ``.to(dtype)``).

    ``q (B, 1, Hq*D)`` or ``(B, Hq, 1, D)``, contiguous.
    ``il_segments``: up to two ``(k, v)`` pairs of ``(B, rows, Hkv*D)`` views (last dim contiguous), or ``(k, v, r)``: the
    rows of one buffer in front of and behind row ``r``.
    ``k_mn`` / ``v_mn``: token-major ``(B, >=L_m, Cn)`` tensors or ``MidStore`` objects (paged).
    ``stats_*``: ``(avg_u, avg_d, scale)`` fp32 ``(B, C)``.  ``lists``: the eight int32 tensors
    ``kc, kc_h, kn, kn_h, vc, vc_h, vn, vn_h`` (``*_h`` with the leading 0).
    ``no_alloc``: call ``fa_decode_attn_noalloc`` (partial results in the library's own fixed buffer, no workspace
    tensor; pass ``out`` as well and nothing is allocated on the device at all).
    ``balance_heads``: hand the per-head padded dim counts of a paged store over on the host side too, so that heads
    that store more dims get more splits (``False``: every head the same number, for comparison).
    ``no_fuse``: keep the sink/window tiles, the mid rows and the merge as launches of their own where the library
    would run them as one (for comparison); an int is passed on as the bits of ``fa_decode_args.no_fuse`` (2: fused,
    but without the four sub-splits per workgroup that a batch of one sequence otherwise runs).
    ``pending``: ``(k_row, v_row, phase, T_c)``, a rank-1 update the coefficients are still owed (``stream_update``
    with ``skip_coef``): ``k_row, v_row (B, Hkv*D)`` are the rows that left the window (same strides).  The call
    applies it to ``k_mc`` / ``v_mc`` IN PLACE while it streams them, once; pass it to one call only.
    ``step``: the arguments of ``stream_update`` as a tuple: that update, then the attention over the state it leaves
    (which the other arguments describe), in one launch less where the shapes allow it.  In a list of their own they are
    taken out of it when the update is launched: what raises before leaves them there."""
    if seq_len_m >= _REPACK_MIN_ROWS and not force_generic:
        _warn_if_off_the_matrix_cores(q.dtype, num_head_q, num_head_kv, q.numel() // (q.shape[0] * num_head_q),
                                      (k_mc if lists[0].numel() else v_mc).shape[1] // 2, not isinstance(k_mn, torch.Tensor))
    cast = out_dtype is not None and out_dtype != torch.float32
    assert not cast or out_dtype == q.dtype, "out_dtype must be float32 or the dtype of q"
    return _lib.load_host().decode_attn(q, il_segments, k_mc, v_mc, k_mn, v_mn, stats_k, stats_v, lists, num_head_q,
                                        num_head_kv, seq_len_m, T, sm_scale, out, cast, tables, force_generic, balance_heads,
                                        no_fuse, pending, no_alloc, timings, step)


_warned_shapes = set()
_SIXTEEN_BIT = (torch.bfloat16, torch.float16)


def _warn_if_off_the_matrix_cores(dtype, num_head_q, num_head_kv, head_dim, n_f, paged):
    """Long contexts outside the shapes of the matrix-core kernels (16-bit paged storage, 128 / 256 / 512 / 1024
    frequencies, heads of at most 128 dims, at most 8 query heads per KV head) run on vector-ALU kernels that take any
    shape and are slower (one sequence of 32k 167 us a layer against 41, eight 954 / 110, four of 128k 3373 / 320): say so once
    per shape instead of being silently slow."""
    if (dtype in _SIXTEEN_BIT and paged and n_f in (128, 256, 512, 1024) and head_dim <= 128
            and num_head_q // max(num_head_kv, 1) <= 8):
        return
    key = (dtype, num_head_q, num_head_kv, head_dim, n_f, paged)
    if key in _warned_shapes:
        return
    _warned_shapes.add(key)
    import warnings
    warnings.warn(
        f"fourier decode attention: dtype={dtype}, {num_head_q}/{num_head_kv} heads of {head_dim} dims, {n_f} frequencies, "
        f"{'paged' if paged else 'token-major'} mid rows run on the any-shape vector kernels, 3 to 11 times slower than the "
        "matrix-core kernels (16-bit paged storage, 128/256/512/1024 frequencies, head_dim <= 128, <= 8 query heads per KV head)",
        RuntimeWarning, stacklevel=3)


def triton_fourier_attn(q, k_il, v_il, k_mc, v_mc, k_mn, v_mn,
                        avg_k_u, avg_k_d, scale_k, avg_v_u, avg_v_d, scale_v,
                        kc_list, kc_h_list, kn_list, kn_h_list,
                        vc_list, vc_h_list, vn_list, vn_h_list,
                        num_head_q, num_head_kv, seq_len_m, T, sm_scale=-1):
    """Drop-in for the reference function of the same name (TRI:684-779): returns
    ``(B, Hq, 1, D)`` float32."""
    batch_size, seq_len_q, feature_dim = q.shape
    assert seq_len_q == 1, f"{q.shape = }"  # TRI:692
    _require_gpu(q, "q")
    k_mc = k_mc if k_mc.dtype == torch.float32 else k_mc.float()
    v_mc = v_mc if v_mc.dtype == torch.float32 else v_mc.float()
    repage = _repage_worthwhile(q, k_mn, k_mc if kc_list.numel() else v_mc, num_head_q, num_head_kv, int(seq_len_m))
    lists, stats, paging = _lib.load_host().operands(
        (kc_list, kc_h_list, kn_list, kn_h_list, vc_list, vc_h_list, vn_list, vn_h_list),
        (avg_k_u, avg_k_d, scale_k, avg_v_u, avg_v_d, scale_v),
        _lib.K_DIM_PAD if repage else 0, _lib.V_DIM_PAD if repage else 0)
    if repage:
        k_mn = _repaged(k_mn, lists[3], paging[0], paging[2], num_head_kv, q.shape[2] // num_head_q, int(seq_len_m), False)
        v_mn = _repaged(v_mn, lists[7], paging[1], paging[3], num_head_kv, q.shape[2] // num_head_q, int(seq_len_m), True)
    return decode_attn_raw(q.contiguous(), [(k_il, v_il)], k_mc.contiguous(), v_mc.contiguous(), k_mn, v_mn,
                           stats[:3], stats[3:], lists, num_head_q, num_head_kv, seq_len_m, T, sm_scale)


# below this many mid rows the any-layout kernels are quicker than re-paging first
_REPACK_MIN_ROWS = 2048


def _repage_worthwhile(q, k_mn, coef, num_head_q, num_head_kv, seq_len_m) -> bool:
    """The reference hands ``k_mn`` / ``v_mn`` over token-major (``torch.cat`` of gathered columns,
    cache_utils_fourier.py:735, 741).  The matrix-core kernels stream pages; for long contexts copying the
    rows into a temporary page store first (two passes over them) and taking those kernels is several times
    faster than the kernels that read the token-major layout in place.  ``DynamicCache`` keeps its rows paged
    and never comes through here."""
    from .midstore import MidStore
    if isinstance(k_mn, MidStore) or seq_len_m < _REPACK_MIN_ROWS or q.dtype not in _SIXTEEN_BIT:
        return False
    D = q.shape[2] // num_head_q
    return coef.shape[1] // 2 in (128, 256, 512, 1024) and D <= 128 and num_head_q // num_head_kv <= 8 and k_mn.dtype == q.dtype


def _repaged(t, n_h32, n_h_host, pad_h32, num_head_kv, head_dim, rows, is_v):
    """A page store of the first ``rows`` rows of ``t``, whose columns are the stored dims in order."""
    from .midstore import MidStore
    st = MidStore(t.shape[0], None, n_h32, n_h_host, num_head_kv, head_dim, rows, t.dtype, t.device, is_v, pad_h32=pad_h32,
                  zeroed=False)
    st.pack(t, 0, rows, in_order=True)
    return st


fourier_attn = triton_fourier_attn
