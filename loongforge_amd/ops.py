"""Tensor-level entry points of the gfx950 DSA kernels.

Every function here checks its arguments, allocates outputs and workspaces with torch (the C
library allocates nothing), and calls libdsa_hip.so on the current HIP stream; the hot ones do all of that
in C++ (csrc/host/host.cpp), the others here through ctypes.
The raw kernels are also registered as torch custom ops in the ``dsa::`` namespace so that they
can be used from compiled graphs and carry fake-tensor shape functions.

There is no CPU path and no fallback: tensors must live on a HIP device.
"""
import os
from typing import Optional, Tuple

import torch

from . import _lib

_FP8 = torch.float8_e4m3fn


_host = None


def _native():
    """The C++ host layer: checks, allocations and kernel calls (csrc/host/host.cpp)."""
    global _host
    if _host is None:
        _host = _lib.load_host()
    return _host


def _direct(name: str, op, *args):
    """``op(*args)``, called in C++ without the custom-op dispatcher when this is an ordinary eager call on ordinary
    tensors (the native function returns None otherwise: fake or traced tensors, dispatch modes, recorded gradients)."""
    if not torch.compiler.is_compiling():
        res = getattr(_native(), name)(*args, False)
        if res is not None:
            return res
    return op(*args)


def ordinary(*tensors) -> bool:
    """Whether this is an eager call on ordinary tensors, which kernels may take past the dispatcher: not compiled or traced, no
    functorch transform, forward-mode level or dispatch mode, no batched, fake or otherwise dispatched tensor."""
    if torch.compiler.is_compiling() or torch.jit.is_tracing():
        return False
    if torch._C._are_functorch_transforms_active() or torch.autograd.forward_ad._current_level >= 0:
        return False
    return _native().ordinary(tensors)


def _stream(t: torch.Tensor):
    return torch.cuda.current_stream(t.device).cuda_stream


def _need_gpu(*tensors):
    tensors = [t for t in tensors if t is not None]
    for t in tensors:
        if not t.is_cuda:
            raise RuntimeError("DSA kernels need tensors on a HIP device; got a %s tensor" % t.device.type)
        if t.device != tensors[0].device:
            raise RuntimeError("DSA kernels need tensors on one device; got %s and %s" % (tensors[0].device, t.device))


def _c(t: torch.Tensor) -> torch.Tensor:
    return t if t.is_contiguous() else t.contiguous()


# --------------------------------------------------------------------------------------------
# quantiser
# --------------------------------------------------------------------------------------------
@torch.library.custom_op("dsa::quant_rowwise_e4m3", mutates_args=())
def _quant_op(x: torch.Tensor, eps: float, pow2: bool) -> Tuple[torch.Tensor, torch.Tensor]:
    return _native().quant_rowwise(x, eps, pow2, True)


@_quant_op.register_fake
def _(x, eps, pow2):
    return x.new_empty(x.shape, dtype=torch.uint8), x.new_empty(x.shape[:-1], dtype=torch.float32)


def quant_rowwise_e4m3(x: torch.Tensor, eps: float = 1e-12, pow2: bool = True):
    """bf16 ``[..., 128]`` -> (float8_e4m3fn payload, fp32 ``scale_inv`` per row)."""
    x8, scale_inv = _direct("quant_rowwise", _quant_op, x, eps, pow2)
    return _fp8(x8), scale_inv


@torch.library.custom_op("dsa::rotate_quant_e4m3", mutates_args=())
def _rotate_quant_op(x: torch.Tensor, eps: float, pow2: bool, want_payload: bool,
                     want_rotated: bool) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    return _native().rotate_quant(x, eps, pow2, want_payload, want_rotated, True)


@_rotate_quant_op.register_fake
def _(x, eps, pow2, want_payload, want_rotated):
    return (x.new_empty(x.shape if want_payload else (0,), dtype=torch.uint8),
            x.new_empty(x.shape[:-1] if want_payload else (0,), dtype=torch.float32),
            x.new_empty(x.shape if want_rotated else (0,), dtype=torch.bfloat16))


def rotate_quant_e4m3(x: torch.Tensor, eps: float = 1e-12, pow2: bool = True, return_rotated: bool = False):
    """Hadamard rotation (x 128^-0.5, rounded to bf16) fused with :func:`quant_rowwise_e4m3`:
    bf16 ``[..., 128]`` -> (fp8 payload, ``scale_inv``[, rotated bf16])."""
    x8, scale_inv, y = _direct("rotate_quant", _rotate_quant_op, x, eps, pow2, True, return_rotated)
    return (_fp8(x8), scale_inv, y) if return_rotated else (_fp8(x8), scale_inv)


@torch.library.custom_op("dsa::indexer_front_e4m3", mutates_args=())
def _indexer_front_op(x: torch.Tensor, rows_per_token: int, ln_weight: Optional[torch.Tensor],
                      ln_bias: Optional[torch.Tensor], ln_eps: float, cos: Optional[torch.Tensor],
                      sin: Optional[torch.Tensor], pairing: int, positions: Optional[torch.Tensor], batch: int,
                      rotate: bool, weights: Optional[torch.Tensor], factor: float, want_payload: bool,
                      want_rows: bool, eps: float,
                      pow2: bool) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    return _native().indexer_front(x, rows_per_token, ln_weight, ln_bias, ln_eps, cos, sin, pairing, positions, batch, rotate,
                                   weights, factor, want_payload, want_rows, eps, pow2, True)


@_indexer_front_op.register_fake
def _(x, rows_per_token, ln_weight, ln_bias, ln_eps, cos, sin, pairing, positions, batch, rotate, weights, factor,
      want_payload, want_rows, eps, pow2):
    return (x.new_empty(x.shape if want_payload else (0,), dtype=torch.uint8),
            x.new_empty(x.shape[:-1] if want_payload else (0,), dtype=torch.float32),
            x.new_empty(x.shape if want_rows else (0,), dtype=torch.bfloat16),
            x.new_empty(x.shape[:-1] if weights is not None else (0,), dtype=torch.float32))


def indexer_front_e4m3(x: torch.Tensor, rows_per_token: int = 1, ln_weight=None, ln_bias=None, ln_eps: float = 1e-5,
                       cos=None, sin=None, pairing: int = -1, positions=None, batch: int = 1, rotate: bool = True,
                       weights=None, factor: float = 1.0, return_payload: bool = True, return_rows: bool = False,
                       eps: float = 1e-12, pow2: bool = True):
    """The indexer front end behind its projections in one kernel: bf16 ``[..., 128]`` rows through
    [LayerNorm] -> [RoPE of the leading 64 elements, ``pairing`` ROPE_ADJACENT / ROPE_SPLIT, -1 none] ->
    [Hadamard rotation] -> quantiser.  Returns ``(x8, scale_inv, rows, weight_scaled)``; ``rows`` (the bf16
    values that were quantised) and ``weight_scaled`` (``weights * scale_inv * factor``) are ``None`` unless
    asked for."""
    x8, scale_inv, y, ws = _direct("indexer_front", _indexer_front_op, x, rows_per_token, ln_weight, ln_bias, ln_eps, cos, sin, pairing,
                                   positions, batch, rotate, weights, float(factor), return_payload, return_rows, eps, pow2)
    return (_fp8(x8) if return_payload else None, scale_inv if return_payload else None,
            y if return_rows else None, ws if weights is not None else None)


@torch.library.custom_op("dsa::quant_rowwise_e4m3_weights", mutates_args=())
def _quant_weights_op(x: torch.Tensor, weights: torch.Tensor, factor: float, rotate: bool, eps: float,
                      pow2: bool) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    return _native().quant_weights(x, weights, factor, rotate, eps, pow2, True)


@_quant_weights_op.register_fake
def _(x, weights, factor, rotate, eps, pow2):
    return (x.new_empty(x.shape, dtype=torch.uint8), x.new_empty(x.shape[:-1], dtype=torch.float32),
            x.new_empty(x.shape[:-1], dtype=torch.float32))


def quant_rowwise_e4m3_weights(x: torch.Tensor, weights: torch.Tensor, factor: float, rotate: bool = False,
                               eps: float = 1e-12, pow2: bool = True):
    """:func:`quant_rowwise_e4m3` (after the Hadamard rotation when ``rotate``) that also returns
    ``(weights * scale_inv) * factor`` per row: (fp8 payload, ``scale_inv``, scaled weights fp32)."""
    x8, scale_inv, w_scaled = _direct("quant_weights", _quant_weights_op, x, weights, float(factor), bool(rotate), eps, pow2)
    return _fp8(x8), scale_inv, w_scaled


def rotate_bf16(x: torch.Tensor):
    """Hadamard rotation of bf16 rows of 128 (x 128^-0.5), the kernel form of ``rotate_activation``."""
    return _direct("rotate_quant", _rotate_quant_op, x, 1e-12, True, False, True)[2]


def quant_padded_e4m3(x, heads: int, weights=None, factor: float = 1.0):
    """:func:`quant_rowwise_e4m3_weights` of ``x [tokens, heads_in, dim]`` padded with zeros to ``[tokens, heads, 128]``, the
    padding done on the way: (fp8 payload, ``scale_inv``, scaled weights or None)."""
    return _native().quant_padded(x, int(heads), weights, float(factor))


# --------------------------------------------------------------------------------------------
# separate operations of the indexer's front end
# --------------------------------------------------------------------------------------------
def rotary_angles(inv_freq, n: int, offset: float = 0.0):
    """``[n, 1, 1, dim]`` angles ``(i + offset) * inv_freq`` (twice side by side), one kernel; None for arguments it does not take
    (other tensors, a length that is no integer, an offset on the device or one per position)."""
    if not isinstance(n, int) or not isinstance(offset, (int, float)):
        return None
    return _native().rotary_angles(inv_freq, n, float(offset))


def rotary_cos_sin(inv_freq, n: int, offset: float, dtype):
    """Cosines and sines of :func:`rotary_angles` in ``dtype`` (fp32 or bf16), one kernel; None for arguments it does not take."""
    if not isinstance(n, int) or not isinstance(offset, (int, float)):
        return None
    return _native().rotary_cos_sin(inv_freq, n, float(offset), dtype)


class _RopeSteps(torch.autograd.Function):
    @staticmethod
    def forward(ctx, t, angles, mscale, interleaved, transpose):
        ctx.save_for_backward(angles)
        ctx.args = (mscale, interleaved, not transpose)
        return _native().rope_steps(t, angles, mscale, interleaved, transpose)

    @staticmethod
    def backward(ctx, grad):
        return rope_steps(grad, ctx.saved_tensors[0], *ctx.args), None, None, None, None


def rope_steps(t, angles, mscale: float = 1.0, interleaved: bool = False, transpose: bool = False):
    """``t * cos + rotate_half(t) * sin`` for bf16 ``t [s, (b,) h, d]`` and fp32 ``angles [>= s, 1, 1, d]``, with the rounding of
    the separate bf16 operations, or the transpose of that map; differentiable in ``t`` any number of times.
    ``interleaved``: the pairs of ``t`` are adjacent elements.  Tensors that are not :func:`ordinary` (a batched gradient, for
    instance) take the separate operations."""
    if ordinary(t, angles):
        return _RopeSteps.apply(t, angles, float(mscale), bool(interleaved), bool(transpose))
    half = t.shape[-1] // 2
    f = angles[:t.shape[0]].reshape(t.shape[0], *([1] * (t.ndim - 2)), angles.shape[-1])
    cos, sin = (torch.cos(f) * mscale).to(t.dtype), (torch.sin(f) * mscale).to(t.dtype)
    if transpose:
        u = t * sin
        y = t * cos + torch.cat((u[..., half:], -u[..., :half]), dim=-1)
        return torch.stack((y[..., :half], y[..., half:]), dim=-1).reshape(t.shape) if interleaved else y
    if interleaved:
        t = torch.cat((t[..., 0::2], t[..., 1::2]), dim=-1)
    return t * cos + torch.cat((-t[..., half:], t[..., :half]), dim=-1) * sin


HADAMARD_SIZES = (32, 64, 128, 256, 512)


class _Hadamard(torch.autograd.Function):
    """The rotation is symmetric: its transpose is itself."""

    @staticmethod
    def forward(ctx, x):
        return _native().hadamard(x)

    @staticmethod
    def backward(ctx, grad):
        from .dsa_fused import rotate_activation      # this kernel, or tensor operations for what it does not take

        return rotate_activation(grad.to(torch.bfloat16))


def hadamard(x):
    """bf16 rows of 32 .. 512 elements (an :func:`ordinary` tensor) times the Hadamard matrix and ``n ** -0.5``; differentiable
    any number of times."""
    return _Hadamard.apply(x)


def _fp8(t: torch.Tensor) -> torch.Tensor:
    return t if t.dtype == _FP8 else t.view(_FP8)


def _as_u8(t: torch.Tensor) -> torch.Tensor:
    if t.dtype == _FP8:
        return t.view(torch.uint8)
    if t.dtype != torch.uint8:
        raise ValueError("expected an fp8-e4m3 (or raw uint8) tensor, got %s" % t.dtype)
    return t


# --------------------------------------------------------------------------------------------
# indexer forward
# --------------------------------------------------------------------------------------------
def _check_indexer(q8, q_w, k8, k_scale, ks, ke):
    _need_gpu(q8, q_w, k8, k_scale, ks, ke)
    if q8.ndim != 3 or k8.ndim != 2 or q_w.ndim != 2:
        raise ValueError("indexer expects q8 [S,H,128], k8 [Sk,128], q_w [S,H]")
    S, Hi, D = q8.shape
    if D != 128 or k8.shape[1] != 128:
        raise ValueError("Only support dim with size 128.")
    if q_w.shape != (S, Hi) or k_scale.shape != (k8.shape[0],) or ks.shape != (S,) or ke.shape != (S,):
        raise ValueError("indexer: inconsistent shapes")
    return S, Hi, k8.shape[0]


@torch.library.custom_op("dsa::indexer_logits", mutates_args=())
def _indexer_logits_op(q8: torch.Tensor, q_w: torch.Tensor, k8: torch.Tensor, k_scale: torch.Tensor,
                       ks: torch.Tensor, ke: torch.Tensor, width: int, relative: bool) -> torch.Tensor:
    S, Hi, Sk = _check_indexer(q8, q_w, k8, k_scale, ks, ke)
    q8, k8 = _c(_as_u8(q8)), _c(_as_u8(k8))
    q_w, k_scale = _c(q_w.float()), _c(k_scale.float())
    ks, ke = _c(ks.int()), _c(ke.int())
    logits = torch.empty(S, width, dtype=torch.float32, device=q8.device)
    lib = _lib.load()
    with torch.cuda.device(q8.device):
        _lib.check(lib.dsa_indexer_logits(q8.data_ptr(), q_w.data_ptr(), k8.data_ptr(), k_scale.data_ptr(),
                                          ks.data_ptr(), ke.data_ptr(), S, Hi, Sk, logits.data_ptr(), width, width,
                                          int(relative), _stream(q8)), "dsa_indexer_logits")
    return logits


@_indexer_logits_op.register_fake
def _(q8, q_w, k8, k_scale, ks, ke, width, relative):
    return q_w.new_empty(q8.shape[0], width, dtype=torch.float32)


def indexer_logits(q8, q_w, k8, k_scale, ks, ke, width: Optional[int] = None, relative: bool = False):
    """Dense ``[S, width]`` fp32 logits, -inf outside ``[ks, ke)`` (column ``j - ks`` if relative)."""
    return _indexer_logits_op(q8, q_w, k8, k_scale, ks, ke, int(width if width is not None else k8.shape[0]),
                              bool(relative))


@torch.library.custom_op("dsa::topk", mutates_args=())
def _topk_op(logits: torch.Tensor, K: int, row_begin: Optional[torch.Tensor], row_end: Optional[torch.Tensor],
             id_base: Optional[torch.Tensor], sort: bool) -> Tuple[torch.Tensor, torch.Tensor]:
    return _native().topk(logits, K, row_begin, row_end, id_base, sort, True)


@_topk_op.register_fake
def _(logits, K, row_begin, row_end, id_base, sort):
    return logits.new_empty(logits.shape[0], K), logits.new_empty(logits.shape[0], K, dtype=torch.int32)


def topk(logits, K: int, row_begin=None, row_end=None, id_base=None, sorted: bool = True):
    """Per-row top-K (scores, int32 ids); unused slots are (-inf, -1)."""
    return _direct("topk", _topk_op, logits, int(K), row_begin, row_end, id_base, bool(sorted))


@torch.library.custom_op("dsa::indexer_topk", mutates_args=())
def _indexer_topk_op(q8: torch.Tensor, q_w: torch.Tensor, k8: torch.Tensor, k_scale: torch.Tensor, ks: torch.Tensor,
                     ke: torch.Tensor, K: int, sort: bool) -> Tuple[torch.Tensor, torch.Tensor]:
    return _native().indexer_topk(q8, q_w, k8, k_scale, ks, ke, K, sort, True)


@_indexer_topk_op.register_fake
def _(q8, q_w, k8, k_scale, ks, ke, K, sort):
    return q_w.new_empty(q8.shape[0], K, dtype=torch.float32), q_w.new_empty(q8.shape[0], K, dtype=torch.int32)


def indexer_topk(q8, q_w, k8, k_scale, ks, ke, K: int, sorted: bool = True):
    """Fused logits + top-K: (scores [S,K] fp32, global key ids [S,K] int32, -1 padded)."""
    return _direct("indexer_topk", _indexer_topk_op, q8, q_w, k8, k_scale, ks, ke, int(K), bool(sorted))


@torch.library.custom_op("dsa::indexer_bwd", mutates_args=())
def _indexer_bwd_op(g: torch.Tensor, q8: torch.Tensor, k8: torch.Tensor, k_scale: torch.Tensor, q_w: torch.Tensor,
                    ids: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    return _native().indexer_bwd(g, q8, k8, k_scale, q_w, ids, True)


@_indexer_bwd_op.register_fake
def _(g, q8, k8, k_scale, q_w, ids):
    return (q_w.new_empty(q8.shape, dtype=torch.float32), q_w.new_empty(k8.shape, dtype=torch.float32),
            q_w.new_empty(q_w.shape, dtype=torch.float32))


def indexer_bwd(g, q8, k8, k_scale, q_w, ids):
    """Gradients of the selected logits w.r.t. the fp8 payloads and the scaled weights (fp32)."""
    return _direct("indexer_bwd", _indexer_bwd_op, g, q8, k8, k_scale, q_w, ids)


def indexer_grads(g, q8, k8, k_scale, q_w, ids, q_scale, w_scale: float, heads: int, dim: int, dtypes, rotate: bool = False,
                  front=None, k_in=None, ln_weight=None, span: int = 0, narrow=None):
    """:func:`indexer_bwd` carried on to the outputs of the projections: ``(d_q [S, heads, dim], d_k [Sk, dim], d_weights
    [S, heads], d_ln_weight, d_ln_bias)`` in ``dtypes`` (of q, k, weights), the last two fp32 or None.  Unscaled (rows on the
    quantiser's epsilon floor, loongforge/models/foundation/deepseek_v4/deepseek_v4_csa.py:1525-1541, get zero), back
    through the Hadamard rotation if ``rotate``, and with ``front`` (an ``IndexerFrontEnd``) through the rotary embedding
    and the LayerNorm of the keys (input ``k_in``, weight ``ln_weight``).  ``span``: the most neighbouring keys that a query
    sees, 0 if that is not known (-1, -2: by rows, by key tiles); it decides how the keys' gradients are summed, not what they are.
    ``narrow``: the ``(cos, sin)`` of :func:`indexer_forward_narrow`."""
    f = front
    if narrow is not None:
        if not ordinary(g, q8, k8, k_scale, q_w, ids, q_scale, *narrow):
            return _indexer_grads_narrow(g, q8, k8, k_scale, q_w, ids, q_scale, w_scale, heads, dim, dtypes, *narrow)
        return _native().indexer_grads(g, q8, k8, k_scale, q_w, ids, q_scale, float(w_scale), 2, *narrow, ROPE_SPLIT, None, None, 1, None, None,
                                       0.0, int(heads), int(dim), int(span), *dtypes)
    if f is None and not ordinary(g, q8, k8, k_scale, q_w, ids, q_scale):
        return _indexer_grads_composed(g, q8, k8, k_scale, q_w, ids, q_scale, w_scale, heads, dim, dtypes, rotate)
    return _native().indexer_grads(g, q8, k8, k_scale, q_w, ids, q_scale, float(w_scale), bool(rotate), f and f.cos, f and f.sin,
                                   f.pairing if f else -1, f and f.positions_q, f and f.positions_k, f.batch if f else 1,
                                   k_in, ln_weight, f.k_norm_eps if f else 0.0, int(heads), int(dim), int(span), *dtypes)


def _indexer_grads_composed(g, q8, k8, k_scale, q_w, ids, q_scale, w_scale, heads, dim, dtypes, rotate):
    """:func:`indexer_grads` without a front end as the custom op and tensor operations, for traced and fake tensors."""
    from .dsa_fused import _hadamard
    from .dsa_fused_kernels import _unscale_indexer_grad

    g = torch.where(ids >= 0, g.float(), torch.zeros_like(g, dtype=torch.float32))
    d_q, d_k, d_w = indexer_bwd(g.contiguous(), q8, k8, k_scale, q_w, ids.int())
    d_w, d_q, d_k = d_w * q_scale * w_scale, _unscale_indexer_grad(d_q, q_scale), _unscale_indexer_grad(d_k, k_scale)
    if rotate:
        h = _hadamard(128, d_q.device, torch.float32)
        d_q, d_k = (d_q @ h) * 128 ** -0.5, (d_k @ h) * 128 ** -0.5
    return d_q[:, :heads, :dim].to(dtypes[0]), d_k[:, :dim].to(dtypes[1]), d_w[:, :heads].to(dtypes[2]), None, None


def _indexer_grads_narrow(g, q8, k8, k_scale, q_w, ids, q_scale, w_scale, heads, dim, dtypes, cos, sin):
    """:func:`indexer_grads` of :func:`indexer_forward_narrow` as tensor operations, for traced and batched tensors."""
    from .dsa_fused import _hadamard

    d_q, d_k, d_w, _, _ = _indexer_grads_composed(g, q8, k8, k_scale, q_w, ids, q_scale, w_scale, heads, dim,
                                                  (torch.float32, torch.float32, dtypes[2]), False)

    def back(d, dtype, c, s):
        d = ((d @ _hadamard(dim, d.device, torch.float32)) * dim ** -0.5).to(torch.bfloat16)
        u, half = d.float() * s, dim // 2
        return (d.float() * c + torch.cat((u[..., half:], -u[..., :half]), dim=-1)).to(dtype)

    c, s = cos.reshape(-1, dim).float(), sin.reshape(-1, dim).float()
    S, Sk = q8.shape[0], k8.shape[0]
    return back(d_q, dtypes[0], c[:S, None], s[:S, None]), back(d_k, dtypes[1], c[:Sk], s[:Sk]), d_w, None, None


class _Unchecked:
    def wait(self):
        pass


def indexer_window(cu_seqlens: Optional[torch.Tensor], queries: int, chunk_offset: int, like: torch.Tensor):
    """``(ks, ke, check)``: the key window of every causal query ``chunk_offset + i`` (int32, on ``like``'s device) over
    the packed sequences of ``cu_seqlens`` (None: one sequence).  ``check.wait()`` raises ValueError if the sequences
    end before the queries do, or their cumulative lengths decrease; call it behind the launches that use the window.
    While a HIP graph is captured nothing can be checked; in any case a query behind the last sequence has an empty window
    (no keys, ids -1)."""
    if not ordinary(cu_seqlens, like):
        dev = like.device
        ke = torch.arange(queries, dtype=torch.int32, device=dev) + chunk_offset + 1
        if cu_seqlens is None:
            return torch.zeros(queries, dtype=torch.int32, device=dev), ke, _Unchecked()
        cu = cu_seqlens.to(dev)
        lens = cu[1:] - cu[:-1]
        seq = torch.repeat_interleave(torch.arange(len(lens), device=dev, dtype=torch.int32), lens)
        return cu[seq[chunk_offset:chunk_offset + queries].long()].int(), ke, _Unchecked()
    return _native().indexer_window(cu_seqlens, int(queries), int(chunk_offset), like)


def indexer_forward(index_q, index_k, weights, rotate: bool, factor: float, cu_seqlens, chunk_offset: int, K: int, sorted: bool, front=None,
                    ln_weight=None, ln_bias=None, ratio: int = 0, weights_scale: float = 1.0):
    """Quantisers (with ``front``, an ``IndexerFrontEnd``, behind the front end), :func:`indexer_window` and :func:`indexer_topk` of bf16
    ``index_q [S, 32 or 64, 128]`` and ``index_k [Sk, 128]`` in one native call: (scores, ids, q8, q_scale, scaled weights, k8,
    k_scale, check or None); None for other arguments and for calls that are not eager ones on ordinary tensors.  ``ratio`` > 0: one
    sequence, query ``i`` sees the first ``(chunk_offset + i + 1) // ratio`` keys, at least one.  ``weights_scale`` (with ``front``): the
    weights count times this, rounded to their type."""
    if torch.compiler.is_compiling():
        return None
    f = front
    return _native().indexer_forward(index_q, index_k, weights, bool(rotate), float(factor), cu_seqlens, int(chunk_offset), int(K), bool(sorted),
                                     f and f.cos, f and f.sin, f.pairing if f else -1, f and f.positions_q, f and f.positions_k,
                                     f.batch if f else 1, ln_weight, ln_bias, f.k_norm_eps if f else 0.0, int(ratio), float(weights_scale))


def indexer_forward_narrow(index_q, index_k, weights, cos, sin, factor: float, chunk_offset: int, K: int, sorted: bool,
                           weights_scale: float = 1.0):
    """:func:`indexer_forward` over one sequence for bf16 ``index_q [S, <= 64, 64]`` and ``index_k [Sk, 64]`` that still need their
    rotary embedding (bf16 ``cos`` / ``sin [positions, .., 64]``, every channel rotary, split pairs, rounded like
    :func:`rope_steps`) and their Hadamard rotation: (scores, ids, q8, q_scale, scaled weights, k8, k_scale), padded to
    32 or 64 heads of 128; None for arguments it does not take."""
    return _native().indexer_forward_narrow(index_q, index_k, weights, cos, sin, float(weights_scale), float(factor), int(chunk_offset), int(K),
                                            bool(sorted))


# --------------------------------------------------------------------------------------------
# sparse MLA
# --------------------------------------------------------------------------------------------
@torch.library.custom_op("dsa::sparse_mla_fwd", mutates_args=())
def _mla_fwd_op(q: torch.Tensor, kv: torch.Tensor, ids: torch.Tensor, q_start: int, sm_scale: float, d_v: int,
                p_out_mode: int, attn_sink: Optional[torch.Tensor] = None,
                p_out_skip: int = 0) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    return _native().mla_fwd(q, kv, ids, q_start, sm_scale, d_v, p_out_mode, attn_sink, p_out_skip, True)


@_mla_fwd_op.register_fake
def _(q, kv, ids, q_start, sm_scale, d_v, p_out_mode, attn_sink=None, p_out_skip=0):
    S, H, _ = q.shape
    p = q.new_empty(0) if p_out_mode == 0 else q.new_empty(S, H, ids.shape[1] - p_out_skip, dtype=torch.float32 if p_out_mode == 2 else torch.bfloat16)
    return q.new_empty(S, H, d_v), q.new_empty(S, H, dtype=torch.float32), p


def sparse_mla_fwd(q, kv, ids, q_start: int = 0, sm_scale: Optional[float] = None, d_v: int = 512,
                   return_p_out: bool = False, p_out_dtype: torch.dtype = torch.bfloat16,
                   attn_sink: Optional[torch.Tensor] = None, p_out_skip: int = 0):
    """(out bf16 [S,H,d_v], natural-log lse fp32 [S,H], p_out or None).  ``attn_sink`` [H]: per-head
    sink logit added to the softmax denominator (and to lse).  ``p_out_skip``: p_out leaves out that
    many leading slots (a multiple of 32) and is [S,H,K - p_out_skip]."""
    if sm_scale is None:
        sm_scale = q.shape[-1] ** -0.5
    mode = 0 if not return_p_out else (2 if p_out_dtype == torch.float32 else 1)
    out, lse, p_out = _direct("mla_fwd", _mla_fwd_op, q, kv, ids, int(q_start), float(sm_scale), int(d_v), mode, attn_sink,
                              int(p_out_skip) if return_p_out else 0)
    return out, lse, (p_out if return_p_out else None)


@torch.library.custom_op("dsa::sparse_mla_fwd_dist", mutates_args=())
def _mla_fwd_dist_op(q: torch.Tensor, kv: torch.Tensor, ids: torch.Tensor, q_start: int, sm_scale: float, d_v: int,
                     dist_heads: int, block: int, attn_sink: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    return _native().mla_fwd_dist(q, kv, ids, q_start, sm_scale, d_v, dist_heads, block, attn_sink, True)


@_mla_fwd_dist_op.register_fake
def _(q, kv, ids, q_start, sm_scale, d_v, dist_heads, block, attn_sink=None):
    S, H, _ = q.shape
    return q.new_empty(S, H, d_v), q.new_empty(S, H, dtype=torch.float32), q.new_empty(S, ids.shape[1], dtype=torch.float32)


def sparse_mla_fwd_dist(q, kv, ids, q_start: int, sm_scale: float, d_v: int, dist_heads: int, block: int,
                        attn_sink: Optional[torch.Tensor] = None):
    """(out, lse, dist): the forward together with the head-averaged attention distribution over the first
    ``dist_heads`` heads (``attn_dist`` of the forward's raw logits), ``block`` queries at a time, so that the logits
    ``[block, H, K]`` are a passing buffer whatever the number of queries (a block's forward writes them, the
    reduction reads them back while they are still in the caches).  Every block is worked on as the whole would be: the
    results are those of :func:`sparse_mla_fwd` and :func:`attn_dist` on all queries, bit for bit.  Tiles of 32 slots without a valid
    one are neither written nor read."""
    return _direct("mla_fwd_dist", _mla_fwd_dist_op, q, kv, ids, int(q_start), float(sm_scale), int(d_v), int(dist_heads), int(block),
                   attn_sink)


_BWD_WS = {}      # device index -> workspace kept between calls; its `stream` is the one it was allocated and used on
BWD_MAX_SLOTS = 2048      # slots per query the backward kernels take in one call
ATTN_DIST_QK_MAX_SLOTS = 4096


def _bwd_workspace(full_bytes: int, device, stream: Optional[int] = None, capturing: bool = False):
    """Workspace of the sparse-MLA backward: ``full_bytes`` lets it take all queries in one sweep (22 GiB at 8k
    tokens, top-k 2048; 89 GiB at 32k); given less, the library walks the queries in chunks.  The size handed to
    the library - and with it the chunking, on which the last bits of dKV depend (those of dQ do not) - follows from the shapes and
    from ``DSA_BWD_WORKSPACE_GIB`` (default 48) alone, never from what happens to be free or from earlier calls.
    The buffer is kept per device and reused by later calls on the same stream (held until :func:`release_bwd_workspace`;
    ``DSA_BWD_WORKSPACE_CACHE=0`` keeps none).  A call on another stream, which may overlap, lets go of it - the allocator
    hands it out again behind the work of its own stream only - and allocates one there.  A graph that is being captured gets
    one of its own, which lives as long as the graph.  ``stream`` (and whether it is ``capturing``): from a caller that knows it."""
    want = max(int(full_bytes), 256)
    cap = os.environ.get("DSA_BWD_WORKSPACE_GIB", "48")
    want = min(want, max(int(float(cap) * 2 ** 30), 256))
    idx = device.index if device.index is not None else torch.cuda.current_device()
    if stream is None:
        capturing, stream = torch.cuda.is_current_stream_capturing(), torch.cuda.current_stream(device).cuda_stream
    if not capturing:
        kept = _BWD_WS.get(idx)
        if kept is not None and kept.numel() >= want and kept.stream == stream:
            return kept, want
        _BWD_WS.pop(idx, None)
        del kept
    try:
        ws = torch.empty(want, dtype=torch.uint8, device=device)
    except torch.OutOfMemoryError as e:
        raise RuntimeError("sparse_mla_bwd: cannot allocate its %.1f GiB workspace; lower DSA_BWD_WORKSPACE_GIB "
                           "(the library then walks the queries in more chunks)" % (want / 2 ** 30)) from e
    if os.environ.get("DSA_BWD_WORKSPACE_CACHE", "1") != "0" and not capturing:
        ws.stream = stream
        _BWD_WS[idx] = ws
    return ws, want


def release_bwd_workspace(device=None):
    """Drops the backward workspace kept for ``device`` (all devices if None)."""
    if device is None:
        _BWD_WS.clear()
    else:
        d = torch.device(device)
        _BWD_WS.pop(d.index if d.index is not None else torch.cuda.current_device(), None)


@torch.library.custom_op("dsa::sparse_mla_bwd", mutates_args=())
def _mla_bwd_op(q: torch.Tensor, kv: torch.Tensor, out: torch.Tensor, dout: torch.Tensor, ids: torch.Tensor,
                lse: torch.Tensor, q_start: int, sm_scale: float, d_v: int) -> Tuple[torch.Tensor, torch.Tensor]:
    return _native().mla_bwd(q, kv, out, dout, ids, lse, q_start, sm_scale, d_v, 0, _bwd_workspace, True)


@_mla_bwd_op.register_fake
def _(q, kv, out, dout, ids, lse, q_start, sm_scale, d_v):
    return torch.empty_like(q), torch.empty_like(kv)


def _mla_bwd(q, kv, out, dout, ids, lse, q_start, sm_scale, d_v, heads):
    if not torch.compiler.is_compiling():
        res = _native().mla_bwd(q, kv, out, dout, ids, lse, q_start, sm_scale, d_v, heads, _bwd_workspace, False)
        if res is not None:
            return res
    if not 0 < heads < q.shape[1]:
        return _mla_bwd_op(q, kv, out, dout, ids, lse, q_start, sm_scale, d_v)
    dq, dkv = _mla_bwd_op(q, kv, out, pad_heads(dout, q.shape[1]), ids, lse, q_start, sm_scale, d_v)
    return dq[:, :heads].contiguous(), dkv


def pad_heads(x, heads: int):
    """``x [S, h, width]`` with zero heads behind its own, ``heads`` in all."""
    padded = None if torch.compiler.is_compiling() else _native().pad_heads(x, int(heads))
    return torch.nn.functional.pad(x, (0, 0, 0, heads - x.shape[1])) if padded is None else padded


def sparse_mla_bwd(q, kv, out, dout, ids, lse, q_start: int = 0, sm_scale: Optional[float] = None, d_v: int = 512, heads: int = 0):
    """(dq, dkv) in bf16; dkv is accumulated in a fixed order (bit-reproducible).  ``heads`` > 0: only that many leading heads of ``q``
    are real and the rest padding; ``dout`` has the real ones, and so has dq.

    The kernels take up to 2048 slots per query.  Longer lists are walked 2048 slots at a time: with the
    softmax statistics (``lse``) and ``out`` of the whole list given, the gradients are sums over the slots, so the
    parts add up (in fp32 here; an id that a query holds in two different parts is not detected)."""
    if sm_scale is None:
        sm_scale = q.shape[-1] ** -0.5
    K = ids.shape[1]
    if K <= BWD_MAX_SLOTS:
        return _mla_bwd(q, kv, out, dout, ids, lse, int(q_start), float(sm_scale), int(d_v), int(heads))
    dq32 = dkv32 = None
    for k0 in range(0, K, BWD_MAX_SLOTS):
        part = ids[:, k0:k0 + BWD_MAX_SLOTS]
        if part.shape[1] % 64:
            part = torch.nn.functional.pad(part, (0, 64 - part.shape[1] % 64), value=-1)
        dq, dkv = _mla_bwd(q, kv, out, dout, part.contiguous(), lse, int(q_start), float(sm_scale), int(d_v), int(heads))
        dq32 = dq.float() if dq32 is None else dq32.add_(dq)
        dkv32 = dkv.float() if dkv32 is None else dkv32.add_(dkv)
    return dq32.to(torch.bfloat16), dkv32.to(torch.bfloat16)


@torch.library.custom_op("dsa::attn_dist", mutates_args=())
def _attn_dist_op(p_out: torch.Tensor, sm_scale: float) -> torch.Tensor:
    return _native().attn_dist(p_out, sm_scale, True)


@_attn_dist_op.register_fake
def _(p_out, sm_scale):
    return p_out.new_empty(p_out.shape[0], p_out.shape[2], dtype=torch.float32)


def attn_dist(p_out, sm_scale: float):
    """fp32 ``[S,K]``: mean over heads of softmax over slots of ``p_out * sm_scale``."""
    return _direct("attn_dist", _attn_dist_op, p_out, float(sm_scale))


def attn_dist_as_input(p_out, sm_scale: float):
    """:func:`attn_dist` in ``p_out.dtype``."""
    return _direct("attn_dist_as_input", lambda *a: _attn_dist_op(*a).to(p_out.dtype), p_out, float(sm_scale))


@torch.library.custom_op("dsa::attn_dist_qk", mutates_args=())
def _attn_dist_qk_op(q: torch.Tensor, kv: torch.Tensor, ids: torch.Tensor, lse: torch.Tensor, q_start: int,
                     sm_scale: float, heads_in_mean: int) -> torch.Tensor:
    _need_gpu(q, kv, ids, lse)
    if q.ndim != 3 or q.shape[-1] != 576 or q.dtype != torch.bfloat16:
        raise ValueError("attn_dist_qk expects q [S,H,576] in bf16")
    if kv.ndim != 2 or kv.shape[-1] != 576 or kv.dtype != torch.bfloat16:
        raise ValueError("attn_dist_qk expects kv [Skv,576] in bf16")
    S, H, _ = q.shape
    K = ids.shape[1]
    if ids.shape[0] != S or lse.shape != (S, H):
        raise ValueError("attn_dist_qk: ids [S,K] and lse [S,H] must match q")
    q, kv, ids, lse = _c(q), _c(kv), _c(ids.to(torch.int32)), _c(lse.float())
    target = torch.empty(S, K, dtype=torch.float32, device=q.device)
    lib = _lib.load()
    with torch.cuda.device(q.device):
        _lib.check(lib.dsa_attn_dist_qk(q.data_ptr(), kv.data_ptr(), ids.data_ptr(), lse.data_ptr(), S, H, int(heads_in_mean),
                                        kv.shape[0], K, int(q_start), float(sm_scale), target.data_ptr(), _stream(q)),
                   "dsa_attn_dist_qk")
    return target


@_attn_dist_qk_op.register_fake
def _(q, kv, ids, lse, q_start, sm_scale, heads_in_mean):
    return q.new_empty(q.shape[0], ids.shape[1], dtype=torch.float32)


def attn_dist_qk(q, kv, ids, lse, q_start: int, sm_scale: float, heads_in_mean: Optional[int] = None,
                 attn_sink: Optional[torch.Tensor] = None):
    """fp32 ``[S,K]``: the same distribution as ``attn_dist(p_out, sm_scale)`` - mean over the first
    ``heads_in_mean`` heads of the softmax over slots - recomputed from q, kv and the forward's
    natural-log ``lse`` instead of from materialised logits.  With an attention sink the forward's
    lse includes the sink term; the softmax over the slots alone has the log-sum-exp
    ``lse + log(1 - exp(sink - lse))``, which is what the kernel is given then."""
    if attn_sink is not None:
        lse = lse + torch.log1p(-torch.exp(attn_sink.to(lse.dtype).view(1, -1) - lse).clamp(max=1.0 - 1e-7))
    hm = int(heads_in_mean or q.shape[1])
    K = ids.shape[1]
    if K <= ATTN_DIST_QK_MAX_SLOTS:
        return _attn_dist_qk_op(q, kv, ids, lse, int(q_start), float(sm_scale), hm)
    # the kernel takes up to 4096 slots; with lse given every slot's value stands alone, so longer lists go in parts
    parts = []
    for k0 in range(0, K, ATTN_DIST_QK_MAX_SLOTS):
        part = ids[:, k0:k0 + ATTN_DIST_QK_MAX_SLOTS]
        n = part.shape[1]
        if n % 64:
            part = torch.nn.functional.pad(part, (0, 64 - n % 64), value=-1)
        parts.append(_attn_dist_qk_op(q, kv, part.contiguous(), lse, int(q_start), float(sm_scale), hm)[:, :n])
    return torch.cat(parts, dim=1)


# --------------------------------------------------------------------------------------------
# rotary position embedding fused with the surrounding copies
# --------------------------------------------------------------------------------------------
ROPE_ADJACENT, ROPE_SPLIT = 0, 1   # where pair i sits in a row: (2i, 2i+1) or (i, i + emb_dim/2)


@torch.library.custom_op("dsa::indexer_kl_loss", mutates_args=())
def _kl_loss_op(scores: torch.Tensor, target: torch.Tensor, eps: float) -> Tuple[torch.Tensor, torch.Tensor]:
    return _native().kl_loss(scores, target, eps, True)


@_kl_loss_op.register_fake
def _(scores, target, eps):
    return scores.new_empty(scores.shape[0], dtype=torch.float32), scores.new_empty(scores.shape, dtype=torch.float32)


def _scaled_kl_gradient(grad, g, factor: float):
    """``grad * (g * factor)``, one launch where nothing records or traces it; never ``grad`` itself, which a hook may write to."""
    if not torch.is_grad_enabled() and not torch.compiler.is_compiling() and ordinary(grad, g):
        scaled = _native().kl_scale(grad, g, factor)
        if scaled is not None:
            return scaled
    return grad * (g * factor)


class _IndexerKLLoss(torch.autograd.Function):
    """The loss and its gradient come out of the same kernel; backward only scales what forward kept."""

    @staticmethod
    def forward(ctx, scores, target, eps, factor):
        row_loss, grad = _direct("kl_loss", _kl_loss_op, scores.detach(), target.detach(), eps)
        ctx.save_for_backward(grad)
        ctx.in_dtype, ctx.factor = scores.dtype, factor
        total = None if torch.compiler.is_compiling() else _native().kl_total(row_loss, factor)
        return row_loss.sum() * factor if total is None else total

    @staticmethod
    def backward(ctx, g):
        (grad,) = ctx.saved_tensors
        return _scaled_kl_gradient(grad, g, ctx.factor).to(ctx.in_dtype), None, None, None


def indexer_kl_loss(scores: torch.Tensor, target: torch.Tensor, eps: float = 1e-10, factor: float = 1.0) -> torch.Tensor:
    """``F.kl_div((softmax(scores, -1) + eps).log(), target + eps, reduction="sum")`` as one kernel
    (dsa_fused.py:931-937 of the reference), times ``factor``; differentiable in ``scores``, the target is a constant."""
    return _IndexerKLLoss.apply(scores, target, float(eps), float(factor))


class _AttachedKLLoss(torch.autograd.Function):
    """:class:`_IndexerKLLoss` and the auto-scaler that feeds its backward, in one node (a node and a fill less)."""

    @staticmethod
    def forward(ctx, output, scores, target, eps, factor, scaler):
        loss, grad = _native().kl_loss_total(scores.detach(), target.detach(), eps, factor)
        ctx.save_for_backward(grad)
        ctx.in_dtype, ctx.factor, ctx.scaler = scores.dtype, factor, scaler
        ctx.mark_non_differentiable(loss)
        ctx.set_materialize_grads(False)
        return output, loss

    @staticmethod
    def backward(ctx, grad_output, _):
        d_scores, scale = None, ctx.scaler.main_loss_backward_scale
        if ctx.needs_input_grad[1]:
            (grad,) = ctx.saved_tensors
            if scale is None:
                d_scores = grad * ctx.factor
            else:
                g = scale.to(grad.device).to(torch.float32)
                d_scores = _scaled_kl_gradient(grad, g.reshape(()) if g.numel() == 1 else g.sum(), ctx.factor)
            d_scores = d_scores.to(ctx.in_dtype)
        return grad_output, d_scores, None, None, None, None


def attached_indexer_kl_loss(output, scores: torch.Tensor, target: torch.Tensor, eps: float, factor: float, scaler):
    """``(output, loss)``: the loss of :func:`indexer_kl_loss`, detached, and ``output`` with it attached as ``scaler`` (the class
    with the loss's ``main_loss_backward_scale``) attaches an auxiliary loss; for :func:`ordinary` tensors."""
    return _AttachedKLLoss.apply(output, scores, target, float(eps), float(factor), scaler)


def _rows_view(t: torch.Tensor, what: str):
    """(data_ptr, token stride, head stride) of a [tokens, heads, width] bf16 view with unit inner stride."""
    if t.dtype != torch.bfloat16 or t.ndim != 3 or (t.shape[-1] > 1 and t.stride(-1) != 1):
        raise ValueError("%s must be a bf16 [tokens, heads, width] view with unit inner stride" % what)
    return t.data_ptr(), t.stride(0), t.stride(1)


def _cos_sin(cos: torch.Tensor, sin: torch.Tensor, emb_dim: int):
    cos2, sin2 = cos.reshape(-1, emb_dim), sin.reshape(-1, emb_dim)
    if cos2.dtype not in (torch.float32, torch.bfloat16):
        cos2, sin2 = cos2.float(), sin2.float()
    if sin2.dtype != cos2.dtype:
        sin2 = sin2.to(cos2.dtype)
    return _c(cos2), _c(sin2)


def thd_positions(cu_seqlens: torch.Tensor, tokens: int, offset: int = 0) -> torch.Tensor:
    """Position of every packed token inside its own sequence (int32 [tokens]); token t of the call
    is global token t + offset.  Tokens past the last sequence get position 0."""
    if cu_seqlens.is_cuda and not torch.compiler.is_compiling():
        pos = _native().thd_positions(cu_seqlens, tokens, int(offset))
        if pos is not None:
            return pos
    cu = cu_seqlens.to(torch.int64)
    t = torch.arange(tokens, device=cu.device, dtype=torch.int64) + int(offset)
    seq = torch.searchsorted(cu[1:].contiguous(), t, right=True)
    inside = seq < cu.numel() - 1
    start = cu[seq.clamp(max=cu.numel() - 2)]
    return torch.where(inside, t - start, torch.zeros_like(t)).to(torch.int32)


def rope_rows(pe_src: Optional[torch.Tensor], pe_dst: Optional[torch.Tensor], cos: Optional[torch.Tensor],
              sin: Optional[torch.Tensor], in_pairing: int, out_pairing: int, inverse: bool = False,
              positions: Optional[torch.Tensor] = None, batch: int = 1,
              main_src: Optional[torch.Tensor] = None, main_dst: Optional[torch.Tensor] = None) -> None:
    """Rotates the pe part of every (token, head) row and copies the main part (either may be absent).

    All tensors are [tokens, heads, width] bf16 views (any token / head strides, rows starting on
    16-byte boundaries); ``pe_src`` may be ``pe_dst`` when both pairings are equal; a head stride of 0
    in ``pe_src`` broadcasts one row.  cos / sin: [positions, emb_dim] fp32 or bf16.  Writes in place
    into ``pe_dst`` / ``main_dst``.
    """
    _native().rope_rows(pe_src, pe_dst, cos, sin, int(in_pairing), int(out_pairing), bool(inverse), positions, int(batch),
                        main_src, main_dst)


def rope_headsum_inverse(grad_pe: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, in_pairing: int,
                         positions: Optional[torch.Tensor] = None, batch: int = 1) -> torch.Tensor:
    """d_emb [tokens, emb_dim] bf16 = inverse rotation of bf16(sum over heads of grad_pe [tokens, heads, emb_dim])."""
    _need_gpu(grad_pe, cos, sin, positions)
    g = _rows_view(grad_pe, "grad_pe")
    tokens, heads, emb = grad_pe.shape
    cos2, sin2 = _cos_sin(cos, sin, emb)
    if positions is not None:
        positions = _c(positions.int())
        if positions.numel() != tokens:
            raise ValueError("positions must hold one entry per token")
    elif batch > 0 and -(-tokens // batch) > min(cos2.shape[0], sin2.shape[0]):
        raise ValueError("cos / sin tables are shorter than the sequence")
    d_emb = torch.empty(tokens, emb, dtype=torch.bfloat16, device=grad_pe.device)
    lib = _lib.load()
    with torch.cuda.device(grad_pe.device):
        _lib.check(lib.dsa_rope_headsum_inverse(g[0], g[1], g[2], d_emb.data_ptr(), emb, emb, cos2.data_ptr(), sin2.data_ptr(),
                                                int(cos2.dtype == torch.float32),
                                                positions.data_ptr() if positions is not None else None, int(batch),
                                                tokens, heads, int(in_pairing), _stream(grad_pe)),
                   "dsa_rope_headsum_inverse")
    return d_emb


# --------------------------------------------------------------------------------------------
# MLA weight absorption (per-head projections written in place)
# --------------------------------------------------------------------------------------------
def mla_absorb_into(a: torch.Tensor, w: torch.Tensor, c: torch.Tensor) -> None:
    """``c[s, h, :] = a[s, h, :] @ w[h].T`` for bf16 views ``a [S, H, k]``, ``c [S, H, n]`` (any token / head
    strides that are multiples of 8 elements, unit stride inside a row) and contiguous ``w [H, n, k]`` with
    ``(k, n)`` = (128, 512) or (512, 128).  Writes into ``c``; no autograd (see :class:`MlaAbsorb`)."""
    _native().absorb_into(a, w, c)


def absorb_rope_query_into(q_up: torch.Tensor, w: torch.Tensor, query: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                           out_pairing: int, positions: Optional[torch.Tensor] = None, batch: int = 1) -> None:
    """``query[s, h, :512] = q_up[s, h, :128] @ w[h].T`` and ``query[s, h, 512:] = rope(q_up[s, h, 128:])`` (pairs adjacent
    in ``q_up``), one kernel: :func:`mla_absorb_into` and :func:`rope_rows` over the rows of ``q_up [S, H, 192]`` and
    ``query [S, H, 576]``.  No autograd."""
    _native().absorb_rope_query_into(q_up, w, query, cos, sin, int(out_pairing), positions, int(batch))


def absorbed_query(q_up, w, cos, sin, positions, out_pairing: int):
    """:func:`absorb_rope_query_into` over ``q_up [.., H, 192]`` into a new ``[.., H, 576]``; None if that needs autograd or
    the widths are others."""
    return _native().absorbed_query(q_up, w, cos, sin, positions, int(out_pairing))


def absorbed_key(kv, k_pos_emb, cos, sin, positions, emb_dim: int, packed: bool, out_pairing: int):
    """``cat(kv, rope(k_pos_emb))`` over the heads of ``kv [s, b, h, d]`` (``packed``: ``[t, h, d]``) as a new tensor; None if that needs
    autograd, or for layouts and widths that are looked at one by one elsewhere."""
    return _native().absorbed_key(kv, k_pos_emb, cos, sin, positions, int(emb_dim), bool(packed), int(out_pairing))


def absorb_flat(a, w):
    """:func:`mla_absorb` with heads and width flattened, ``[.., H * n]``; None if that needs autograd."""
    return _native().absorb(a, w, True)


class MlaAbsorb(torch.autograd.Function):
    """``out[s, h, :] = a[s, h, :] @ w[h].T`` through the HIP kernel, written into ``out`` (a view of a larger
    tensor, returned as is and marked dirty), with the two gradient products as plain library GEMMs."""

    @staticmethod
    def forward(ctx, a, w, out):
        mla_absorb_into(a.detach(), w.detach(), out)
        ctx.save_for_backward(a, w)
        ctx.mark_dirty(out)
        return out

    @staticmethod
    def backward(ctx, grad):
        a, w = ctx.saved_tensors
        g = grad.transpose(0, 1)                       # [H, S, n]
        d_a = torch.bmm(g, _c(w)).transpose(0, 1) if ctx.needs_input_grad[0] else None          # [S, H, k]
        # [H, n, k]; the right operand of a batched bf16 product is laid out contiguously: as a transposed view it has faulted
        d_w = torch.bmm(g.transpose(1, 2), a.transpose(0, 1).contiguous()) if ctx.needs_input_grad[1] else None
        return d_a, d_w, None


def mla_absorb(a: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Differentiable per-head projection ``a [S, H, k] , w [H, n, k] -> [S, H, n]``; ``out`` may be a view into
    a larger tensor (for instance the latent columns of the attention query)."""
    if out is None:
        if not torch.compiler.is_compiling():
            res = _native().absorb(a, w, False)
            if res is not None:
                return res
        out = a.new_empty(a.shape[0], a.shape[1], w.shape[1])
    return MlaAbsorb.apply(a, w, out)
