"""The attention block of a full-attention decoder layer over the quantized cache
(``laguna_mlx/laguna.py:75-111``), MI355X side.

``Attention.__call__`` keeps the reference's protocol: projections, q/k RMSNorm, RoPE at
``cache.offset``, ``update_and_fetch``, then ``cache.attend`` on fused steps, quantized attention
over the returned packed K/V when the cache exposes ``bits`` (a ``quantized_decode`` step, as
mlx-lm's SDPA routes it), SDPA over the returned K/V otherwise, then the softplus output gate and
``o_proj``. The pieces:

* one GEMM for q, k, v and the gate logits (the four projection weights concatenated), one for
  ``o_proj``: ``lq_gemv_bf16`` for a single row (a decode step), ``lq_gemm_rows_bf16`` for up to
  16 (a verify block), hipBLASLt through torch for more;
* ``lq_qkv_norm_rope``: the projection taken apart, the q and k RMSNorms and the rotary embedding
  of both in one launch
  (frequencies from :func:`rope_frequencies`: mlx-lm's default or YaRN RoPE, partial rotary);
* the cache: the fused decode / verify kernels, or dequantized K/V for the unfused path;
* ``lq_gate_heads_strided``: softplus gate times the attention output, written in ``o_proj``'s layout.

Activations and weights are bf16, as in the reference's MLX model.
"""
from __future__ import annotations

import math

import torch
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

from . import _lib


def rope_frequencies(head_dim: int, params: dict):
    """``(inv_freq fp32 [rot_dims / 2], rot_dims, mscale)`` of mlx-lm's ``initialize_rope`` for a
    rope config (``laguna.py:69-72``): ``rope_theta``, ``partial_rotary_factor`` (rotated dims =
    head_dim x factor), ``rope_type`` "default" or "yarn" (``factor``,
    ``original_max_position_embeddings`` 4096, ``beta_fast`` 32, ``beta_slow`` 1, ``mscale`` 1,
    ``mscale_all_dim`` 0). YaRN (Peng et al. 2023, "YaRN: Efficient Context Window Extension of
    Large Language Models"): dims rotating more than ``beta_fast`` times over the original context
    keep their frequency, those rotating fewer than ``beta_slow`` times are divided by ``factor``,
    a linear ramp in between; the rotated dims are scaled by ``0.1 mscale ln(factor) + 1`` over the
    same with ``mscale_all_dim``."""
    dims = int(head_dim * params.get("partial_rotary_factor", 1.0))
    base = float(params["rope_theta"])
    rtype = params.get("rope_type", params.get("type", "default"))
    idx = torch.arange(0, dims, 2, dtype=torch.float64)
    inv_extra = base ** (-idx / dims)
    if rtype == "default":
        return inv_extra.float(), dims, 1.0
    if rtype != "yarn":
        raise ValueError(f"rope_type {rtype!r} is not supported")
    factor = float(params["factor"])
    orig = float(params.get("original_max_position_embeddings", 4096))
    beta_fast = float(params.get("beta_fast", 32))
    beta_slow = float(params.get("beta_slow", 1))

    def corr_dim(rotations):
        return dims * math.log(orig / (rotations * 2 * math.pi)) / (2 * math.log(base))

    low = max(math.floor(corr_dim(beta_fast)), 0)
    high = min(math.ceil(corr_dim(beta_slow)), dims - 1)
    if low == high:
        high += 0.001
    ramp = ((torch.arange(dims // 2, dtype=torch.float64) - low) / (high - low)).clamp(0, 1)
    keep = 1.0 - ramp  # 1: extrapolate (original frequency), 0: interpolate (divided by factor)
    inv = inv_extra * keep + inv_extra / factor * (1.0 - keep)

    def get_mscale(scale, m):
        return 1.0 if scale <= 1 else 0.1 * m * math.log(scale) + 1.0

    mscale = get_mscale(factor, float(params.get("mscale", 1))) / \
        get_mscale(factor, float(params.get("mscale_all_dim", 0)))
    return inv.float(), dims, mscale


def _sdpa(q, k, v, mask, scale):
    """Attention over the returned K/V for steps the fused kernels do not take: float32, GQA by
    grouping query heads, ``mask`` None, "causal" (bottom-right) or a boolean [Lq, Lk] array."""
    B, Hq, Lq, D = q.shape
    Hkv, Lk = k.shape[1], k.shape[2]
    G = Hq // Hkv
    qf = q.float().reshape(B, Hkv, G * Lq, D)
    s = torch.matmul(qf, k.float().transpose(-1, -2).contiguous()) * scale
    s = s.reshape(B, Hkv, G, Lq, Lk)
    if isinstance(mask, str):
        mask = torch.arange(Lk)[None, :] <= torch.arange(Lk - Lq, Lk)[:, None]
    if mask is not None:
        s = s.masked_fill(~mask.to(s.device), float("-inf"))
    p = torch.softmax(s, dim=-1).reshape(B, Hkv, G * Lq, Lk)
    return torch.matmul(p, v.float()).reshape(B, Hq, Lq, D).to(q.dtype)


# looked up once: the checks run on every product of a short block, which the host bounds
_C = torch._C
_peek_functorch, _is_tracing, _is_compiling = (_C._functorch.peek_interpreter_stack, _C._is_tracing,
                                               torch.compiler.is_compiling)
_dispatch_modes, _function_modes = _C._len_torch_dispatch_stack, _C._len_torch_function_stack
_autocast, _grad_enabled, _Tensor = _C._is_any_autocast_enabled, torch.is_grad_enabled, torch.Tensor


def _unwatched(x, w):
    """Whether an operation on these may be launched past torch's dispatcher: plain tensors, and nothing
    that records, rewrites or casts what the dispatcher sees -- autograd, forward mode, function
    transforms (vmap, grad), jit and fx tracing, compilation, dispatch and function modes (other than a
    default device's) and autocast. Those get the library product, which they can see."""
    return (type(x) is type(w) is _Tensor
            and not ((x.requires_grad or w.requires_grad) and _grad_enabled())
            and not _dispatch_modes() and _peek_functorch() is None and not _is_tracing()
            and forward_ad._current_level < 0 and not _autocast() and not _is_compiling()
            and (not _function_modes() or all(type(_C._get_function_stack_at(i)) is DeviceContext
                                              for i in range(_function_modes()))))


def _row_form_pays(rows, N, K):
    """Whether ``lq_gemm_rows_bf16`` is the faster of the two for ``rows`` x K against N outputs. A wave
    has an eighth of K in steps of 32, eight of them in flight, so up to 2,048 it is one round of loads
    and to 4,096 two (worth it from the second's half); a workgroup has 16 outputs, so up to 4,096 there
    is one on each of the 256 CUs, and every workgroup reads all rows. us per call, row form / library,
    weights not cached, in a graph:

    * one workgroup per CU -- 1,024 outputs of 1,024, 16 rows 5.7 / 5.8; 2,048 of 4,096, 8 rows 8.3 /
      14.3, 16 rows 9.7 / 14.3; 4,096 of 3,072, 16 rows 10.5 / 12.6. Not with a second round hardly
      used (1,024 of 2,304, 8 rows 7.8 / 7.6) or three (2,048 of 6,144, 8 rows 11.4 / 11.0; 1,024 of
      5,120, 16 rows 14.3 / 9.9), nor with short rows (512 of 512, 8 rows 4.8 / 4.4);
    * two -- 6,176 of 2,048, 8 rows 8.8 / 12.4; 8,192 of 1,536, 12 rows 10.2 / 10.7, 16 rows 11.2 / 10.6;
      6,176 of 1,024, 5 rows 7.7 / 8.1, 8 rows 8.3 / 8.2; with two rounds 6,176 of 4,096, 8 rows 15.0 /
      14.3;
    * three, all eight steps of a round used -- 8,240 of 2,048, 8 rows 11.2 / 12.9; 12,288 of 1,920, 8
      rows 12.7 / 13.4, 12 rows 14.3 / 13.5; 10,240 of 1,792, 8 rows 13.0 / 12.6; 16,384 of 1,920, 8
      rows 16.5 / 14.8."""
    if N < 1024 or not (1024 <= K <= 2048 or 3072 <= K <= 4096):
        return False
    if N <= 4096:
        return True
    if K > 2048:
        return False
    if N <= 8192:
        return rows <= (12 if K >= 1536 else 4)
    return N <= 12288 and K > 1792 and rows <= 8


def _row_form(x, w, rows, K):
    """Whether ``lq_gemm_rows_bf16`` takes this product: what the kernel reads (bf16, contiguous,
    16-byte aligned), in a call that nothing watches."""
    return (w.dim() == 2 and w.shape[1] == K and K % 8 == 0 and _row_form_pays(rows, w.shape[0], K)
            and x.dtype == w.dtype == torch.bfloat16 and x.is_cuda and x.device == w.device
            and x.is_contiguous() and w.is_contiguous() and _unwatched(x, w)
            and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``x @ w.T`` for bf16 ``x [..., K]`` and ``w [N, K]``: one row (a decode step) runs
    ``lq_gemv_bf16`` (weight-streaming, HBM-bound), 2 to 16 rows (a verify block) the matrix-core
    form of it, ``lq_gemm_rows_bf16``, where it is faster, more rows the library GEMM."""
    K = x.shape[-1]
    rows = x.numel() // K if K else 1  # no inputs: refused by the row's entry
    if rows != 1 and not (2 <= rows <= 16 and _row_form(x, w, rows, K)):
        return torch.matmul(x, w.t())
    lib = _lib.load()
    dev = _lib.require_device(x, w)
    x = x.contiguous()
    y = torch.empty((*x.shape[:-1], w.shape[0]), dtype=torch.bfloat16, device=dev)
    if rows == 1:
        _lib.check(lib.lq_gemv_bf16(w.data_ptr(), x.data_ptr(), y.data_ptr(), w.shape[0], K,
                                    _lib.stream_ptr(dev)), "lq_gemv_bf16")
    else:
        _lib.check(lib.lq_gemm_rows_bf16(w.data_ptr(), x.data_ptr(), y.data_ptr(), rows, w.shape[0],
                                         K, _lib.stream_ptr(dev)), "lq_gemm_rows_bf16")
    return y


class Attention:
    """``laguna_mlx.laguna.Attention`` for a full-attention layer, head_dim 128.

    Weights (bf16, on the GPU): ``wq [Hq*128, C]``, ``wk``/``wv [Hkv*128, C]``, ``wo [C, Hq*128]``,
    ``wg [Hq, C]`` (per-head gate) or ``[Hq*128, C]``, ``q_norm``/``k_norm [128]``."""

    def __init__(self, wq, wk, wv, wo, wg, q_norm, k_norm, n_heads, n_kv_heads, rope: dict,
                 eps: float = 1e-6, head_dim: int = 128):
        if head_dim != 128:
            raise ValueError("head_dim must be 128")
        self.n_heads, self.n_kv_heads, self.head_dim, self.eps = n_heads, n_kv_heads, head_dim, eps
        self.scale = head_dim ** -0.5
        self.per_head_gate = wg.shape[0] == n_heads
        dev = wq.device
        self.w_in = torch.cat([wq, wk, wv, wg], dim=0).to(torch.bfloat16).contiguous()
        self.wo = wo.to(torch.bfloat16).contiguous()
        self.q_norm = q_norm.to(device=dev, dtype=torch.bfloat16).contiguous()
        self.k_norm = k_norm.to(device=dev, dtype=torch.bfloat16).contiguous()
        inv, self.rot_dims, self.mscale = rope_frequencies(head_dim, rope)
        self.inv_freq = inv.to(dev)
        H, Hkv, D = n_heads, n_kv_heads, head_dim
        self._splits = [H * D, Hkv * D, Hkv * D, wg.shape[0]]

    def __call__(self, x: torch.Tensor, mask=None, cache=None) -> torch.Tensor:
        lib = _lib.load()
        dev = _lib.require_device(x)
        B, L, _ = x.shape
        H, Hkv, D = self.n_heads, self.n_kv_heads, self.head_dim
        x = x.to(torch.bfloat16)
        proj = linear(x, self.w_in)  # [B, L, (H + 2 Hkv) D + gate]
        N = proj.shape[-1]
        q = torch.empty((B, H, L, D), dtype=torch.bfloat16, device=dev)
        k = torch.empty((B, Hkv, L, D), dtype=torch.bfloat16, device=dev)
        v = torch.empty((B, Hkv, L, D), dtype=torch.bfloat16, device=dev)
        offset = cache.offset if cache is not None else 0
        _lib.check(lib.lq_qkv_norm_rope(proj.data_ptr(), N, q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                        self.q_norm.data_ptr(), self.k_norm.data_ptr(), B, H, Hkv,
                                        L, D, self.eps, self.inv_freq.data_ptr(), self.rot_dims,
                                        self.mscale, int(offset), _lib.stream_ptr(dev)),
                   "lq_qkv_norm_rope")
        if cache is not None:
            k, v = cache.update_and_fetch(k, v)
        if getattr(cache, "fused_step", False):
            out = cache.attend(q, self.scale)
        elif hasattr(cache, "bits"):  # quantized_decode step: packed K/V, quantized attention
            from .q8_attn import quantized_scaled_dot_product_attention
            out = quantized_scaled_dot_product_attention(q, k, v, self.scale, mask,
                                                         cache.group_size, cache.bits)
        else:
            out = _sdpa(q, k, v, mask, self.scale)
        out = out.to(torch.bfloat16).contiguous()
        y = torch.empty((B, L, H, D), dtype=torch.bfloat16, device=dev)
        gate = proj.data_ptr() + 2 * (H + 2 * Hkv) * D  # the last columns of the projection rows
        _lib.check(lib.lq_gate_heads_strided(out.data_ptr(), gate, N, y.data_ptr(), B, H, L, D,
                                             0 if self.per_head_gate else 1, _lib.stream_ptr(dev)),
                   "lq_gate_heads_strided")
        return linear(y.reshape(B, L, H * D), self.wo)
