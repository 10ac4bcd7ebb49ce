"""Attention without a map on the gfx950 matrix cores (hyc_flash_fwd / hyc_flash_bwd).

The reference calls flash-attn's varlen kernels at these places
(models/llama_flash_attn/fused_llama_layer_intra_inter.py:169-180, :459-468).  Tensors are [B, heads, S, D] like there;
views of hidden-layout memory ([B, S, heads * D]), which is what the layers hold, are read in place, and the results come
as such views.  Grouped key / value heads are read as they are: no repeat_kv copies, and their gradients come summed."""
import math

import torch

from .. import _lib

BF16 = torch.bfloat16


def flash_supported(q, k, v):
    """Whether flash_forward / flash_backward take these operands."""
    return (q.is_cuda and q.device == k.device == v.device and q.dtype == k.dtype == v.dtype == BF16 and q.dim() == 4 and k.shape == v.shape and q.shape[0] == k.shape[0]
            and q.shape[2:] == k.shape[2:] and q.shape[3] in (64, 128) and q.shape[1] % k.shape[1] == 0 and q.numel() > 0
            and q.shape[2] <= 1 << 20 and q[0].numel() <= 1 << 30 and -(-q.shape[2] // 128) * q.shape[0] * q.shape[1] <= 1 << 23)


def _hidden(t):
    """[B, heads, S, D] -> contiguous [B, S, heads, D]; free for views of hidden-layout memory."""
    t = t.transpose(1, 2).contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _check(q, k, v):
    if not flash_supported(q, k, v):
        raise ValueError(f"attention takes bf16 [B, H, S, D] queries and [B, KV, S, D] keys / values with D 64 or 128 on one GPU, got "
                         f"{tuple(q.shape)} {q.dtype} {q.device}, {tuple(k.shape)} {k.dtype} {k.device}, {tuple(v.shape)} {v.dtype} {v.device}")


def flash_forward(q, k, v, causal=True):
    """-> (o [B, H, S, D], log-sum-exp of the scaled scores fp32 [B, H, S])."""
    _check(q, k, v)
    B, H, S, D = q.shape
    q, k, v = _hidden(q), _hidden(k), _hidden(v)
    o = torch.empty_like(q)
    lse = torch.empty((B, H, S), device=q.device, dtype=torch.float32)
    _lib.call("hyc_flash_fwd", q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), B, S, H, k.shape[2], D,
              1.0 / math.sqrt(D), int(causal), _lib.stream_of(q))
    return o.transpose(1, 2), lse


def flash_backward(grad_o, q, k, v, o, lse, causal=True):
    """-> (grad_q, grad_k, grad_v), shaped like q, k and v.  `o` need not be the forward's output bit for bit: the layers
    hand in the dequantised one, as the reference does."""
    _check(q, k, v)
    B, H, S, D = q.shape
    if grad_o.shape != q.shape or o.shape != q.shape or grad_o.dtype != BF16 or o.dtype != BF16:
        raise ValueError(f"grad_o and o must be bf16 {tuple(q.shape)}, got {tuple(grad_o.shape)} {grad_o.dtype}, {tuple(o.shape)} {o.dtype}")
    if lse.dtype != torch.float32 or lse.numel() != B * H * S:
        raise ValueError(f"lse must be float32 [{B}, {H}, {S}], got {lse.dtype} {tuple(lse.shape)}")
    _lib.require_gpu(grad_o, o, lse)
    grad_o, q, k, v, o = _hidden(grad_o), _hidden(q), _hidden(k), _hidden(v), _hidden(o)
    lse = lse.contiguous()
    gq, gk, gv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    delta = torch.empty((2, B, H, S), device=q.device, dtype=torch.float32)
    _lib.call("hyc_flash_bwd", grad_o.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(),
              delta.data_ptr(), gq.data_ptr(), gk.data_ptr(), gv.data_ptr(), B, S, H, k.shape[2], D, 1.0 / math.sqrt(D), int(causal),
              _lib.stream_of(q))
    return gq.transpose(1, 2), gk.transpose(1, 2), gv.transpose(1, 2)
