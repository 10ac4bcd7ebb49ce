"""Attention through a sparsely kept softmax map (hyc_map_fwd / hyc_map_emit / hyc_map_bwd): what the layers' attention
computes between the rotated q, k, v and the output projection, without a dense map in memory.

The reference forms it from torch products, a softmax and `to_sparse`, and in backward from `to_dense`, four products and
softmax_backward (models/llama/fused_llama_layer_intra_inter_full_fuse.py:153-180, :403-447).  Tensors are [B, heads, S, D]
views of hidden-layout memory, keys and values may have fewer (grouped) heads."""
import math

import torch

from .. import _lib
from .compress_function import PendingCount, _threshold_tensor, check_map_lists
from .flash_kernels import _hidden, flash_supported

BF16 = torch.bfloat16
MAX_ROW = 4096


def map_supported(q, k, v, mask=None):
    """Whether map_forward takes these operands; mask: None or additive [B or 1, 1, S or 1, S]."""
    if not flash_supported(q, k, v) or q.shape[2] % 8 or q.shape[2] > MAX_ROW:
        return False
    B, H, S, _ = q.shape
    if -(-S // 32) * B * H > 1 << 22:
        return False
    return mask is None or (mask.dim() == 4 and mask.device == q.device and mask.shape[0] in (1, B) and mask.shape[1] == 1 and
                            mask.shape[2] in (1, S) and mask.shape[3] == S)


def map_backward_supported(q, k, v, idx):
    """Whether map_backward takes these operands and a list `idx` of kept entries: the kernels count entries in 32 bits."""
    return map_supported(q, k, v) and idx.numel() < 1 << 31


class MapAttention:
    """One forward: `o` [B, H, S, D], `map` (the dense map, if asked for), and with a threshold the kept entries on demand."""

    def __init__(self, q, k, v, mask=None, threshold=None, want_map=False):
        if not map_supported(q, k, v, mask):
            raise ValueError(f"map attention takes bf16 q [B, H, S, D], k and v [B, KV, S, D] with D 64 or 128, S a multiple of 8 up to "
                             f"{MAX_ROW}, and a mask [B or 1, 1, S or 1, S]; got {tuple(q.shape)}, {tuple(k.shape)}, "
                             f"{None if mask is None else tuple(mask.shape)}")
        B, H, S, D = q.shape
        self.shape, self.KV, self.scale = (B, H, S, D), k.shape[1], 1.0 / math.sqrt(D)
        self.q, self.k, v = _hidden(q), _hidden(k), _hidden(v)
        self.mask, self.mask_strides = None, (0, 0)
        if mask is not None:
            if mask.dtype != BF16:
                mask = mask.to(BF16)
            if mask.stride(-1) != 1 or mask.stride(2) % 8 or mask.stride(0) % 8 or mask.data_ptr() % 16:
                mask = mask.contiguous()
            self.mask = mask
            self.mask_strides = (mask.stride(0) if mask.shape[0] > 1 else 0, mask.stride(2) if mask.shape[2] > 1 else 0)
        self.threshold = None if threshold is None else _threshold_tensor(threshold, q.device)
        o = torch.empty_like(self.q)
        self.map = torch.empty((B, H, S, S), device=q.device, dtype=BF16) if want_map else None
        self.workspace = torch.empty(_lib.lib().hyc_map_workspace(B, S, H), device=q.device, dtype=torch.uint8)
        _lib.call("hyc_map_fwd", self.q.data_ptr(), self.k.data_ptr(), v.data_ptr(), _lib.ptr(self.mask), *self.mask_strides, o.data_ptr(),
                  _lib.ptr(self.map), _lib.ptr(self.threshold), self.workspace.data_ptr(), self.workspace.numel(), B, S, H, self.KV, D,
                  self.scale, _lib.stream_of(o))
        self.o = o.transpose(1, 2)

    def entries(self, capacity, seg_offsets=None):
        """(indices int64 [capacity], values bf16 [capacity], seg_offsets): the kept entries as compress_attention_map lists
        them.  seg_offsets[-1] is their number; a list that is shorter holds the first `capacity`."""
        B, H, S, D = self.shape
        dev = self.q.device
        idx = torch.empty(capacity, device=dev, dtype=torch.int64)
        val = torch.empty(capacity, device=dev, dtype=BF16)
        nseg = -(-B * H * S * S // 4096)
        if seg_offsets is None:
            seg_offsets = torch.empty(nseg + 1, device=dev, dtype=torch.int64)
        elif seg_offsets.device != dev or seg_offsets.dtype != torch.int64 or seg_offsets.numel() != nseg + 1 or not seg_offsets.is_contiguous():
            raise ValueError(f"seg_offsets must be int64 [{nseg + 1}] on {dev}, got {seg_offsets.dtype} {tuple(seg_offsets.shape)} on {seg_offsets.device}")
        _lib.call("hyc_map_emit", self.q.data_ptr(), self.k.data_ptr(), _lib.ptr(self.mask), *self.mask_strides, self.threshold.data_ptr(),
                  self.workspace.data_ptr(), self.workspace.numel(), capacity, idx.data_ptr() if capacity else None,
                  val.data_ptr() if capacity else None, seg_offsets.data_ptr(), B, S, H, self.KV, D, self.scale, _lib.stream_of(idx))
        return idx, val, seg_offsets

    def bounded_entries(self, capacity):
        """entries(capacity) and a PendingCount of their number: nothing is read back here."""
        idx, val, seg = self.entries(int(capacity))
        return idx, val, seg, PendingCount(seg[-1:])


def map_backward(grad_o, q, k, v, idx, val, seg_offsets):
    """-> (grad_q, grad_k, grad_v), shaped like q, k, v, from the kept entries of the map."""
    if not map_backward_supported(q, k, v, idx):
        raise ValueError(f"map attention does not take {tuple(q.shape)}, {tuple(k.shape)} and a list of {idx.numel()} entries")
    B, H, S, D = q.shape
    if grad_o.shape != q.shape or grad_o.dtype != BF16:
        raise ValueError(f"grad_o must be bf16 {tuple(q.shape)}, got {tuple(grad_o.shape)} {grad_o.dtype}")
    check_map_lists(idx, val, seg_offsets, B * H * S * S)
    _lib.require_gpu(grad_o, idx, val, seg_offsets)
    if val.dtype != BF16:
        raise ValueError(f"map values must be bfloat16, got {val.dtype}")
    idx, val, seg_offsets = idx.reshape(-1).contiguous(), val.reshape(-1).contiguous(), seg_offsets.contiguous()
    grad_o, q, k, v = _hidden(grad_o), _hidden(q), _hidden(k), _hidden(v)
    gq, gk, gv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    n = idx.numel()
    ws = torch.empty(max(16, _lib.lib().hyc_map_bwd_workspace(B, S, H, k.shape[2], D, n)), device=q.device, dtype=torch.uint8)
    _lib.call("hyc_map_bwd", grad_o.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), idx.data_ptr() if n else None,
              val.data_ptr() if n else None, seg_offsets.data_ptr(), n, ws.data_ptr(), ws.numel(), gq.data_ptr(), gk.data_ptr(),
              gv.data_ptr(), B, S, H, k.shape[2], D, 1.0 / math.sqrt(D), _lib.stream_of(q))
    return gq.transpose(1, 2), gk.transpose(1, 2), gv.transpose(1, 2)
