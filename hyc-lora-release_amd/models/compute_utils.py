"""Torch-side glue of the fused layers (reference: models/utils/compute_utils.py:7-51 and
operators/rope_kernels.py:81-126).  The frozen-weight GEMMs and the attention products are library /
torch operations in the reference as well; only what surrounds them is compressed.  RoPE is the
in-place HIP kernel of operators/rope_kernels.py, re-exported here."""
import torch

from .. import _lib
from ..operators import lora_kernels
from ..operators.nf4 import dequantize_nf4


def hidden_to_head_shape(x: torch.Tensor, num_heads: int):
    bsz, seq_len, hidden = x.shape
    return x.reshape(bsz, seq_len, num_heads, hidden // num_heads).transpose(1, 2)


def head_to_hidden_shape(x: torch.Tensor):
    bsz, _, seq_len, _ = x.shape
    return x.transpose(1, 2).reshape(bsz, seq_len, -1).contiguous()


_MAX_BATCH_LOOP = 16


def heads_matmul(a: torch.Tensor, b: torch.Tensor, out_hidden: bool = False):
    """a @ b for [B, H, M, K] x [B, H, K, N] operands that are *views* of hidden-layout tensors
    ([B, S, H*D] seen as [B, H, S, D]).  torch.matmul would first copy such a view into head-major
    memory (the reference pays that copy at every attention product); a batched GEMM over the heads
    of one batch element reads it in place (row stride H*D, batch stride D), so this loops over the
    batch.  out_hidden=True writes the result [B, H, M, N] into a hidden-layout buffer and returns
    its [B, H, M, N] view, which makes the following head_to_hidden_shape free."""
    B, H, M, _ = a.shape
    N = b.shape[-1]
    if B > _MAX_BATCH_LOOP or not a.is_cuda or a.dtype != b.dtype:
        r = torch.matmul(a, b)
        return r.transpose(1, 2).contiguous().transpose(1, 2) if out_hidden else r
    if out_hidden:
        out = a.new_empty(B, M, H, N).transpose(1, 2)
    else:
        out = a.new_empty(B, H, M, N)
    for i in range(B):
        torch.bmm(a[i], b[i], out=out[i])
    return out


def frozen_matmul(x: torch.Tensor, w: torch.Tensor):
    """x @ w for a frozen weight (or its transposed view) w [K, N]: the kernel for a few rows (csrc/few_rows.hip) where that is the
    faster one, else the library product, in the calls that suit its tiles (the rules stand in csrc/host/native.cpp)."""
    if x.is_cuda:
        done = _lib.native().frozen_matmul(x, w)
        if done is not None:
            return done
    return x @ w


def dense_weight(w: torch.Tensor, quant_state):
    """Frozen weight as a dense [out, in] matrix.  quant_state None = already dense (the benchmark
    configurations); otherwise a bitsandbytes-format NF4 weight, dequantised by the HIP kernel (the
    reference calls BF.dequantize_nf4 at the same place, compute_utils.py:19, :29)."""
    if quant_state is None:
        return w
    return dequantize_nf4(w, quant_state)


def lora_forward(w, w_quant_state, w_lora_a, w_lora_b, b, x, residual=None, x_lora_a=None):
    """-> (x @ W^T [+ b] + (x @ A) @ B, the frozen part alone, x @ A).  Reference :18-25.  The LoRA
    product and the add are one MFMA kernel over the frozen part (bf16 operands); other dtypes
    take the torch expression.  `residual` (not in the reference's signature) is added to the first
    result in the same pass - the `x + o_final` that follows the projection in the layers.
    `x_lora_a`: x @ A where the producer of x has already formed it."""
    if b is None and x.is_cuda:
        w, w_quant_state = dense_weight(w, w_quant_state), None
        done = _lib.native().lora_forward(w, w_lora_a, w_lora_b, x, residual, x_lora_a)
        if done is not None:
            return done
    x_main, x_lora_a = lora_parts(w, w_quant_state, w_lora_a, b, x, x_lora_a)
    w_lora_b = w_lora_b.to(x_main.dtype)
    if lora_kernels.supported(x_main, x_lora_a, w_lora_b) and (residual is None or residual.dtype == x_main.dtype):
        return lora_kernels.lora_add(x_main, x_lora_a, w_lora_b, residual=residual), x_main, x_lora_a
    y = x_main + x_lora_a @ w_lora_b
    return (y if residual is None else residual + y), x_main, x_lora_a


def lora_parts(w, w_quant_state, w_lora_a, b, x, x_lora_a=None):
    """-> (x @ W^T [+ b], x @ A): what lora_forward computes before the LoRA add.  x @ A is taken
    from `x_lora_a` when the caller has it already (the fused norm kernel forms it)."""
    w = dense_weight(w, w_quant_state)
    if b is None and x.is_cuda:
        done = _lib.native().lora_parts(w, w_lora_a, x, x_lora_a)
        if done is not None:
            return done
    wt = w.t()
    x = x.to(wt.dtype)
    x_main = frozen_matmul(x, wt)
    if b is not None:
        x_main = x_main + b.to(wt.dtype)
    if x_lora_a is None:
        x_lora_a = x @ w_lora_a.to(wt.dtype)
    return x_main, x_lora_a.to(wt.dtype)


def lora_backward(w, w_quant_state, w_lora_a, w_lora_b, x, x_lora_a, grad_y, x_codes=None, accumulate=None,
                  defer_input=False):
    """-> (grad lora_A, grad lora_B, grad x).  Reference :28-36.

    With bf16 operands the rank-R products stream their wide operand once on the matrix cores:
    grad_y gives `grad_y @ B^T` and `xa^T @ grad_y` in one pass, and `x^T @ grad_medium` is taken
    from x - or straight from its packed codes `x_codes = (q, scale, zero_point or None, q_bit)`,
    in which case x may be None and is never dequantised.  Those results are summed over the batch in
    fp32 and have the parameters' shapes; the torch expressions below return one gradient per batch
    element, as the reference does, and leave the sum to autograd.  `accumulate`, a running sum of
    input gradients, is added to grad x in the pass that adds its LoRA part (`grad_x += grad_x_temp`
    in the layers) and may be overwritten.  With `defer_input` the third result is not grad x but its
    two terms and the operand that joins them, `(grad_y @ W, grad_y @ B^T, A^T)`, for lora_input_sum, which
    adds up the input gradients of projections that share their input in one pass."""
    wd = dense_weight(w, w_quant_state)          # [out, in]
    if grad_y.is_cuda:
        q, scale, zero_point, q_bit = x_codes or (None, None, None, 0)
        if zero_point is not None and zero_point.dtype != torch.bfloat16:
            zero_point = _lib.bf16_vector(zero_point)
        done = _lib.native().lora_backward(wd, w_lora_a, w_lora_b, None if x_codes else x, q, scale, zero_point, q_bit, x_lora_a, grad_y,
                                           accumulate, defer_input)
        if done is not None:
            return done
    dt = wd.dtype
    grad_y = grad_y.to(dt)
    w_lora_a, w_lora_b = w_lora_a.to(dt), w_lora_b.to(dt)
    r = w_lora_b.shape[0]
    if lora_kernels.contract_supported(grad_y, grad_y.shape[-1], r) and x_lora_a.dtype == dt:
        # xa^T @ grad_y written as [N, R], the layout of the lora_B weight this gradient ends up in: what is
        # returned is its [R, N] view, and autograd's transpose back is then contiguous and stored without a copy
        grad_b, grad_mid = lora_kernels.lora_products(grad_y, u=x_lora_a, v=w_lora_b, p1_transposed=True)
        grad_b = grad_b.t()
    else:
        grad_mid = grad_y @ w_lora_b.mT
        grad_b = x_lora_a.to(dt).mT @ grad_y
    if x_codes is not None and lora_kernels.contract_supported(grad_mid, w_lora_a.shape[0], r):
        q, scale, zero_point, q_bit = x_codes
        grad_a = lora_kernels.lora_product_from_codes(q, scale, grad_mid, zero_point, q_bit).t()
    else:
        if x is None:
            from ..operators.compress_function import (decompression_dequantization,
                                                       decompression_dequantization_with_zero_point)
            q, scale, zero_point, q_bit = x_codes
            x = decompression_dequantization(q, scale, q_bit) if zero_point is None else \
                decompression_dequantization_with_zero_point(q, scale, zero_point, q_bit)
        if lora_kernels.contract_supported(x, x.shape[-1], r) and grad_mid.dtype == x.dtype:
            grad_a = lora_kernels.lora_products(x, u=grad_mid)[0].t()
        else:
            grad_a = x.to(dt).mT @ grad_mid
    grad_x = frozen_matmul(grad_y, wd)
    if defer_input:
        return grad_a, grad_b, (grad_x, grad_mid, w_lora_a.mT)
    if lora_kernels.supported(grad_x, grad_mid, w_lora_a.mT) and (accumulate is None or accumulate.dtype == dt):
        grad_x = lora_kernels.lora_add(grad_x, grad_mid, w_lora_a.mT, inplace=True, residual=accumulate)
    else:
        grad_x += grad_mid @ w_lora_a.mT
        if accumulate is not None:
            grad_x = accumulate + grad_x
    return grad_a, grad_b, grad_x


def lora_backward_shared(members, x, x_codes=None):
    """lora_backward(..., defer_input=True) of two or three projections that share their input x, given like there:
    members [(w, w_quant_state, w_lora_a, w_lora_b, x_lora_a, grad_y), ...] -> the list of its results, the same bits.
    The rank-R products of all members take two launches and their reductions, and x (or its codes) is read once; the
    weights are dequantised one at a time."""
    out = None
    if x_codes is None or x_codes[2] is None or x_codes[2].dtype == torch.bfloat16:
        q, scale, zero_point, q_bit = x_codes or (None, None, None, 0)
        if all(gy.is_cuda and (w.dtype if qs is None else getattr(qs, "dtype", torch.bfloat16)) == torch.bfloat16 for w, qs, _, _, _, gy in members):
            out = _lib.native().lora_products_shared([(la, lb, xa, gy) for _, _, la, lb, xa, gy in members], None if x_codes else x, q, scale,
                                                     zero_point, q_bit)
    if out is None:
        return [lora_backward(w, qs, la, lb, x, xa, gy, x_codes=x_codes, defer_input=True) for w, qs, la, lb, xa, gy in members]
    results = []
    for (w, qs, la, _, _, gy), (grad_a, grad_b, grad_mid) in zip(members, out):
        wd = dense_weight(w, qs)
        grad_x = _lib.native().frozen_input_grad(gy, wd)
        results.append((grad_a, grad_b, (frozen_matmul(gy, wd) if grad_x is None else grad_x, grad_mid, la.mT)))
        del wd
    return results


def lora_backward_sum(members, x, x_codes=None, residual=None):
    """lora_backward_shared with the input gradients added up: -> ([(grad lora_A, grad lora_B), ...], their sum [+ residual]), the
    additions in bf16 and in order.  Where the products are small enough for this package's kernel they, their LoRA adds
    and the sum are one launch."""
    if all(qs is None and gy.is_cuda and w.dtype == torch.bfloat16 for w, qs, _, _, _, gy in members) and x_codes is not None and x_codes[2] is None:
        out = _lib.native().lora_products_shared([(la, lb, xa, gy) for _, _, la, lb, xa, gy in members], None, x_codes[0], x_codes[1], None, x_codes[3])
        if out is not None:
            grads = [(ga, gb) for ga, gb, _ in out]
            grad_x = _lib.native().lora_input_grad([(gy, w, mid, la.mT) for (w, _, la, _, _, gy), (_, _, mid) in zip(members, out)], residual)
            if grad_x is None:
                grad_x = lora_input_sum([(frozen_matmul(gy, w), mid, la.mT) for (w, _, la, _, _, gy), (_, _, mid) in zip(members, out)])
                grad_x = grad_x if residual is None else grad_x + residual
            return grads, grad_x
    terms = lora_backward_shared(members, x, x_codes)
    grad_x = lora_input_sum([t for _, _, t in terms])
    return [(ga, gb) for ga, gb, _ in terms], grad_x if residual is None else grad_x + residual


def lora_input_sum(parts):
    """Sum of the input gradients of projections that share their input, from the deferred terms lora_backward
    returns: acc = t_0; acc += t_1; ... with t_i = (grad_y @ W)_i + (grad_y @ B^T)_i @ A_i^T, every operation
    rounded as the chain of lora_backward(..., accumulate=acc) calls rounds it (the reference's
    `grad_x += grad_x_temp`).  Two or three bf16 terms of rank <= 16 take one pass over their operands."""
    terms = list(parts)
    if lora_kernels.supported_sum(terms):
        return lora_kernels.lora_add_sum(terms)
    acc = None
    for grad_x, grad_mid, a_t in terms:
        if lora_kernels.supported(grad_x, grad_mid, a_t) and (acc is None or acc.dtype == grad_x.dtype):
            acc = lora_kernels.lora_add(grad_x, grad_mid, a_t, inplace=True, residual=acc)
        else:
            grad_x += grad_mid @ a_t
            acc = grad_x if acc is None else acc + grad_x
    return acc


def repeat_kv(hidden_states: torch.Tensor, n_rep: int):
    """[B, KV, S, D] -> [B, KV * n_rep, S, D], every key / value head n_rep times in a row.  Reference :38-43."""
    if n_rep == 1:
        return hidden_states
    b, kv, s, d = hidden_states.shape
    return hidden_states[:, :, None, :, :].expand(b, kv, n_rep, s, d).reshape(b, kv * n_rep, s, d)


def repeat_kv_backward(grad_output: torch.Tensor, n_rep: int):
    """Gradient of repeat_kv: the n_rep copies of a head summed.  Reference :46-50."""
    if n_rep == 1:
        return grad_output
    return grad_output.unflatten(1, (grad_output.shape[1] // n_rep, n_rep)).sum(dim=2)


def unpad_input(hidden_states, attention_mask):
    """[B, S, ...] and a key-padding mask [B, S] (non-zero = a real token) -> (the real tokens' rows
    [nnz, ...], their positions in the flattened [B * S] axis, cumulative sequence lengths int32 [B + 1], the
    longest sequence as an int).  Reference :69-97 (flash-attn's padding helper; its map-free layers call it,
    the ones in this package mask instead).  Reads the longest length back from the device, as there."""
    lengths = attention_mask.sum(dim=-1, dtype=torch.int32)
    indices = torch.nonzero(attention_mask.flatten(), as_tuple=False).flatten()
    cu_seqlens = torch.nn.functional.pad(torch.cumsum(lengths, dim=0, dtype=torch.int32), (1, 0))
    rows = hidden_states.reshape(-1, *hidden_states.shape[2:])
    return rows[indices], indices, cu_seqlens, int(lengths.max().item())


def pad_input(hidden_states, indices, batch, seqlen):
    """Inverse of unpad_input: rows [nnz, ...] back at `indices` of a zero-filled [batch, seqlen, ...].
    Reference :53-66."""
    out = hidden_states.new_zeros((batch * seqlen,) + tuple(hidden_states.shape[1:]))
    out[indices] = hidden_states
    return out.reshape(batch, seqlen, *hidden_states.shape[1:])


from ..operators.rope_kernels import rope_backward, rope_forward  # noqa: E402,F401  (in place, HIP)
