"""The torch-side glue of the layers (reference: models/utils/compute_utils.py:7-51) on the GPU:
lora_forward / lora_backward against the reference's expressions evaluated in float64, with and
without the kernels' extra arguments, and the attention products on hidden-layout views."""
import math

import numpy as np
import pytest
import torch

from helpers import BF16, assert_close_bf16, bits
from oracle import hyc_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def CU():
    import hyclora_amd  # noqa: F401
    from hyclora_amd.models import compute_utils
    return compute_utils


def lora_case(dev, seed, B=2, M=48, n_in=256, n_out=384, R=16, dtype=BF16):
    g = torch.Generator().manual_seed(seed)
    w = (torch.randn(n_out, n_in, generator=g) * 0.05).to(dtype).to(dev)
    a_w = torch.empty(R, n_in)
    torch.nn.init.kaiming_uniform_(a_w, a=math.sqrt(5), generator=g)
    a_w = a_w.to(dtype).to(dev)                              # lora_A.weight [R, in]
    b_w = (torch.randn(n_out, R, generator=g) * 0.05).to(dtype).to(dev)     # lora_B.weight [out, R]
    bias = (torch.randn(n_out, generator=g) * 0.1).to(dtype).to(dev)
    x = torch.randn(B, M, n_in, generator=g).to(dtype).to(dev)
    gy = torch.randn(B, M, n_out, generator=g).to(dtype).to(dev)
    return w, a_w, b_w, bias, x, gy


@pytest.mark.parametrize("dtype", [BF16, torch.float32])
@pytest.mark.parametrize("with_bias", [False, True])
def test_lora_forward_and_backward_match_the_reference_expressions(CU, dev, dtype, with_bias):
    w, a_w, b_w, bias, x, gy = lora_case(dev, 1, dtype=dtype)
    bias = bias if with_bias else None
    y, main, xa = CU.lora_forward(w, None, a_w.T, b_w.T, bias, x)
    X, Wd, A, Bm = x.double(), w.double(), a_w.double(), b_w.double()
    main_ref = X @ Wd.T + (bias.double() if with_bias else 0.0)
    assert_close_bf16(main, main_ref, what="frozen part")
    assert_close_bf16(xa, X @ A.T, what="x @ A")
    assert_close_bf16(y, main_ref + (X @ A.T) @ Bm.T, what="projection output")
    ga, gb, gx = CU.lora_backward(w, None, a_w.T, b_w.T, x, xa, gy)
    G = gy.double()
    gm = G @ Bm
    ga_ref = torch.einsum("bmi,bmr->ir", X, gm)
    gb_ref = torch.einsum("bmr,bmo->ro", xa.double(), G)
    # the torch path returns one gradient per batch element (autograd sums them), the kernels the sum
    ga = ga if ga.dim() == 2 else ga.sum(0)
    gb = gb if gb.dim() == 2 else gb.sum(0)
    assert ga.shape == (x.shape[-1], 16) and gb.shape == (16, gy.shape[-1])
    assert_close_bf16(ga, ga_ref, what="grad lora_A")
    assert_close_bf16(gb, gb_ref, what="grad lora_B")
    assert_close_bf16(gx, G @ Wd + gm @ A, what="grad x")


@pytest.mark.parametrize("q_bit", [2, 4, 8])
def test_lora_backward_from_codes_residual_and_accumulate(CU, dev, q_bit):
    from hyclora_amd.operators import compress_function as cf
    w, a_w, b_w, _, x, gy = lora_case(dev, 2 + q_bit)
    s = cf.get_statistics_only_quant(x, q_bit, 'per-channel')
    q = cf.compression_quantization(x, s, q_bit)
    x_hat = cf.decompression_dequantization(q, s, q_bit)
    xa = x @ a_w.T
    acc = torch.randn_like(x)
    ga0, gb0, gx0 = CU.lora_backward(w, None, a_w.T, b_w.T, x_hat, xa, gy)
    ga1, gb1, gx1 = CU.lora_backward(w, None, a_w.T, b_w.T, None, xa, gy, x_codes=(q, s, None, q_bit),
                                     accumulate=acc.clone())
    assert np.array_equal(bits(ga0), bits(ga1)), "codes path == dequantise first"
    assert np.array_equal(bits(gb0), bits(gb1))
    assert np.array_equal(bits(gx1), bits(acc + gx0)), "accumulate == add afterwards"
    res = torch.randn_like(gy)
    y0, _, _ = CU.lora_forward(w, None, a_w.T, b_w.T, None, x)
    y1, _, _ = CU.lora_forward(w, None, a_w.T, b_w.T, None, x, residual=res)
    assert np.array_equal(bits(y1), bits(res + y0))


@pytest.mark.parametrize("B", [2, 17])
@pytest.mark.parametrize("n_rep", [1, 4])
def test_attention_products_on_hidden_layout_views(CU, dev, B, n_rep):
    """heads_matmul == torch.matmul on [B, S, H*D] tensors seen as [B, H, S, D]; with out_hidden the
    result already lies in hidden layout.  B = 17 takes the plain matmul (more batch elements than
    the per-batch loop is used for)."""
    S, H, D = 24, 8, 16
    KV = H // n_rep
    g = torch.Generator().manual_seed(B)
    q = CU.hidden_to_head_shape(torch.randn(B, S, H * D, generator=g).to(BF16).to(dev), H)
    k = CU.repeat_kv(CU.hidden_to_head_shape(torch.randn(B, S, KV * D, generator=g).to(BF16).to(dev), KV), n_rep)
    v = CU.repeat_kv(CU.hidden_to_head_shape(torch.randn(B, S, KV * D, generator=g).to(BF16).to(dev), KV), n_rep)
    s = CU.heads_matmul(q, k.transpose(-2, -1))
    assert s.shape == (B, H, S, S) and s.is_contiguous()
    assert_close_bf16(s, q.double() @ k.double().transpose(-2, -1), what="q k^T")
    a = torch.softmax(s.float(), dim=-1).to(BF16)
    o = CU.heads_matmul(a, v, out_hidden=True)
    assert o.shape == (B, H, S, D) and o.transpose(1, 2).is_contiguous(), "result lies in [B, S, H, D] memory"
    assert_close_bf16(o, a.double() @ v.double(), what="a v")
    hid = CU.head_to_hidden_shape(o)
    assert hid.data_ptr() == o.data_ptr() and hid.shape == (B, S, H * D), "head_to_hidden_shape is then free"
    # grads of k, v summed over the query heads that share them, on the strided view
    gk = CU.heads_matmul(s.transpose(-2, -1), q, out_hidden=True)
    want = (s.double().transpose(-2, -1) @ q.double()).reshape(B, KV, n_rep, S, D).sum(2)
    assert_close_bf16(CU.repeat_kv_backward(gk, n_rep), want, what="repeat_kv_backward on a strided view")


@pytest.mark.parametrize("rows,n,k", [(2048, 2816 + 8192, 128), (1024, 17152, 96), (8192, 2304, 64), (2000, 8448, 64), (256, 65792, 32), (2048, 13824, 64)])
@pytest.mark.parametrize("transposed", [True, False])
def test_frozen_matmul_in_whole_rounds(rows, n, k, transposed):
    """The product in one or two library calls, at sizes on both sides of the rule: the calls' columns meet exactly."""
    import hyclora_amd  # noqa: F401
    from hyclora_amd.models import compute_utils as CU
    g = torch.Generator(device="cuda").manual_seed(rows + n)
    x = torch.randn(1, rows, k, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(*((n, k) if transposed else (k, n)), generator=g, device="cuda").to(torch.bfloat16)
    w = w.t() if transposed else w
    with torch.no_grad():
        got = CU.frozen_matmul(x, w)
    want = x.float() @ w.float()
    assert got.shape == want.shape and got.is_contiguous()
    # one bf16 rounding (half a unit of 2^-8) and the order of up to 128 fp32 additions
    assert ((got.float() - want).abs() <= 2 ** -8 * want.abs() + 1e-4).all()


@pytest.mark.parametrize("shape", [(0, 48), (2, 0)])
def test_products_of_an_empty_batch(CU, dev, shape):
    w, a_w, b_w, _, _, _ = lora_case(dev, 7)
    x, gy = (torch.zeros(*shape, n, device=dev, dtype=BF16) for n in (w.shape[1], w.shape[0]))
    with torch.no_grad():
        assert CU.frozen_matmul(x, w.t()).shape == gy.shape
        y, main, xa = CU.lora_forward(w, None, a_w.T, b_w.T, None, x)
        assert y.shape == main.shape == gy.shape and xa.shape == (*shape, 16)
        ga, gb, gx = CU.lora_backward(w, None, a_w.T, b_w.T, x, xa, gy)
    assert gx.shape == x.shape and ga.shape[-2:] == a_w.T.shape and gb.shape[-2:] == b_w.T.shape


@pytest.mark.parametrize("M,n_in,n_out", [(96, 256, 4096), (5, 256, 4096), (2048, 13824, 64), (2048, 64, 11008)])
def test_backward_and_forward_of_a_projection_on_either_side_of_the_rules(CU, dev, M, n_in, n_out):
    """One call of the native host side each: few rows against a long contraction, and products in whole rounds (forward of the
    last shape, backward of the one before it)."""
    w, a_w, b_w, _, x, gy = lora_case(dev, 9, B=1, M=M, n_in=n_in, n_out=n_out)
    with torch.no_grad():
        y, main, xa = CU.lora_forward(w, None, a_w.T, b_w.T, None, x)
        gx = CU.lora_backward(w, None, a_w.T, b_w.T, x, xa, gy)[2]
    X, Wd, G = x.double(), w.double(), gy.double()
    assert_close_bf16(main, X @ Wd.T, what="frozen part")
    assert_close_bf16(y, X @ Wd.T + (X @ a_w.double().T) @ b_w.double().T, what="projection output")
    assert_close_bf16(gx, G @ Wd + (G @ b_w.double()) @ a_w.double(), what="grad x")


@pytest.mark.parametrize("shape", [(2, 48, 224), (1, 48, 256), (2, 47, 256)])
def test_a_running_sum_of_another_shape_is_refused(CU, dev, shape):
    w, a_w, b_w, _, x, gy = lora_case(dev, 13)
    xa = x @ a_w.T
    with torch.no_grad(), pytest.raises(ValueError, match="residual"):
        CU.lora_backward(w, None, a_w.T, b_w.T, x, xa, gy, accumulate=torch.zeros(*shape, device=dev, dtype=BF16))


@pytest.mark.parametrize("M,n_in,n_out", [(48, 256, 384), (96, 256, 4096), (2048, 64, 11008), (2048, 11008, 64)])
def test_products_under_autocast(CU, dev, M, n_in, n_out):
    """Autocast to float16 makes the products float16, as torch's own; autocast to bfloat16 changes nothing."""
    w, a_w, b_w, _, x, gy = lora_case(dev, 11, B=1, M=M, n_in=n_in, n_out=n_out)
    with torch.no_grad():
        plain = CU.lora_forward(w, None, a_w.T, b_w.T, None, x)
        plain_back = CU.lora_backward(w, None, a_w.T, b_w.T, x, plain[2], gy)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert all(torch.equal(a, b) for a, b in zip(CU.lora_forward(w, None, a_w.T, b_w.T, None, x), plain))
            assert all(torch.equal(a, b) for a, b in zip(CU.lora_backward(w, None, a_w.T, b_w.T, x, plain[2], gy), plain_back))
        with torch.autocast("cuda", dtype=torch.float16):
            y, main, _ = CU.lora_forward(w, None, a_w.T, b_w.T, None, x)
            ga, gb, gx = CU.lora_backward(w, None, a_w.T, b_w.T, x, plain[2], gy)
            assert CU.frozen_matmul(x, w.t()).dtype == CU.lora_parts(w, None, a_w.T, None, x)[0].dtype == torch.float16
    assert y.dtype == main.dtype == gx.dtype == torch.float16
    for a, b, what in zip((y, main, ga, gb, gx), (plain[0], plain[1], *plain_back), ("output", "frozen part", "grad A", "grad B", "grad x")):
        assert_close_bf16(a, b, what=what)
