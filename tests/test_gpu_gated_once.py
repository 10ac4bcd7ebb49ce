"""The gated product in one kernel each way for the layers that round silu once, against the kernels it stands for: the same
operations in the same order, so the same bits."""
import pytest
import torch

from hyclora_amd.operators import lora_kernels
from hyclora_amd.operators._fuse import fuse_backward
from hyclora_amd.operators.compress_function import get_statistics_only_quant
from hyclora_amd.operators.silu_kernels import silu_hadamard, silu_hadamard_backward, silu_once_hadamard
from hyclora_amd.operators.triton_fuse_lora_silu_hadamard_forward_kernels import triton_fuse_silu_forward


@pytest.mark.gpu
@pytest.mark.parametrize("q_bit", [2, 4, 8])
@pytest.mark.parametrize("t,n,r", [(1, 32, 4), (15, 160, 16), (97, 1024, 16), (128, 1056, 32), (2048, 5504, 16), (31, 128, 64)])
def test_same_bits_as_the_separate_kernels(t, n, r, q_bit):
    g = torch.Generator(device="cuda").manual_seed(t + n + q_bit)
    rn = lambda *s, sc=1.0: (sc * torch.randn(s, generator=g, device="cuda")).bfloat16()       # noqa: E731
    x1, x2, grad = rn(1, t, n, sc=3.0), rn(1, t, n), rn(1, t, n)
    xa1, xa2, b1, b2 = rn(1, t, r), rn(1, t, r), rn(n, r, sc=0.1).T, rn(n, r, sc=0.1).T
    s1, s2 = (get_statistics_only_quant(x, q_bit, "per-channel") for x in (x1, x2))
    items = [dict(x_main=x1, xa=xa1, b=b1, scale=s1, zero_point=None, rope=None), dict(x_main=x2, xa=xa2, b=b2, scale=s2, zero_point=None, rope=None)]
    (q1, y1), (q2, y2) = lora_kernels.lora_add_quant_group(items, q_bit, inplace=False)
    got = triton_fuse_silu_forward(xa1, b1, x1, s1, xa2, b2, x2, s2, q_bit)
    for a, b in zip(got, (q1, q2, silu_hadamard(y1, y2))):
        assert torch.equal(a, b)
    y1, y2 = lora_kernels.lora_add_restore_group([dict(q=q1, scale=s1, xa=xa1, b=b1, zero_point=None, rope=None),
                                                  dict(q=q2, scale=s2, xa=xa2, b=b2, zero_point=None, rope=None)], q_bit)
    got = fuse_backward(xa1, b1, q1, s1, xa2, b2, q2, s2, grad, q_bit, round_once=True)
    for a, b in zip(got, (silu_once_hadamard(y1, y2), *silu_hadamard_backward(y1, y2, grad))):
        assert torch.equal(a, b)
