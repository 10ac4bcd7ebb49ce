"""Rows of 2^28 channels, the widest that the entry points take, at 8 bits: the bytes of a row times 8 do not fit 32 bits.  Each call on two
rows against the calls on the single rows, whose addresses do not depend on a row's length."""
import pytest
import torch

from helpers import BF16

pytestmark = pytest.mark.gpu

N = 1 << 28


@pytest.fixture(scope="module")
def rows():
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.empty(1, 2, N, device="cuda", dtype=BF16).normal_(generator=g)
    scale = torch.empty(N, device="cuda", dtype=BF16).uniform_(0.01, 0.05, generator=g)
    yield x, x.flip(1).contiguous(), scale
    torch.cuda.empty_cache()


def halves(call, *whole):
    """call(operands) -> tensors [1, rows, ...], on both rows and on each"""
    both = call(*whole)
    for r in range(2):
        for t, one in zip(both, call(*(w[:, r:r + 1] for w in whole))):
            assert torch.equal(t[:, r:r + 1], one), f"row {r}"


def test_quantiser_and_dequantiser(rows):
    import hyclora_amd  # noqa: F401
    from hyclora_amd.operators import compress_function as cf
    x, _, scale = rows

    def call(x):
        q = cf.compression_quantization(x, scale, 8)
        return q, cf.decompression_dequantization(q, scale, 8)
    halves(call, x)


def test_gated_product_of_codes(rows):
    import hyclora_amd  # noqa: F401
    from hyclora_amd.operators import silu_kernels as K
    x, y, scale = rows
    scales = [scale] * 4

    def call(gate, up):
        done = K.silu_hadamard_codes(gate, up, scales, 8)
        return *done, *K.silu_hadamard_backward_codes(done[:3], scales[:3], up, 8)
    halves(call, x, y)


def test_lora_add_with_codes(rows):
    import hyclora_amd  # noqa: F401
    from hyclora_amd.operators import lora_kernels as lk
    x, _, scale = rows
    g = torch.Generator(device="cuda").manual_seed(2)
    b = torch.empty(4, N, device="cuda", dtype=BF16).normal_(0, 0.1, generator=g)
    xa = torch.empty(1, 2, 4, device="cuda", dtype=BF16).normal_(generator=g)

    def call(x, xa):
        q, y = lk.lora_add_quant(x, xa, b, scale, None, 8)
        return q, y, lk.lora_add_restore(q, scale, xa, b, None, 8)
    halves(call, x, xa)


def test_fused_gated_product(rows):
    import hyclora_amd  # noqa: F401
    from hyclora_amd.operators._fuse import fuse_backward, fuse_forward
    x, y, scale = rows
    g = torch.Generator(device="cuda").manual_seed(3)
    b = torch.empty(4, N, device="cuda", dtype=BF16).normal_(0, 0.1, generator=g)
    xa = torch.empty(1, 2, 4, device="cuda", dtype=BF16).normal_(generator=g)

    def call(x, y, xa):
        q1, q2, o = fuse_forward(xa, b, x, scale, xa, b, y, scale, 8)
        return q1, q2, o, *fuse_backward(xa, b, q1, scale, xa, b, q2, scale, y, 8)
    halves(call, x, y, xa)
