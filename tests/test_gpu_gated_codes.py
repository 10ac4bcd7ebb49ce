"""The gated product of layers that keep every activation as codes: bit for bit the separate passes, over every bf16 gate, at rows around
a wave's and columns around a tile's and the smallest."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def bits(t):
    return torch.where(t.isnan(), torch.full_like(t, float("nan")), t).view(torch.int16)


@pytest.mark.parametrize("q_bit", [2, 4, 8])
@pytest.mark.parametrize("shape", [(1, 1, 32), (1, 33, 544), (3, 21, 1024), (2, 64, 512), (1, 65541, 32)])       # the last: 8 rows a wave
def test_against_the_separate_passes(shape, q_bit):
    import hyclora_amd  # noqa: F401
    from hyclora_amd.operators import silu_kernels as K
    from hyclora_amd.operators.compress_function import compression_quantization, decompression_dequantization
    n = shape[-1]
    g = torch.Generator().manual_seed(n + q_bit)
    count = shape[0] * shape[1] * n
    every = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)       # with infinities and NaN
    gate = every.repeat(-(-count // 65536))[:count] if count >= 65536 else torch.randn(count, generator=g).to(torch.bfloat16) * 3
    gate = gate.reshape(shape).cuda()
    up, grad = ((torch.randn(shape, generator=g) * 2).to(torch.bfloat16).cuda() for _ in range(2))
    scales = [(torch.rand(n, generator=g) * 0.1 + 1e-3).to(torch.bfloat16).cuda() for _ in range(4)]
    scales[2][::7] = 0.0
    *codes, out = K.silu_hadamard_codes(gate, up, scales, q_bit)
    fn = F.silu(gate)
    want = (gate, up, fn, up * fn)
    assert torch.equal(bits(out), bits(want[3]))
    for t, s, q in zip(want, scales, codes):
        assert torch.equal(q, compression_quantization(t, s, q_bit))
    dq = [decompression_dequantization(q, s, q_bit) for q, s in zip(codes, scales)]
    gg, gu = K.silu_hadamard_backward_codes(codes[:3], scales[:3], grad, q_bit)
    assert torch.equal(bits(gg), bits(K.silu_backward(dq[0], grad * dq[1])))
    assert torch.equal(bits(gu), bits(grad * dq[2]))


def test_what_it_does_not_take():
    import hyclora_amd  # noqa: F401
    from hyclora_amd.operators import silu_kernels as K
    x = torch.zeros(2, 4, 40, dtype=torch.bfloat16, device="cuda")
    s = [torch.ones(40, dtype=torch.bfloat16, device="cuda")] * 4
    assert K.silu_hadamard_codes(x, x, s, 8) is None                               # columns no multiple of 32
    y = x[..., :32].contiguous()
    assert K.silu_hadamard_codes(y.float(), y.float(), [t[:32].contiguous() for t in s], 8) is None
    assert K.silu_hadamard_codes(y, y, s, 8) is None                               # steps of another length
