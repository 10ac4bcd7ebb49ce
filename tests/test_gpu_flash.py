"""Map-free attention on the GPU against float64 of the same formulas."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def reference(q, k, v, g, causal, given_o=None):
    """Output, log-sum-exps and gradients in float64, from the bf16 operands; the gradients take `given_o` for the output."""
    n_rep = q.shape[1] // k.shape[1]
    q, k, v, g = (t.double() for t in (q, k, v, g))
    kr, vr = k.repeat_interleave(n_rep, 1), v.repeat_interleave(n_rep, 1)
    s = (q @ kr.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    if causal:
        n = s.shape[-1]
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    lse = torch.logsumexp(s, -1)
    p = (s - lse[..., None]).exp()
    o = p @ vr
    dp = g @ vr.transpose(-1, -2).contiguous()
    ds = p * (dp - (g * (o if given_o is None else given_o.double())).sum(-1, keepdim=True)) / math.sqrt(q.shape[-1])
    group = lambda t: t.unflatten(1, (k.shape[1], n_rep)).sum(2)                      # noqa: E731
    return o, lse, ds @ kr, group(ds.transpose(-1, -2).contiguous() @ q), group(p.transpose(-1, -2).contiguous() @ g)


# sizes around the tiles: 32 query rows a wave, 128 a workgroup, 64 keys a step
@pytest.mark.parametrize("s", [1, 31, 64, 65, 127, 128, 129, 200, 385])
@pytest.mark.parametrize("b,h,kv,d", [(1, 2, 2, 128), (2, 8, 2, 128), (3, 3, 1, 64), (1, 16, 8, 64)])
@pytest.mark.parametrize("causal", [True, False])
def test_flash_attention(b, h, kv, d, s, causal):
    from hyclora_amd.operators.flash_kernels import flash_backward, flash_forward
    gen = torch.Generator(device="cuda").manual_seed(s * 7 + h + d)
    hidden = lambda heads: torch.randn(b, s, heads, d, generator=gen, device="cuda").to(BF16).transpose(1, 2)      # noqa: E731
    q, k, v, g = hidden(h), hidden(kv), hidden(kv), hidden(h)
    q = (q * 2).to(BF16)
    want = reference(q, k, v, g, causal)
    o, lse = flash_forward(q, k, v, causal)
    grads = flash_backward(g, q, k, v, o, lse, causal)
    assert (lse.double() - want[1]).abs().max() < 1e-4              # fp32 sums of exponentials of fp32 scores
    # bf16 probabilities and score gradients (relative 2^-9 each, random in sign) and one bf16 rounding of the result:
    # 2-norm relative errors of about 2^-9 * sqrt(2); four times that is allowed
    for got, ref, name in zip((o,) + grads, (want[0],) + want[2:], ("o", "grad_q", "grad_k", "grad_v")):
        assert got.shape == ref.shape
        err = (got.double() - ref).norm() / ref.norm().clamp_min(1e-30) if ref.norm() > 1e-6 else (got.double() - ref).norm()
        assert err < 4 * 2 ** -8.5, (name, err.item())
    again = flash_backward(g, q, k, v, o, lse, causal)
    assert all(torch.equal(x, y) for x, y in zip(grads, again))


def check(got, want):
    for x, ref, name in zip(got, want, ("o", "grad_q", "grad_k", "grad_v")):
        assert x.shape == ref.shape
        err = (x.double() - ref).norm() / ref.norm()
        assert err < 4 * 2 ** -8.5, (name, err.item())              # as above


@pytest.mark.parametrize("s,h,kv", [(8192, 2, 1), (5001, 1, 1)])
def test_long_sequences(s, h, kv):
    from hyclora_amd.operators.flash_kernels import flash_backward, flash_forward
    gen = torch.Generator(device="cuda").manual_seed(s)
    hidden = lambda heads: torch.randn(1, s, heads, 128, generator=gen, device="cuda").to(BF16).transpose(1, 2)      # noqa: E731
    q, k, v, g = hidden(h), hidden(kv), hidden(kv), hidden(h)
    o, lse = flash_forward(q, k, v)
    want = reference(q, k, v, g, True)
    assert (lse.double() - want[1]).abs().max() < 1e-4
    check((o,) + flash_backward(g, q, k, v, o, lse), (want[0],) + want[2:])


@pytest.mark.parametrize("layout", ["heads", "odd", "wide"])
def test_operands_in_any_layout(layout):
    """[B, H, S, D] in memory, an address that is no multiple of 16 bytes, a slice of a wider tensor: copied first, same results."""
    from hyclora_amd.operators.flash_kernels import flash_backward, flash_forward
    b, h, kv, s, d = 2, 4, 2, 200, 128
    gen = torch.Generator(device="cuda").manual_seed(3)
    hidden = lambda heads: torch.randn(b, s, heads, d, generator=gen, device="cuda").to(BF16).transpose(1, 2)      # noqa: E731
    plain = hidden(h), hidden(kv), hidden(kv), hidden(h)

    def lay(t):
        if layout == "heads":
            return t.contiguous()
        if layout == "odd":
            hidden_t = t.transpose(1, 2)
            return torch.empty(t.numel() + 1, device="cuda", dtype=BF16)[1:].view(hidden_t.shape).copy_(hidden_t).transpose(1, 2)
        return torch.empty(*t.shape[:-1], 2 * d, device="cuda", dtype=BF16)[..., d:].copy_(t)
    q, k, v, g = (lay(t) for t in plain)
    o, lse = flash_forward(q, k, v)
    o2, lse2 = flash_forward(*plain[:3])
    assert torch.equal(o, o2) and torch.equal(lse, lse2)
    for x, y in zip(flash_backward(g, q, k, v, lay(o), lse), flash_backward(plain[3], *plain[:3], o2, lse2)):
        assert torch.equal(x, y)


def test_operands_that_are_not_on_the_gpu_are_refused():
    """Before anything is launched: a host address would be read on the device."""
    from hyclora_amd.operators.flash_kernels import flash_backward, flash_forward, flash_supported
    from hyclora_amd.operators.map_kernels import MapAttention, map_backward, map_supported
    q, k, v, g = (torch.zeros(1, 2, 64, 64, device="cuda", dtype=BF16) for _ in range(4))
    lse = torch.zeros(1, 2, 64, device="cuda")
    lists = torch.empty(0, device="cuda", dtype=torch.int64), torch.empty(0, device="cuda", dtype=BF16), torch.zeros(3, device="cuda", dtype=torch.int64)
    mask = torch.zeros(1, 1, 64, 64, device="cuda", dtype=BF16)
    assert flash_supported(q, k, v) and map_supported(q, k, v, mask) and not map_supported(q, k, v, mask.cpu())
    for i in range(3):
        ops = [t.cpu() if j == i else t for j, t in enumerate((q, k, v))]
        assert not flash_supported(*ops) and not map_supported(*ops, mask)
        for call in (lambda: flash_forward(*ops), lambda: flash_backward(g, *ops, q, lse), lambda: MapAttention(*ops, mask), lambda: map_backward(g, *ops, *lists)):
            with pytest.raises(ValueError):
                call()
    with pytest.raises(ValueError):
        MapAttention(q, k, v, mask.cpu())
    att = MapAttention(q, k, v, threshold=torch.zeros(()))
    for offsets in (torch.empty(3, dtype=torch.int64), torch.empty(2, device="cuda", dtype=torch.int64), torch.empty(3, device="cuda", dtype=torch.int32)):
        with pytest.raises(ValueError):
            att.entries(8, offsets)
    for call in (lambda: flash_backward(g.cpu(), q, k, v, q, lse), lambda: flash_backward(g, q, k, v, q.cpu(), lse), lambda: flash_backward(g, q, k, v, q, lse.cpu()),
                 lambda: map_backward(g.cpu(), q, k, v, *lists), *(lambda i=i: map_backward(g, q, k, v, *(t.cpu() if j == i else t for j, t in enumerate(lists))) for i in range(3))):
        with pytest.raises(RuntimeError, match="GPU only"):
            call()


@pytest.mark.parametrize("causal", [True, False])
def test_backward_of_another_output(causal):
    """The layers hand in the dequantised output, a few percent off the forward's."""
    from hyclora_amd.operators.flash_kernels import flash_backward, flash_forward
    b, h, kv, s, d = 2, 4, 2, 333, 128
    gen = torch.Generator(device="cuda").manual_seed(4)
    hidden = lambda heads: torch.randn(b, s, heads, d, generator=gen, device="cuda").to(BF16).transpose(1, 2)      # noqa: E731
    q, k, v, g = hidden(h), hidden(kv), hidden(kv), hidden(h)
    o, lse = flash_forward(q, k, v, causal)
    given = (o.float() + 0.05 * hidden(h).float()).to(BF16)
    want = reference(q, k, v, g, causal, given)
    check((o,) + flash_backward(g, q, k, v, given, lse, causal), (want[0],) + want[2:])
