"""Outlier lists with positions that have no column of their own, and codes with zero points at the edges of the rule without a division."""
import pytest
import torch

from helpers import BF16
from oracle import hyc_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def N():
    import hyclora_amd  # noqa: F401
    from hyclora_amd import _lib
    return _lib.native()


# lists of one batch of 64 entries and more, up to and past the length whose unused positions the kernel clears
@pytest.mark.parametrize("k", [1, 2, 20, 63, 64, 65, 130, 256, 257])
@pytest.mark.parametrize("B,M,n", [(1, 1, 32), (2, 37, 512), (1, 70, 1056)])
def test_unused_list_positions_read_as_zeros(N, k, B, M, n):
    g = torch.Generator().manual_seed(k * 1000 + n)
    x = torch.randn(B, M, n, generator=g).to(BF16)
    s = O.scale_only_quant(x, 4)
    idx = torch.randint(-3, n + 5, (k,), generator=g)              # outside on both sides; repeated once k is large against n
    if k > 2:
        idx[k // 2] = idx[0] = 7                                   # a repeated one in any case
    poison = torch.full((B, M, k), float("nan"), dtype=BF16, device="cuda")
    del poison                                                     # what the allocator hands out next is not zeros
    kept, q = N.quantize(x.cuda(), s.cuda(), None, idx.cuda(), 4)
    want = torch.zeros(B, M, k, dtype=BF16)
    dense = x.clone()
    last = {int(c): i for i, c in enumerate(idx) if 0 <= c < n}
    for c, i in last.items():
        want[..., i] = x[..., c]
        dense[..., c] = 0
    assert torch.equal(kept.cpu(), want)
    assert torch.equal(q.cpu(), O.compress(dense, s, 4))


@pytest.mark.parametrize("q_bit", [2, 4, 8])
@pytest.mark.parametrize("B,M,n", [(1, 1, 32), (3, 11, 512), (1, 33, 544), (2, 64, 1024)])
@pytest.mark.parametrize("slow", [False, True])
def test_codes_with_zero_points(N, q_bit, B, M, n, slow):
    """Wave tiles that are full and not, one column per wave that takes the division (a tiny step, a zero point past 2^64) and none,
    with infinities, NaN and values at ties in the input."""
    g = torch.Generator().manual_seed(q_bit + n)
    x = torch.randn(B, M, n, generator=g) * 3
    s = (0.05 + torch.rand(n, generator=g)).to(BF16)
    z = torch.randint(-2 ** (q_bit - 1), 2 ** (q_bit - 1), (n,), generator=g).to(BF16)
    z[::5] += 0.5
    x[..., 3::7] = (torch.randint(-4, 4, x[..., 3::7].shape, generator=g) + 0.5) * s[3::7].float()      # near ties
    x = x.to(BF16)
    x[..., 1], x[..., 2], x[..., 5], x[..., 6] = float("inf"), float("-inf"), float("nan"), 3e38
    if slow:
        s[::97], z[9::131] = 1e-20, 1e25
    _, q = N.quantize(x.cuda(), s.cuda(), z.cuda(), None, q_bit)
    assert torch.equal(q.cpu(), O.compress(x, s, q_bit, z))


@pytest.mark.parametrize("B,M,n", [(1, 5, 32), (2, 37, 512), (1, 130, 1056)])
def test_strip_heights(N, B, M, n):
    """Results do not depend on the rows that a wave walks, with and without a list, with and without zero points."""
    from hyclora_amd import _lib
    g = torch.Generator().manual_seed(n)
    x = torch.randn(B, M, n, generator=g).to(BF16).cuda()
    s, z = (0.05 + torch.rand(n, generator=g)).to(BF16).cuda(), torch.randint(-8, 8, (n,), generator=g).to(BF16).cuda()
    idx = torch.randperm(n, generator=g)[:min(n, 70)].cuda()
    keys = ("quant_rows_per_wave", "dequant_rows_per_wave", "quant_outlier_rows_per_wave", "dequant_outlier_rows_per_wave")

    def call():
        kept, q = N.quantize(x, s, None, idx, 4)
        qz, qp = N.quantize(x, s, z, None, 4)[1], N.quantize(x, s, None, None, 4)[1]
        return kept, q, qz, qp, N.dequantize(q, s, None, kept, idx, 4), N.dequantize(qz, s, z, None, None, 4), N.dequantize(qp, s, None, None, None, 4)
    want = call()
    try:
        for rows in (1, 2, 3, 4, 8, 16):
            for key in keys:
                _lib.set_tuning(key, rows)
            assert all(torch.equal(a, b) for a, b in zip(call(), want)), rows
    finally:
        for key in keys:
            _lib.set_tuning(key, -1)
