"""Compaction of a map through the entries that its count left behind: segments with no, few, exactly the most and more entries than are
kept in scratch memory, ragged ends, bounded and exact lists, against the oracle's order of the kept elements."""
import pytest
import torch

from helpers import BF16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 8, 4095, 4096, 4097, 5 * 4096 + 13, 40 * 4096])
@pytest.mark.parametrize("compare_abs", [False, True])
def test_segments_of_every_density(n, compare_abs):
    import hyclora_amd  # noqa: F401
    from hyclora_amd.operators import compress_function as cf
    g = torch.Generator().manual_seed(n)
    x = torch.rand(n, generator=g) * 0.5
    counts = [0, 1, 511, 512, 513, 1024, 1025, 4096, 200]
    for s in range(-(-n // 4096)):
        here = min(4096, n - s * 4096)
        at = torch.randperm(here, generator=g)[:min(counts[s % len(counts)], here)] + s * 4096
        x[at] += 1.0
    x[::3] *= -1 if compare_abs else 1
    x[n // 2] = float("nan")
    x = x.to(BF16)
    thr = torch.tensor(0.75)
    mask = ((x.abs() if compare_abs else x) > thr.to(BF16)) | x.isnan()
    want = mask.nonzero().flatten()
    nnz = want.numel()
    for capacity in (None, nnz + 5, max(nnz - 3, 0), 0):
        out = cf.compress_attention_map(x.cuda(), thr.cuda(), compare_abs=compare_abs, capacity=capacity)
        idx, val, seg = (t.cpu() for t in out[:3])
        fit = nnz if capacity is None else min(nnz, capacity)
        assert int(seg[-1]) == nnz and (capacity is None or out[3].value() == nnz)
        assert torch.equal(idx[:fit], want[:fit]) and torch.equal(val[:fit].view(torch.int16), x[want[:fit]].view(torch.int16))
        # the lists again, exact, from the offsets alone
        again = cf.compress_attention_map(x.cuda(), thr.cuda(), out[2], compare_abs=compare_abs)
        assert torch.equal(again[0].cpu(), want) and torch.equal(again[1].cpu().view(torch.int16), x[want].view(torch.int16))
