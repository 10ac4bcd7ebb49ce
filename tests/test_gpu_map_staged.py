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


@pytest.mark.parametrize("kept,room_mb", [(0.01, 28), (0.05, 68)])
def test_scratch_that_does_not_fit(kept, room_mb):
    """Where memory is left for the lists but not for a quarter of the map (32 of 128 MB) as well, the map is read twice: first the scratch
    itself does not fit, then the lists do not fit beside it."""
    import hyclora_amd  # noqa: F401
    from hyclora_amd.operators import compress_function as cf
    x = torch.rand(1 << 26, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)).to(BF16)
    thr = torch.tensor(1 - kept, device="cuda")
    want = [t.cpu() for t in cf.compress_attention_map(x, thr)]
    nnz = want[0].numel()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (room_mb << 20)) / total)
        for capacity in (None, nnz):
            got = cf.compress_attention_map(x, thr, capacity=capacity)
            assert all(torch.equal(a.cpu(), b) for a, b in zip(got[:3], want))
            del got
            torch.cuda.empty_cache()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
