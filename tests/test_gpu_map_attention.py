"""Attention through a sparsely kept map against the separate operators it replaces: the kept entries bit for bit those of the
compaction of the dense map it writes itself, everything else against float64 of the same formulas."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def operands(b, h, kv, s, d, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    hidden = lambda heads: (1.4 * torch.randn(b, s, heads, d, generator=gen, device="cuda")).to(BF16).transpose(1, 2)     # noqa: E731
    return hidden(h), hidden(kv), hidden(kv), hidden(h)


def masks(kind, b, s):
    low = torch.finfo(BF16).min
    causal = torch.ones(s, s, dtype=torch.bool, device="cuda").triu(1)[None]
    left = torch.arange(s, device="cuda")[None] < torch.tensor([(s * i) // (b + 1) for i in range(b)], device="cuda")[:, None]
    if kind == "none":
        return None
    if kind == "causal":
        return torch.zeros(1, 1, s, s, device="cuda", dtype=BF16).masked_fill_(causal, float("-inf"))
    if kind == "padded":          # left-padded causal batch with a finite mask value: the padded rows attend to nothing of their own
        return torch.zeros(b, 1, s, s, device="cuda", dtype=BF16).masked_fill_((causal | left[:, None, :])[:, None], low)
    if kind == "keys":            # one mask row for all queries
        return torch.zeros(b, 1, 1, s, device="cuda", dtype=BF16).masked_fill_(left.flip(1)[:, None, None], low)
    gen = torch.Generator(device="cuda").manual_seed(5)
    if kind == "low":             # values on both sides of -1e30, where keys begin to cost nothing; a third of the rows have only such
        pick = lambda values, *shape: torch.tensor(values, device="cuda")[torch.randint(len(values), shape, generator=gen, device="cuda")]     # noqa: E731
        m = pick([-0.9e30, -1.1e30, -3e30, -5e31, -1e38, low], b, 1, s, s)
        m[:, :, :, s // 2:] = low
        rows = torch.arange(s, device="cuda") // 40 % 3
        m[:, :, rows == 1, : s // 4] = pick([0.0, -2.0, -0.4e30], b, 1, int((rows == 1).sum()), s // 4)
        m[:, :, rows == 2] = pick([-2e30, -3e30, low], b, 1, int((rows == 2).sum()), s)
        return m.to(BF16)
    return torch.randn(1, 1, s, s, generator=gen, device="cuda").to(BF16)      # a bias


def dense(q, k, mask):
    """The map with the layers' roundings, from float64 scores."""
    n_rep = q.shape[1] // k.shape[1]
    kt = k.repeat_interleave(n_rep, 1).double().transpose(-1, -2).contiguous()
    t = (q.double() @ kt).to(BF16)
    t = (t.float() * (1.0 / math.sqrt(q.shape[-1]))).to(BF16)
    if mask is not None:
        t = (t.float() + mask.float()).to(BF16)
    return torch.softmax(t.double(), -1)


def rel(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm().clamp_min(1e-30)).item()


@pytest.mark.parametrize("kind", ["none", "causal", "padded", "keys", "bias", "low"])
@pytest.mark.parametrize("b,h,kv,s,d", [(1, 2, 2, 8, 64), (2, 4, 4, 32, 128), (2, 3, 1, 72, 64), (3, 8, 2, 136, 128), (1, 4, 2, 200, 128),
                                        (2, 2, 2, 256, 64), (1, 2, 1, 520, 128), (1, 1, 1, 4096, 64)])
def test_forward_and_kept_entries(b, h, kv, s, d, kind):
    from hyclora_amd.operators.compress_function import compress_attention_map, get_statistics_softmax
    from hyclora_amd.operators.map_kernels import MapAttention
    q, k, v, _ = operands(b, h, kv, s, d, seed=s + h)
    mask = masks(kind, b, s)
    full = MapAttention(q, k, v, mask, want_map=True)
    want = dense(q, k, mask)
    # one bf16 rounding of a value that a score's last bit may move (2^-9 of a score of a few units): a few 2^-9 in the 2-norm
    assert rel(full.map, want) < 8 * 2 ** -9
    o = full.map.double() @ v.repeat_interleave(h // kv, 1).double().contiguous()
    assert rel(full.o, o) < 2 ** -8
    thr = get_statistics_softmax(full.map, 0.05)
    for threshold in (thr, torch.zeros((), device="cuda"), torch.full((), -1.0, device="cuda"), torch.full((), 2.0, device="cuda")):
        idx, val, seg = compress_attention_map(full.map, threshold)
        part = MapAttention(q, k, v, mask, threshold=threshold)
        assert torch.equal(part.o, full.o)
        n = idx.numel()
        for capacity in (n, n + 100, n // 2):
            idx2, val2, seg2, count = part.bounded_entries(capacity)
            assert count.value() == n and torch.equal(seg2, seg)
            m = min(n, capacity)
            assert torch.equal(idx2[:m], idx[:m]) and torch.equal(val2[:m], val[:m])


@pytest.mark.parametrize("b,h,s", [(33, 16, 136), (5, 9, 1000), (260, 1, 8), (70000, 2, 8)])
def test_entries_of_many_rows(b, h, s):
    """More rows than a workgroup of the scan takes, starting inside a head and inside its blocks of 32 rows."""
    from hyclora_amd.operators.compress_function import compress_attention_map
    from hyclora_amd.operators.map_kernels import MapAttention
    q, k, v, _ = operands(b, h, h, s, 64, seed=s)
    mask = masks("keys", b, s)
    threshold = torch.full((), 0.1, device="cuda")
    idx, val, seg = compress_attention_map(MapAttention(q, k, v, mask, want_map=True).map, threshold)
    idx2, val2, seg2 = MapAttention(q, k, v, mask, threshold=threshold).entries(idx.numel())
    assert torch.equal(idx2, idx) and torch.equal(val2, val) and torch.equal(seg2, seg)


def test_very_many_rows_and_very_long_lists_go_through_memory():
    from hyclora_amd.operators.flash_kernels import flash_supported
    from hyclora_amd.operators.map_kernels import map_backward_supported, map_supported
    like = lambda b, h, s: torch.empty(1, device="cuda", dtype=BF16).expand(b, h, s, 64)          # noqa: E731
    q = like(2, 4, 512)
    idx = torch.empty(1, device="cuda", dtype=torch.int64)
    assert map_backward_supported(q, q, q, idx.expand((1 << 31) - 1)) and not map_backward_supported(q, q, q, idx.expand(1 << 31))
    for b, s, fits in ((70000, 8, True), ((1 << 22) // 4, 8, True), ((1 << 22) // 4 + 1, 8, False), ((1 << 22) // 64, 512, True), ((1 << 22) // 64 + 1, 512, False)):
        q = like(b, 4, s)
        assert map_supported(q, q, q) is fits
    for b, s, fits in (((1 << 23) // 4, 1, True), ((1 << 23) // 4 + 1, 1, False), ((1 << 23) // 16, 500, True), ((1 << 23) // 16 + 1, 500, False)):
        q = like(b, 4, s)
        assert flash_supported(q, q, q) is fits


def same_bits(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("s", [8, 72, 96, 128, 200])
def test_rows_without_a_finite_sum_keep_nothing_past_their_end(s):
    """Rows of nothing but -inf and rows of NaN scores: every one of their S entries is kept (NaN is), none past the row."""
    from hyclora_amd.operators.compress_function import compress_attention_map
    from hyclora_amd.operators.map_kernels import MapAttention
    b, h = 2, 3
    q, k, v, _ = operands(b, h, h, s, 64, seed=s)
    mask = torch.zeros(b, 1, s, s, device="cuda", dtype=BF16)
    mask[0, :, 0] = mask[1, :, s - 1] = mask[1, :, s // 2] = float("-inf")
    q = q.clone()
    q[0, 1, s - 1] = q[1, 2, 3] = float("nan")
    empty = mask.isinf().all(-1).expand(b, h, s) | q.isnan().any(-1)
    full = MapAttention(q, k, v, mask, want_map=True)
    assert torch.equal(full.map.isnan(), empty[..., None].expand(b, h, s, s))
    for threshold in (0.05, 0.0, -1.0, 2.0):
        threshold = torch.full((), threshold, device="cuda")
        idx, val, seg = compress_attention_map(full.map, threshold)
        part = MapAttention(q, k, v, mask, threshold=threshold)
        idx2, val2, seg2, count = part.bounded_entries(idx.numel() + 100)
        assert count.value() == idx.numel() and torch.equal(seg2, seg)
        assert torch.equal(idx2[:idx.numel()], idx) and same_bits(val2[:idx.numel()], val)


@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("where", ["q", "k", "v", "mask"])
@pytest.mark.parametrize("kind", ["causal", "padded", "keys"])
@pytest.mark.parametrize("h,kv,s,d", [(2, 2, 72, 64), (4, 2, 200, 128), (2, 1, 520, 64)])
def test_values_that_are_not_finite_spread_as_over_a_dense_map(h, kv, s, d, kind, where, value):
    """A masked key counts as well: its weight is 0, and 0 times an infinite value is NaN.  The dense map of the operators that go
    through memory says which elements are NaN."""
    from hyclora_amd.operators.compress_function import compress_attention_map
    from hyclora_amd.operators.map_kernels import MapAttention
    from hyclora_amd.operators.softmax_kernels import softmax_forward
    b = 3
    q, k, v, _ = (t.clone() for t in operands(b, h, kv, s, d, seed=s + h))
    mask = masks(kind, b, s)
    mask = mask.expand(mask.shape[0], 1, s, s).clone()
    if where == "mask":
        mask[-1, 0, s // 3, s - 2] = value
    else:
        {"q": q, "k": k, "v": v}[where][1, 0, s - 2, 5] = value
    kr, vr = (t.repeat_interleave(h // kv, 1).float() for t in (k, v))
    scores = (q.float() @ kr.transpose(-1, -2).contiguous()).to(BF16)
    want = softmax_forward(scores, 1.0 / math.sqrt(d), mask)
    o = want.float() @ vr.contiguous()
    full = MapAttention(q, k, v, mask, want_map=True)
    for got, ref in ((full.map, want), (full.o, o)):
        assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
        finite = ref.isfinite()
        assert rel(got[finite], ref[finite]) < 8 * 2 ** -9       # as in test_forward_and_kept_entries
    threshold = torch.full((), 0.02, device="cuda")
    part = MapAttention(q, k, v, mask, threshold=threshold)
    assert same_bits(part.o, full.o)
    idx, val, seg = compress_attention_map(full.map, threshold)
    idx2, val2, seg2, count = part.bounded_entries(idx.numel() + 9)
    assert count.value() == idx.numel() and torch.equal(seg2, seg)
    assert torch.equal(idx2[:idx.numel()], idx) and same_bits(val2[:idx.numel()], val)


def dense_backward(go, q, k, v, a):
    """The gradients through the dense map `a`, from float64 products with the layers' roundings."""
    kv, n_rep, d = k.shape[1], q.shape[1] // k.shape[1], q.shape[-1]
    kr, vr = (t.repeat_interleave(n_rep, 1).double().contiguous() for t in (k, v))
    g = (go.double() @ vr.transpose(-1, -2).contiguous()).to(BF16)
    dsum = (a.float() * g.float()).to(BF16).double().sum(-1, keepdim=True)
    ds = (((g.double() - dsum) * a.double()).to(BF16).float() / math.sqrt(d)).to(BF16).double()
    group = lambda t: t.unflatten(1, (kv, n_rep)).sum(2)                              # noqa: E731
    return ds @ kr, group(ds.transpose(-1, -2).contiguous() @ q.double()), group(a.double().transpose(-1, -2).contiguous() @ go.double())


@pytest.mark.parametrize("ratio", [0.0, 0.05, 1.0])
@pytest.mark.parametrize("b,h,kv,s,d", [(1, 2, 2, 8, 64), (2, 4, 4, 32, 128), (2, 3, 1, 72, 64), (3, 8, 2, 136, 128), (1, 4, 2, 200, 128),
                                        (2, 2, 2, 256, 64), (1, 2, 1, 520, 128), (1, 1, 1, 4096, 64)])
def test_backward_from_kept_entries(b, h, kv, s, d, ratio):
    from hyclora_amd.operators.compress_function import compress_attention_map, get_statistics_softmax, restore_attention_map
    from hyclora_amd.operators.map_kernels import MapAttention, map_backward
    q, k, v, go = operands(b, h, kv, s, d, seed=s + h)
    full = MapAttention(q, k, v, masks("causal", b, s), want_map=True)
    thr = torch.full((), 2.0, device="cuda") if ratio == 0 else torch.zeros((), device="cuda") if ratio == 1 else \
        get_statistics_softmax(full.map, ratio)
    idx, val, seg = compress_attention_map(full.map, thr)
    got = map_backward(go, q, k, v, idx, val, seg)
    want = dense_backward(go, q, k, v, restore_attention_map(idx, val, seg, (b, h, s, s)))
    for x, w, name in zip(got, want, ("grad_q", "grad_k", "grad_v")):
        assert x.shape == w.shape
        # the same bf16 operands on both sides, up to last bits of g; fp32 sums and one rounding
        assert (rel(x, w) < 2 ** -8 if w.norm() > 0 else x.abs().max() == 0), (name, rel(x, w))
    again = map_backward(go, q, k, v, torch.cat([idx, idx.new_full((7,), -1)]), torch.cat([val, val.new_zeros(7)]), seg)
    assert all(torch.equal(x, y) for x, y in zip(got, again))          # room past the entries is not read


@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("where", ["grad_o", "q", "k", "v", "map"])
@pytest.mark.parametrize("threshold", [2.0, 0.1, 0.0])
@pytest.mark.parametrize("h,kv,s,d", [(2, 2, 72, 64), (4, 2, 200, 128), (2, 1, 520, 64)])
def test_gradients_that_are_not_finite_spread_as_over_a_dense_map(h, kv, s, d, threshold, where, value):
    """Entries that are not kept count as well: their 0 times an infinite operand, or an infinite gradient of the map times their
    0, is NaN.  At 2.0 nothing is kept, at 0.1 the later rows keep little or nothing."""
    from hyclora_amd.operators.compress_function import compress_attention_map, restore_attention_map
    from hyclora_amd.operators.map_kernels import MapAttention, map_backward
    b = 3
    q, k, v, go = (t.clone() for t in operands(b, h, kv, s, d, seed=s + h))
    amap = MapAttention(q, k, v, masks("causal", b, s), want_map=True).map
    if where == "map":
        amap[1, 0, s - 3, s // 2] = value                      # kept by a threshold below infinity
    else:
        {"grad_o": go, "q": q, "k": k, "v": v}[where][1, 0, s - 3, 5] = value
    idx, val, seg = compress_attention_map(amap, torch.full((), threshold, device="cuda"))
    got = map_backward(go, q, k, v, idx, val, seg)
    want = dense_backward(go, q, k, v, restore_attention_map(idx, val, seg, (b, h, s, s)))
    for x, w, name in zip(got, want, ("grad_q", "grad_k", "grad_v")):
        finite = w.isfinite()
        assert torch.equal(x.isfinite(), finite), name
        assert rel(x[finite], w[finite]) < 2 ** -8 if w[finite].norm() > 0 else x[finite].abs().max() == 0, name


@pytest.mark.parametrize("s", [72, 96, 200])
def test_gradients_of_rows_without_a_finite_sum(s):
    """Lists of rows that are NaN throughout, at lengths with a partial last tile and a partial last block of rows."""
    from hyclora_amd.operators.compress_function import restore_attention_map
    from hyclora_amd.operators.map_kernels import MapAttention, map_backward
    b, h, d = 2, 3, 64
    q, k, v, go = operands(b, h, h, s, d, seed=s)
    mask = masks("causal", b, s).expand(b, 1, s, s).clone()
    mask[0, :, s - 1] = mask[1, :, 5] = float("-inf")
    part = MapAttention(q, k, v, mask, threshold=torch.full((), 0.1, device="cuda"))
    idx, val, seg = part.entries(int(part.entries(0)[2][-1]))
    got = map_backward(go, q, k, v, idx, val, seg)
    want = dense_backward(go, q, k, v, restore_attention_map(idx, val, seg, (b, h, s, s)))
    for x, w in zip(got, want):
        assert torch.equal(x.isfinite(), w.isfinite()) and rel(x[w.isfinite()], w[w.isfinite()]) < 2 ** -8


@pytest.mark.parametrize("q_bit,b,s,fits", [(2, 1, 1016, False), (2, 1, 1024, True), (2, 2, 512, True), (2, 3, 64, False), (4, 1, 64, True), (8, 1, 8, True),
                                            (None, 1, 64, True)])
def test_short_two_bit_steps_stay_with_the_library(monkeypatch, q_bit, b, s, fits):
    from hyclora_amd.models import fused_decoder_layer as L
    monkeypatch.setattr(L, "map_supported", lambda *a: True)
    q = torch.empty(b, 2, s, 64)
    assert L.map_kernels_fit(q, q, q, None, q_bit) is fits
