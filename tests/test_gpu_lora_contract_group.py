"""The rank-R products of several projections in one launch (hyc_lora_contract_group behind lora_backward_shared) against the
calls of the single projections, bit for bit, and the single calls at the edges of their row strips, planes and column
blocks against float64."""
import ctypes

import pytest
import torch

from helpers import BF16, assert_close_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import hyclora_amd  # noqa: F401
    from hyclora_amd.models import compute_utils
    from hyclora_amd.operators import compress_function, lora_kernels

    class Ns:
        cu, cf, lk = compute_utils, compress_function, lora_kernels
    return Ns


def randn(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).to(BF16).cuda()


# rows: one, around a step of 16, around the 64 rows of a sum of the second product, around strips of 128 and 256 and one plane
@pytest.mark.parametrize("T", [1, 15, 17, 63, 64, 65, 127, 129, 255, 256, 257, 385, 513])
@pytest.mark.parametrize("N,R", [(32, 2), (128, 16), (480, 6), (512, 16), (544, 20), (1056, 64)])
def test_edges_against_float64(M, T, N, R):
    g = torch.Generator().manual_seed(T * 1000 + N + R)
    x, u, v = randn(g, T, N), randn(g, T, R), randn(g, R, N, scale=0.1)
    p1, p2 = M.lk.lora_products(x, u, v)
    d = lambda t: t.double().cpu()
    assert_close_bf16(p1.cpu(), (d(u).t() @ d(x)).to(BF16), what="u^T x")
    assert_close_bf16(p2.cpu(), (d(x) @ d(v).t()).to(BF16), what="x v^T")
    t1, t2 = M.lk.lora_products(x, u, v.t().contiguous().t(), p1_transposed=True)
    assert torch.equal(t1.t(), p1) and torch.equal(t2, p2)


# every height of a strip at rows that leave a short last one, one and several planes; and by size (0) at 64, 128 and 256 rows
@pytest.mark.parametrize("T,N,R,strip", [(T, N, R, s) for T in (65, 257, 513, 777) for N, R in ((544, 20), (1056, 16)) for s in (64, 128, 192, 256)]
                         + [(321, 1056, 16, 0), (1030, 4128, 16, 0), (2041, 10272, 16, 0)])
def test_strip_heights(M, T, N, R, strip):
    from hyclora_amd import _lib
    g = torch.Generator().manual_seed(T + N + strip)
    x, u, v = randn(g, T, N), randn(g, T, R), randn(g, R, N, scale=0.1)
    s = M.cf.get_statistics_only_quant(x[None], 4, "per-channel")
    q = M.cf.compression_pack_quant_base(x[None], 4, "per-channel", 1, 1, {"scale": s})[0]
    dense = M.cf.decompression_dequantization(q, s, 4)[0]
    d = lambda t: t.double()   # noqa: E731
    try:
        _lib.set_tuning("contract_strip_rows", strip)
        p1, p2 = M.lk.lora_products(x, u, v)
        coded = M.lk.lora_product_from_codes(q, s, u[None], None, 4)
        with torch.no_grad():
            members = [(randn(g, R, N, scale=0.1).t(), v, u[None], x[None])] * 2 if R <= 16 else None
            group = members and M.cu._lib.native().lora_products_shared(members, None, q, s, None, 4)
            single = M.lk.lora_product_from_codes(q, s, group[0][2], None, 4) if group else None
    finally:
        _lib.set_tuning("contract_strip_rows", 0)
    assert_close_bf16(p1.cpu(), (d(u).t() @ d(x)).to(BF16).cpu(), what="u^T x")
    assert_close_bf16(p2.cpu(), (d(x) @ d(v).t()).to(BF16).cpu(), what="x v^T")
    assert_close_bf16(coded.cpu(), (d(u).t() @ d(dense)).to(BF16).cpu(), what="u^T x from codes")
    for ga, gb, mid in group or ():
        assert torch.equal(mid[0], p2) and torch.equal(gb, p1) and torch.equal(ga.t(), single)


# x A alone: whole rows in a workgroup of 16 rows and turns of 1024 columns, two ahead, up to 4096 columns; planes beyond
@pytest.mark.parametrize("T", [1, 15, 16, 17, 64, 200])
@pytest.mark.parametrize("N", [32, 96, 992, 1024, 1056, 2048, 3104, 4096, 4128])
@pytest.mark.parametrize("ranks", [(2,), (16,), (40,), (64,), (16, 16), (8, 8, 8)])
def test_adapter_products_against_float64(M, T, N, ranks):
    g = torch.Generator().manual_seed(T * 1000 + N + sum(ranks))
    x, adapters = randn(g, 1, T, N), [randn(g, r, N, scale=0.1) for r in ranks]
    with torch.no_grad():
        got = M.cu._lib.native().adapter_products(x, [a.t() for a in adapters])
        again = M.cu._lib.native().adapter_products(x, [a.t() for a in adapters])
    for p2, p2_again, a in zip(got, again, adapters):
        assert p2.shape == (1, T, a.shape[0]) and torch.equal(p2, p2_again)
        assert_close_bf16(p2.cpu(), (x.double().cpu() @ a.double().cpu().t()).to(BF16), what="x A")


@pytest.mark.parametrize("T,N,r,lies_kr,library", [
    (1536, 4608, 16, False, False), (1537, 4608, 16, False, True), (2040, 5120, 16, False, True), (4096, 96, 16, False, False), (4097, 96, 16, False, True),
    (2048, 1024, 64, False, False), (2049, 1024, 64, False, True), (1600, 5504, 16, False, False), (300, 768, 16, True, True), (300, 2048, 16, True, False)])
def test_sides_of_the_adapter_rule(M, T, N, r, lies_kr, library):
    """Past the rows, widths and layouts where this package's kernels are the shorter, one adapter is the library's product, bit for bit."""
    g = torch.Generator().manual_seed(T + N)
    x, a = randn(g, 1, T, N), randn(g, r, N, scale=0.1).t()
    a = a.contiguous() if lies_kr else a
    with torch.no_grad():
        got, = M.cu._lib.native().adapter_products(x, [a])
        assert_close_bf16(got.cpu(), (x.double() @ a.double()).to(BF16).cpu(), what="x A")
        if library:
            assert torch.equal(got[0], torch.mm(x[0], a))


def test_rows_past_the_end_do_not_count(M):
    """What lies behind the last row (and right of the last column of a wave's tile) in memory may be anything."""
    g = torch.Generator().manual_seed(1)
    T, N, R = 37, 160, 16
    big = torch.full((T + 200, N), float("nan"), dtype=BF16, device="cuda")
    u_big = torch.full((T + 200, R), float("inf"), dtype=BF16, device="cuda")
    x, u, v = randn(g, T, N), randn(g, T, R), randn(g, R, N, scale=0.1)
    big[:T], u_big[:T] = x, u
    for got, want in zip(M.lk.lora_products(big[:T], u_big[:T], v), M.lk.lora_products(x, u, v)):
        assert torch.equal(got, want) and bool(torch.isfinite(got.float()).all())


@pytest.mark.parametrize("T", [1, 96, 257, 1030])
@pytest.mark.parametrize("widths", [(512, 512), (4096, 1024, 1024), (96, 544, 32)])
@pytest.mark.parametrize("R", [4, 16])
@pytest.mark.parametrize("q_bit", [None, 2, 4, 8])
def test_shared_input_matches_single_calls(M, T, widths, R, q_bit):
    g = torch.Generator().manual_seed(T + sum(widths) + R)
    K = 544
    x = randn(g, 1, T, K)
    codes = None
    if q_bit is not None:
        s = M.cf.get_statistics_only_quant(x, q_bit, "per-channel")
        codes = (M.cf.compression_pack_quant_base(x, q_bit, "per-channel", 1, 1, {"scale": s})[0], s, None, q_bit)
    members = [(randn(g, n, K, scale=0.05), None, randn(g, R, K, scale=0.1).t(), randn(g, n, R, scale=0.1).t(), randn(g, 1, T, R), randn(g, 1, T, n))
               for n in widths]
    with torch.no_grad():
        together = M.cu.lora_backward_shared(members, None if codes else x, codes)
        native = M.cu._lib.native().lora_products_shared([(m[2], m[3], m[4], m[5]) for m in members], None if codes else x,
                                                         *(codes or (None, None, None, 0)))
        assert native is not None                               # the launch that this test is about
        for (w, qs, la, lb, xa, gy), (ga, gb, (gx, mid, at)) in zip(members, together):
            ga1, gb1, (gx1, mid1, at1) = M.cu.lora_backward(w, qs, la, lb, None if codes else x, xa, gy, x_codes=codes, defer_input=True)
            assert torch.equal(ga, ga1) and torch.equal(gb, gb1) and torch.equal(mid, mid1) and torch.equal(gx, gx1) and torch.equal(at, at1)
            assert ga.t().is_contiguous() and gb.t().is_contiguous()


@pytest.mark.parametrize("q_bit", [2, 4, 8])
@pytest.mark.parametrize("T", [1, 300])
def test_shared_input_with_zero_points_matches_single_calls(M, T, q_bit):
    g = torch.Generator().manual_seed(T + q_bit)
    K, R = 544, 16
    x = randn(g, 1, T, K) + 0.5
    s, z = M.cf.get_statistics_only_quant_zero_point(x, q_bit, "per-channel")
    q = M.cf.compression_pack_quant_zp_base(x, q_bit, "per-channel", 1, 1, {"scale": s, "zero_point": z})[0]
    z = z.to(BF16)
    members = [(randn(g, n, K, scale=0.05), None, randn(g, R, K, scale=0.1).t(), randn(g, n, R, scale=0.1).t(), randn(g, 1, T, R), randn(g, 1, T, n))
               for n in (512, 96, 1056)]
    with torch.no_grad():
        assert M.cu._lib.native().lora_products_shared([(m[2], m[3], m[4], m[5]) for m in members], None, q, s, z, q_bit) is not None
        for (w, qs, la, lb, xa, gy), (ga, gb, (gx, mid, at)) in zip(members, M.cu.lora_backward_shared(members, None, (q, s, z, q_bit))):
            ga1, gb1, (gx1, mid1, at1) = M.cu.lora_backward(w, qs, la, lb, None, xa, gy, x_codes=(q, s, z, q_bit), defer_input=True)
            assert torch.equal(ga, ga1) and torch.equal(gb, gb1) and torch.equal(mid, mid1) and torch.equal(gx, gx1)


def test_group_refusals(M):
    """What the group does not take goes the way of the single calls: ranks past 16, ranks that differ, one member, host tensors."""
    g = torch.Generator().manual_seed(2)
    native = M.cu._lib.native()
    x = randn(g, 1, 20, 64)
    member = lambda r, n=96, t=20: (randn(g, r, 64).t(), randn(g, n, r).t(), randn(g, 1, t, r), randn(g, 1, t, n))   # noqa: E731
    with torch.no_grad():
        call = lambda ms: native.lora_products_shared(ms, x, None, None, None, 0)   # noqa: E731
        assert call([member(16), member(16)]) is not None
        assert call([member(20), member(20)]) is None and call([member(16), member(8)]) is None and call([member(16)]) is None
        assert call([member(16)] * 4) is None and call([member(16), member(16, t=10)]) is None and call([member(16), member(16, n=80)]) is None
        host = tuple(t.cpu() for t in member(16))
        assert call([member(16), host]) is None
    assert call([member(16), member(16)]) is None                # gradients are to be recorded


class Job(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("x", "q", "scale", "zero_point", "u", "v", "p1", "p2")] + \
               [("N", ctypes.c_int64), ("v_transposed", ctypes.c_int), ("p1_transposed", ctypes.c_int)]


@pytest.mark.parametrize("q_bit", [0, 2, 8])
@pytest.mark.parametrize("zero", [False, True])
def test_jobs_with_an_input_each(M, q_bit, zero):
    """The form of the C entry that no wrapper uses for codes: every job has its X, dense or as codes, of its own width; the bits of single calls."""
    from hyclora_amd import _lib
    g = torch.Generator().manual_seed(q_bit)
    T, R, widths = 300, 12, (96, 1056, 544)
    jobs, want, got, keep = (Job * 3)(), [], [], []
    for job, n in zip(jobs, widths):
        x, u = randn(g, 1, T, n), randn(g, 1, T, R)
        out = torch.empty(n, R, dtype=BF16, device="cuda")
        job.u, job.p1, job.N, job.p1_transposed = u.data_ptr(), out.data_ptr(), n, 1
        if q_bit:
            s, z = M.cf.get_statistics_only_quant_zero_point(x, q_bit, "per-channel")
            z = z.to(BF16) if zero else None
            q = M.cf.compression_pack_quant_zp_base(x, q_bit, "per-channel", 1, 1, {"scale": s, "zero_point": z})[0] if zero \
                else M.cf.compression_pack_quant_base(x, q_bit, "per-channel", 1, 1, {"scale": s})[0]
            s = s.reshape(-1).contiguous()
            job.q, job.scale, job.zero_point = q.data_ptr(), s.data_ptr(), z.data_ptr() if zero else None
            want.append(M.lk.lora_product_from_codes(q, s, u, z, q_bit))
            keep += [s, z, q]
        else:
            job.x = x.data_ptr()
            want.append(M.lk.lora_products(x, u)[0])
        got.append(out)
        keep += [x, u]
    nbytes = max(16, sum(_lib.lib().hyc_lora_contract_workspace(T, n, R, 1, 0) for n in widths))
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    _lib.call("hyc_lora_contract_group", ctypes.addressof(jobs), 3, 0, q_bit, ws.data_ptr(), nbytes, T, R, _lib.stream_of(ws))
    for a, b in zip(got, want):
        assert torch.equal(a.t(), b)
