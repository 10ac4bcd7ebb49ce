"""Projections and input gradients with the product in the same kernel (hyc_lora_gemm) against float64, and against the library's product
with this package's passes around it, at the edges of its tiles of 128 rows and columns and 64 of the contraction."""
import ctypes

import pytest
import torch

from helpers import BF16, assert_close_bf16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import hyclora_amd  # noqa: F401
    from hyclora_amd import _lib
    from hyclora_amd.models import compute_utils
    from hyclora_amd.operators import compress_function, lora_kernels

    class Ns:
        native, cu, cf, lk = _lib.native(), compute_utils, compress_function, lora_kernels
    return Ns


def randn(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).to(BF16).cuda()


def close_to(got, want, addends, what):
    """`got` against the float64 value of the same bf16 operands: each of the roundings on the way to it (product, LoRA product, sums)
    moves it by half a unit of a value no larger than the largest addend, 2^-9 of it."""
    bound = 2.0 ** -9 * len(addends) * torch.stack([a.abs() for a in addends]).amax(0) + 2.0 ** -9 * want.abs() + 1e-6
    excess = ((got.double() - want).abs() - 2 * bound).max().item()
    assert excess <= 0, f"{what}: {excess} past the bound"


def project_operands(g, T, N, K, R):
    return (randn(g, 1, T, K), randn(g, N, K, scale=K ** -0.5), randn(g, R, K, scale=K ** -0.5).t(), randn(g, N, R, scale=0.1).t(),
            randn(g, N, scale=0.1), randn(g, 1, T, N))


@pytest.mark.parametrize("T", [1, 15, 31, 33, 127, 128, 129, 300])
@pytest.mark.parametrize("N,K,R", [(128, 64, 4), (256, 128, 16), (384, 192, 12)])
def test_projection(M, T, N, K, R):
    g = torch.Generator().manual_seed(T + N)
    x, w, la, lb, bias, res = project_operands(g, T, N, K, R)
    d = lambda t: t.double()
    with torch.no_grad():
        (y, xa, none), = M.native.lora_project(x, [(w, la, lb, bias, None)], 0, False, res)
        assert none is None
        main, low = d(x) @ d(w).t(), d(xa) @ d(lb)
        close_to(y, main + d(bias) + low + d(res), [main, main + d(bias), low, main + d(bias) + low], "y")
        assert torch.equal(xa, M.native.adapter_products(x, [la])[0])
        (bare, _, _), = M.native.lora_project(x, [(w, la, lb, None, None)], 0, False, None)
        close_to(bare, main + low, [main, low], "without bias and residual")
        (act, _, _), = M.native.lora_project(x, [(w, la, lb, None, None)], 0, True, None)
        assert_close_bf16(act.cpu(), torch.nn.functional.gelu(bare.float()).to(BF16).cpu(), what="gelu")
        # LoRA B as it lies, [R, N], instead of the transposed view of its weight
        (again, _, _), = M.native.lora_project(x, [(w, la, lb.contiguous(), bias, None)], 0, False, res)
        assert torch.equal(again, y)


@pytest.mark.parametrize("q_bit", [2, 4, 8])
@pytest.mark.parametrize("T", [1, 40, 129, 260])
def test_codes_are_those_of_the_rounded_product(M, T, q_bit):
    """Codes and results of three projections in one launch against the separate passes over the kernel's own frozen part, bit for bit."""
    g = torch.Generator().manual_seed(T + q_bit)
    K, R = 128, 16
    widths = (128, 384, 256)
    x = randn(g, 1, T, K)
    zero = torch.zeros(R, K, dtype=BF16, device="cuda").t()
    with torch.no_grad():
        members, alone = [], []
        for n in widths:
            _, w, la, lb, bias, _ = project_operands(g, T, n, K, R)
            (main, _, _), = M.native.lora_project(x, [(w, zero, lb, bias, None)], 0, False, None)     # x A = 0: the frozen part alone
            s = M.cf.get_statistics_only_quant(main, q_bit, "per-channel").reshape(-1)
            members.append((w, la, lb, bias, s))
            alone.append((main, s))
        for (w, la, lb, bias, s), (y, xa, q), (main, _) in zip(members, M.native.lora_project(x, members, q_bit, False, None), alone):
            want_q, want_y = M.lk.lora_add_quant(main, xa, lb, s, None, q_bit)
            assert torch.equal(q, want_q) and torch.equal(y, want_y)


@pytest.mark.parametrize("T", [1, 33, 128, 200])
@pytest.mark.parametrize("outs,N", [((64,), 128), ((192, 64), 256), ((128, 64, 320), 384)])
@pytest.mark.parametrize("R", [4, 16])
def test_input_gradients(M, T, outs, N, R):
    g = torch.Generator().manual_seed(T + N + R)
    members = [(randn(g, 1, T, k), randn(g, k, N, scale=k ** -0.5), randn(g, 1, T, R), randn(g, R, N, scale=0.1)) for k in outs]
    res = randn(g, 1, T, N)
    d = lambda t: t.double()
    with torch.no_grad():
        for residual in (None, res):
            got = M.native.lora_input_grad(members, residual)
            terms, addends = [], []
            for gy, w, mid, at in members:
                terms.append((d(gy) @ d(w), d(mid) @ d(at)))
                addends += [terms[-1][0], terms[-1][1], sum(a + b for a, b in terms)]
            want = sum(a + b for a, b in terms) + (0 if residual is None else d(res))
            close_to(got, want, addends, "sum of input gradients")
            assert torch.equal(got, M.native.lora_input_grad(members, residual))


@pytest.mark.parametrize("T", [1, 33, 200])
@pytest.mark.parametrize("outs,N,R", [((64,), 128, 16), ((192, 64), 256, 4), ((128, 64, 320), 384, 16)])
def test_additions_are_bf16_ones_in_order(M, T, outs, N, R):
    """The sum of input gradients, bit for bit: the single ones added up in bf16 in their order, then the residual; and a projection's residual."""
    g = torch.Generator().manual_seed(T + N)
    members = [(randn(g, 1, T, k), randn(g, k, N, scale=k ** -0.5), randn(g, 1, T, R), randn(g, R, N, scale=0.1)) for k in outs]
    res = randn(g, 1, T, N)
    with torch.no_grad():
        total = None
        for m in members:
            one = M.native.lora_input_grad([m], None)
            total = one if total is None else total + one
        assert torch.equal(M.native.lora_input_grad(members, None), total)
        assert torch.equal(M.native.lora_input_grad(members, res), total + res)
        x, w, la, lb, bias, res = project_operands(g, T, N, 64, R)
        (bare, _, _), = M.native.lora_project(x, [(w, la, lb, bias, None)], 0, False, None)
        (y, _, _), = M.native.lora_project(x, [(w, la, lb, bias, None)], 0, False, res)
        assert torch.equal(y, res + bare)
        (act, _, _), = M.native.lora_project(x, [(w, la, lb, bias, None)], 0, True, None)
        (act_res, _, _), = M.native.lora_project(x, [(w, la, lb, bias, None)], 0, True, res)
        assert torch.equal(act_res, res + act)


def kinds(t):
    """0 finite, 1 infinite, 2 negative infinite, 3 NaN"""
    t = t.float()
    return t.isposinf().int() + 2 * t.isneginf().int() + 3 * t.isnan().int()


@pytest.mark.parametrize("T", [40, 200])
def test_infinities_and_nan(M, T):
    """They go where the library's product and the passes after it carry them, and nowhere else: rows, columns and tiles keep apart."""
    g = torch.Generator().manual_seed(T)
    N, K, R = 384, 256, 16
    x, w, la, lb, bias, res = project_operands(g, T, N, K, R)
    x[0, 1, 7], x[0, T - 1, K - 1], x[0, 9, 100] = float("nan"), float("inf"), float("-inf")
    w[130, 5], lb[3, 200], bias[383], res[0, 20, 64] = float("inf"), float("-inf"), float("nan"), float("inf")
    s = (torch.rand(N, generator=g) * 0.1 + 0.01).to(BF16).cuda()
    with torch.no_grad():
        main = x @ w.t() + bias
        (y, xa, q), = M.native.lora_project(x, [(w, la, lb, bias, s)], 4, False, None)
        want_q, want = M.lk.lora_add_quant(main, xa, lb, s, None, 4)
        assert torch.equal(kinds(y), kinds(want)) and torch.equal(kinds(xa), kinds(x @ la))
        (main_only, _, _), = M.native.lora_project(x, [(w, la, lb, bias, None)], 0, False, None, True)
        assert torch.equal(kinds(main_only), kinds(main)) and torch.equal(q, M.lk.lora_add_quant(main_only, xa, lb, s, None, 4)[0])
        (y, _, _), = M.native.lora_project(x, [(w, la, lb, bias, None)], 0, False, res)
        assert torch.equal(kinds(y), kinds(M.lk.lora_add(main, xa, lb, residual=res)))
        # input gradients: gy [T, N] W [N, K]
        gy, mid, at = res, xa, la.t().contiguous()
        gx = M.native.lora_input_grad([(gy, w, mid, at)], None)
        assert torch.equal(kinds(gx), kinds(M.lk.lora_add(gy @ w, mid, at)))
        # x A alone: a row's own
        clean = torch.where(x.isfinite(), x, torch.zeros_like(x))
        a, b = M.native.adapter_products(x, [la])[0], M.native.adapter_products(clean, [la])[0]
        rows = x.isfinite().all(-1)
        assert torch.equal(a[rows], b[rows]) and not a[~rows].isfinite().any()


def test_many_tiles_and_the_library(M):
    """Tiles on every XCD, a remainder of workgroups; the library's product of these operands sums in the same order (where it takes another
    one a few results may differ by a rounding)."""
    g = torch.Generator().manual_seed(5)
    T, N, K, R = 1100, 768, 768, 16
    x, w, la, lb, bias, res = project_operands(g, T, N, K, R)
    with torch.no_grad():
        (y, xa, _), = M.native.lora_project(x, [(w, la, lb, bias, None)], 0, False, res)
        want = M.lk.lora_add(x @ w.t() + bias, xa, lb, residual=res)
        assert (y == want).float().mean().item() >= 0.99 and (y.float() - want.float()).norm() <= 2e-3 * want.float().norm()
        gx = M.native.lora_input_grad([(res, w, xa, la.t())], None)
        want = M.lk.lora_add(res @ w, xa, la.t())
        assert (gx == want).float().mean().item() >= 0.99 and (gx.float() - want.float()).norm() <= 2e-3 * want.float().norm()


def test_what_the_kernel_does_not_take(M):
    g = torch.Generator().manual_seed(6)
    ok = lambda T=20, N=128, K=64, R=8: project_operands(g, T, N, K, R)   # noqa: E731

    def call(x, w, la, lb, bias, res, residual=None):
        return M.native.lora_project(x, [(w, la, lb, bias, None)], 0, False, residual)
    with torch.no_grad():
        assert call(*ok()) is not None
        assert call(*ok(N=160)) is None and call(*ok(K=96)) is None and call(*ok(R=20)) is None and call(*ok(N=2048, K=4096)) is None
        x, w, la, lb, bias, res = ok()
        assert call(x.float(), w, la, lb, bias, res) is None and call(x.cpu(), w, la, lb, bias, res) is None
        assert call(x, w.t().contiguous().t(), la, lb, bias, res) is None and call(x, w, la, lb, bias[:64], res) is None
        assert call(x, w, la, lb, bias, res, residual=res[:, :10]) is None and call(x[:, :, ::2], w, la, lb, bias, res) is None
        assert M.native.lora_input_grad([(res, w, randn(g, 1, 20, 8), la.t()[:4])], None) is None
    assert call(*ok()) is None                                 # gradients are to be recorded


@pytest.mark.parametrize("rows,n,k", [(64, 2048, 2048), (64, 512, 8192), (200, 768, 3072), (100, 1024, 4096), (128, 1024, 4096), (300, 1024, 4096), (130, 896, 4160)])
@pytest.mark.parametrize("gradient", [True, False])
def test_contractions_past_the_rule_are_the_librarys(M, rows, n, k, gradient):
    """Both sides of the rule, and that what follows it gives the projection's input gradient either way."""
    ours = k <= 4096 and not (gradient and rows < 128 and k == 4096)          # the last: the kernel of a few rows takes it
    g = torch.Generator().manual_seed(rows + k)
    with torch.no_grad():
        if gradient:
            gy, w, mid, at = randn(g, 1, rows, k), randn(g, k, n, scale=k ** -0.5), randn(g, 1, rows, 16), randn(g, 16, n, scale=0.1)
            done = M.native.lora_input_grad([(gy, w, mid, at)], None)
            lb, x, xa = randn(g, k, 16, scale=0.1).t(), randn(g, 1, rows, n), randn(g, 1, rows, 16)
            _, _, gx = M.cu.lora_backward(w, None, at.t().contiguous(), lb, x, xa, gy)
            _, _, (_, own_mid, _) = M.cu.lora_backward(w, None, at.t().contiguous(), lb, x, xa, gy, defer_input=True)    # gy B^T, rounded
            low = own_mid.double() @ at.double()
            main = gy.double() @ w.double()
            close_to(gx, main + low, [main, low], "input gradient")
        else:
            x, w, la, lb, bias, _ = project_operands(g, rows, n, k, 16)
            done = M.native.lora_project(x, [(w, la, lb, bias, None)], 0, False, None)
    assert (done is not None) == ours


class Member(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("x", "w", "xa", "b", "bias", "residual", "scale", "q", "y")] + \
               [("N", ctypes.c_int64), ("K", ctypes.c_int64), ("b_transposed", ctypes.c_int)]


@pytest.mark.parametrize("T", [1, 130])
def test_several_input_gradients_with_a_bias_each(M, T):
    """A form of the C entry that no wrapper uses: weights as [K, N], no sum, with a bias; against the same weights as [N, K]."""
    from hyclora_amd import _lib
    g = torch.Generator().manual_seed(T)
    members, keep, got, want = (Member * 2)(), [], [], []
    for m, (n, k) in zip(members, ((128, 192), (384, 64))):
        x, w, xa, b, bias, res = randn(g, T, k), randn(g, k, n, scale=k ** -0.5), randn(g, T, 8), randn(g, 8, n, scale=0.1), randn(g, n), randn(g, T, n)
        y = torch.empty(T, n, dtype=BF16, device="cuda")
        m.x, m.w, m.xa, m.b, m.bias, m.residual, m.y, m.N, m.K = *(t.data_ptr() for t in (x, w, xa, b, bias, res, y)), n, k
        one, wt, out = (Member * 1)(), w.t().contiguous(), torch.empty_like(y)
        ctypes.memmove(one, ctypes.addressof(members) + len(got) * ctypes.sizeof(Member), ctypes.sizeof(Member))
        one[0].w, one[0].y = wt.data_ptr(), out.data_ptr()
        _lib.call("hyc_lora_gemm", ctypes.addressof(one), 1, 0, 0, 0, 0, T, 8, _lib.stream_of(x))
        keep += [x, w, xa, b, bias, res, wt]
        got.append(y)
        want.append(out)
    _lib.call("hyc_lora_gemm", ctypes.addressof(members), 2, 1, 0, 0, 0, T, 8, _lib.stream_of(got[0]))
    for a, b in zip(got, want):
        assert torch.equal(a, b)
