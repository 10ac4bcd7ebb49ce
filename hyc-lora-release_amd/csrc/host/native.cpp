// The host side of the operators in native code: argument checks, output and workspace allocation, the library products and
// the launches that one Python wrapper makes, in one call.  A layer step on a short sequence is bound by the host (7B widths,
// one sample of 96 tokens: 1.7 ms of Python, ctypes and torch calls for 0.7 ms of kernels), so what the wrappers do per call
// matters as much as the kernels there.
//
// Every function takes the operands the layers hand over - bf16, contiguous, 16-byte aligned, on the device, of matching
// shapes - and returns nothing when they are anything else; the Python wrapper then converts, copies or refuses them.  No
// state is kept.
#include <torch/extension.h>

#include <ATen/autocast_mode.h>
#include <c10/hip/HIPStream.h>

#include <optional>
#include <tuple>
#include <vector>

#include "../../../include/hyclora.h"

namespace {

using at::Tensor;
using OptT = std::optional<Tensor>;

void check(const char* fn, int rc) {
    if (rc != HYC_OK) {
        pybind11::gil_scoped_acquire gil;
        pybind11::module_::import("hyclora_amd._lib").attr("raise_error")(fn, rc);
    }
}
void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
bool aligned(const Tensor& t, uintptr_t a = 16) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % a == 0; }
bool is_bf(const Tensor& t) { return t.defined() && t.is_cuda() && t.scalar_type() == at::kBFloat16; }
bool plain(const Tensor& t) { return is_bf(t) && t.is_contiguous() && aligned(t); }
bool vec(const Tensor& t, int64_t n) { return plain(t) && t.numel() == n; }            // per-channel vector
// Whether the library's products of these operands may be called from here: not where a gradient is to be recorded, nor where
// autocast makes them products of another type
bool products_are_plain() {
    return !at::GradMode::is_enabled() && !(at::autocast::is_autocast_enabled(at::kCUDA) && at::autocast::get_autocast_dtype(at::kCUDA) != at::kBFloat16);
}
void* ptr(const OptT& t) { return t ? t->data_ptr() : nullptr; }
// Whether operands lie on the GPU of `like`.  Asked wherever a kernel of this package stands in for library calls, which refuse
// operands of several devices: a kernel would take an address of another GPU's memory for one of its own
bool there(const Tensor& t, const Tensor& like) { return t.defined() && t.device() == like.device(); }
bool there(const OptT& t, const Tensor& like) { return !t || there(*t, like); }
template <class... T>
bool together(const Tensor& like, const T&... others) { return (there(others, like) && ...); }
bool bits_ok(int64_t b) { return b == 2 || b == 4 || b == 8; }
bool packed(const Tensor& q, int64_t numel, int64_t bits) {
    return q.defined() && q.is_cuda() && q.scalar_type() == at::kByte && q.is_contiguous() && q.numel() * 8 == numel * bits;
}
Tensor bytes_like(const Tensor& x, int64_t n, int64_t bits) {                            // packed codes of a [B, M, n] tensor
    auto s = x.sizes().vec();
    s.back() = n * bits / 8;
    return at::empty(s, x.options().dtype(at::kByte));
}

// A LoRA operand [R, N]: as it lies, or as the transposed view of an [N, R] weight
struct Lora {
    const void* p = nullptr;
    int transposed = 0;
    int64_t r = 0, n = 0;
    bool ok = false;
    explicit Lora(const Tensor& b) {
        if (!is_bf(b) || b.dim() != 2) return;
        r = b.size(0);
        n = b.size(1);
        if (b.is_contiguous()) ok = aligned(b);
        else if (b.stride(0) == 1 && b.stride(1) == r) { transposed = 1; ok = aligned(b, 8); }
        p = b.data_ptr();
    }
    bool fits(int64_t width) const { return ok && n == width && n % 32 == 0 && r % 4 == 0 && r >= 4 && r <= 64; }
};

// ---- LoRA adds ----------------------------------------------------------------------------------------------------
OptT lora_add(const Tensor& x, const Tensor& xa, const Tensor& b, const OptT& residual, bool inplace) {
    const Lora B(b);
    if (!plain(x) || x.dim() < 1 || !B.fits(x.size(-1)) || x.numel() == 0) return std::nullopt;
    const int64_t rows = x.numel() / B.n;
    if (!plain(xa) || xa.dim() < 1 || xa.size(-1) != B.r || xa.numel() != rows * B.r) return std::nullopt;
    if (residual && (!plain(*residual) || residual->sizes() != x.sizes())) return std::nullopt;
    Tensor y = inplace ? x : at::empty_like(x);
    check("hyc_lora_add", hyc_lora_add(xa.data_ptr(), B.p, B.transposed, x.data_ptr(), ptr(residual), y.data_ptr(), rows, B.n, B.r, stream_of(x)));
    return y;
}

using Term = std::tuple<Tensor, Tensor, Tensor>;          // x, xa, b
OptT lora_add_sum(const std::vector<Term>& terms) {
    if (terms.size() < 2 || terms.size() > 3) return std::nullopt;
    const Tensor& first = std::get<0>(terms[0]);
    if (!plain(first) || first.dim() < 1 || first.numel() == 0) return std::nullopt;
    hyc_lora_sum_member m[3];
    int64_t r = 0, n = first.size(-1), rows = 0;
    for (size_t i = 0; i < terms.size(); ++i) {
        const auto& [x, xa, b] = terms[i];
        const Lora B(b);
        if (!plain(x) || x.sizes() != first.sizes() || !B.fits(n) || B.r > 16 || (i && B.r != r)) return std::nullopt;
        r = B.r;
        rows = x.numel() / n;
        if (!plain(xa) || xa.size(-1) != r || xa.numel() != rows * r) return std::nullopt;
        m[i] = {xa.data_ptr(), B.p, B.transposed, x.data_ptr()};
    }
    check("hyc_lora_add_sum", hyc_lora_add_sum(m, (int)terms.size(), first.data_ptr(), rows, n, r, stream_of(first)));
    return first;
}

struct Rope {                                              // the two angle tables of a rotation
    Tensor cos, sin;
    bool ok = false, fp32 = false;
    Rope(const Tensor& c, const Tensor& s, int64_t seq, int64_t half) {
        auto table = [&](const Tensor& t) {
            Tensor v = t.dim() == 3 && t.size(0) == 1 ? t.squeeze(0) : t;
            const bool good = v.is_cuda() && v.dim() == 2 && v.size(0) > 1 && v.size(0) >= seq && v.size(1) >= half && v.stride(1) == 1 &&
                              v.stride(0) % 8 == 0 && aligned(v);
            return good ? v : Tensor();
        };
        cos = table(c);
        sin = table(s);
        ok = cos.defined() && sin.defined() && cos.scalar_type() == sin.scalar_type() &&
             (cos.scalar_type() == at::kBFloat16 || cos.scalar_type() == at::kFloat);
        fp32 = ok && cos.scalar_type() == at::kFloat;
    }
};

// (x or codes, xa, b, scale, zero point, cos, sin)
using Item = std::tuple<Tensor, Tensor, Tensor, Tensor, OptT, OptT, OptT>;
bool member(const Item& it, int64_t B, int64_t M, int64_t bits, bool restore, bool with_zero, int64_t& rank, std::vector<Rope>& ropes,
            hyc_lora_add_member& m) {
    const auto& [x, xa, b, scale, zero, cos, sin] = it;
    const Lora L(b);
    if (x.dim() != 3 || x.size(0) != B || x.size(1) != M || x.numel() == 0 || !L.fits(L.n)) return false;
    if (restore ? !(packed(x, B * M * L.n, bits) && aligned(x)) : !(plain(x) && x.size(2) == L.n)) return false;
    if (rank && L.r != rank) return false;
    rank = L.r;
    if (!plain(xa) || xa.size(-1) != L.r || xa.numel() != B * M * L.r || !vec(scale, L.n)) return false;
    if (zero.has_value() != with_zero || (zero && !vec(*zero, L.n))) return false;
    m = {};
    m.xa = xa.data_ptr(); m.b = L.p; m.b_transposed = L.transposed; m.scale = scale.data_ptr(); m.zero_point = ptr(zero); m.N = L.n;
    if (restore) m.q = x.data_ptr();
    else m.x = x.data_ptr();
    if (cos) {
        if (!sin || L.n % 128) return false;
        ropes.emplace_back(*cos, *sin, M, 64);
        const Rope& R = ropes.back();
        if (!R.ok) return false;
        m.cos_t = R.cos.data_ptr(); m.sin_t = R.sin.data_ptr(); m.table_is_fp32 = R.fp32;
        m.seq_len = M; m.stride_cos = R.cos.stride(0); m.stride_sin = R.sin.stride(0);
    }
    return true;
}

std::optional<std::vector<std::tuple<Tensor, Tensor>>> lora_add_quant_group(const std::vector<Item>& items, int64_t bits, bool inplace) {
    if (items.empty() || items.size() > 4 || !bits_ok(bits) || std::get<0>(items[0]).dim() != 3) return std::nullopt;
    const int64_t B = std::get<0>(items[0]).size(0), M = std::get<0>(items[0]).size(1);
    const bool with_zero = std::get<4>(items[0]).has_value();
    hyc_lora_add_member m[4];
    std::vector<Rope> ropes;
    ropes.reserve(4);
    int64_t rank = 0;
    for (size_t i = 0; i < items.size(); ++i)
        if (!member(items[i], B, M, bits, false, with_zero, rank, ropes, m[i])) return std::nullopt;
    std::vector<std::tuple<Tensor, Tensor>> out;
    for (size_t i = 0; i < items.size(); ++i) {
        const Tensor& x = std::get<0>(items[i]);
        Tensor y = inplace ? x : at::empty_like(x), q = bytes_like(x, m[i].N, bits);
        m[i].q = q.data_ptr();
        m[i].y = y.data_ptr();
        out.emplace_back(q, y);
    }
    check("hyc_lora_add_quant_group", hyc_lora_add_quant_group(m, (int)items.size(), B * M, rank, (int)bits, stream_of(std::get<0>(items[0]))));
    return out;
}

std::optional<std::vector<Tensor>> lora_add_restore_group(const std::vector<Item>& items, int64_t bits) {
    if (items.empty() || items.size() > 4 || !bits_ok(bits) || std::get<0>(items[0]).dim() != 3) return std::nullopt;
    const int64_t B = std::get<0>(items[0]).size(0), M = std::get<0>(items[0]).size(1);
    const bool with_zero = std::get<4>(items[0]).has_value();
    hyc_lora_add_member m[4];
    std::vector<Rope> ropes;
    ropes.reserve(4);
    int64_t rank = 0;
    for (size_t i = 0; i < items.size(); ++i)
        if (!member(items[i], B, M, bits, true, with_zero, rank, ropes, m[i])) return std::nullopt;
    std::vector<Tensor> out;
    for (size_t i = 0; i < items.size(); ++i) {
        out.push_back(at::empty({B, M, m[i].N}, std::get<1>(items[i]).options()));
        m[i].y = out.back().data_ptr();
    }
    check("hyc_lora_add_restore_group", hyc_lora_add_restore_group(m, (int)items.size(), B * M, rank, (int)bits, stream_of(out[0])));
    return out;
}

// ---- rank-R products ----------------------------------------------------------------------------------------------
// (u^T x, x v^T) of a dense x [.., N] or, the first only, of packed codes [B, M, N * bits / 8]
std::optional<std::tuple<OptT, OptT>> contract(const OptT& x, const OptT& q, const OptT& scale, const OptT& zero, int64_t bits, const OptT& u,
                                               const OptT& v, int64_t n, bool p1_transposed) {
    if (!u && !v) return std::nullopt;
    const Tensor& src = x ? *x : *q;
    if (n <= 0 || n % 32) return std::nullopt;
    int64_t T = 0;
    if (x) {
        if (!plain(*x) || x->size(-1) != n || x->numel() == 0) return std::nullopt;
        T = x->numel() / n;
    } else {
        if (!bits_ok(bits) || !q->is_contiguous() || q->numel() == 0 || (q->numel() * 8) % (n * bits)) return std::nullopt;
        T = q->numel() * 8 / (n * bits);
        if (!packed(*q, T * n, bits) || !aligned(*q) || v || !scale || !vec(*scale, n) || (zero && !vec(*zero, n))) return std::nullopt;
    }
    int64_t r = u ? u->size(-1) : v->size(0);
    if (r % 2 || r < 2 || r > 64) return std::nullopt;
    if (u && (!plain(*u) || u->numel() != T * r)) return std::nullopt;
    const void* vp = nullptr;
    int vt = 0;
    if (v) {
        const Lora V(*v);
        if (!V.ok || V.r != r || V.n != n) return std::nullopt;
        vp = V.p;
        vt = V.transposed;
    }
    const auto o = src.options().dtype(at::kBFloat16);
    const int64_t bytes = hyc_lora_contract_workspace(T, n, r, u.has_value(), v.has_value());
    Tensor ws = at::empty({std::max<int64_t>(bytes, 16)}, src.options().dtype(at::kByte));
    OptT p1, p2;
    if (u) p1 = p1_transposed ? at::empty({n, r}, o) : at::empty({r, n}, o);
    if (v) {
        auto s = src.sizes().vec();
        s.back() = r;
        p2 = at::empty(s, o);
    }
    check("hyc_lora_contract", hyc_lora_contract(ptr(x), x ? nullptr : q->data_ptr(), x ? nullptr : scale->data_ptr(), x ? nullptr : ptr(zero),
                                                 x ? 0 : (int)bits, ptr(u), vp, vt, ptr(p1), p1_transposed, ptr(p2), ws.data_ptr(), ws.numel(), T,
                                                 n, r, stream_of(src)));
    return std::make_tuple(p1, p2);
}

// The rank-R products of projections that share their input x (dense, or codes): member (A, B, x A, grad_y) -> (grad A, grad B,
// grad_y B^T), each the bits of its own contract() calls, in one launch for all grad_y and one that reads x once
using Adapter = std::tuple<Tensor, Tensor, Tensor, Tensor>;
std::optional<std::vector<std::tuple<Tensor, Tensor, Tensor>>> lora_products_shared(const std::vector<Adapter>& members, const OptT& x, const OptT& q,
                                                                                    const OptT& scale, const OptT& zero, int64_t bits) {
    if (!products_are_plain() || members.size() < 2 || members.size() > 3) return std::nullopt;
    const size_t count = members.size();
    int64_t T = 0, r = 0, k = 0, ws_g = 0, ws_x = 0;
    hyc_contract_job g[3] = {}, s[3] = {};
    for (size_t i = 0; i < count; ++i) {
        const auto& [la, lb, xa, grad] = members[i];
        if (!together(std::get<3>(members[0]), la, lb, xa, grad, x, q, scale, zero)) return std::nullopt;
        const Lora L(lb);
        if (!plain(grad) || grad.dim() < 2 || grad.numel() == 0 || !L.fits(grad.size(-1)) || L.r > 16 || (i && L.r != r)) return std::nullopt;
        const int64_t rows = grad.numel() / L.n;
        if ((i && rows != T) || !plain(xa) || xa.size(-1) != L.r || xa.numel() != rows * L.r) return std::nullopt;
        if (!is_bf(la) || la.dim() != 2 || la.size(1) != L.r || (i && la.size(0) != k)) return std::nullopt;
        T = rows; r = L.r; k = la.size(0);
        if (!Lora(la.t()).fits(k)) return std::nullopt;
        g[i].x = grad.data_ptr(); g[i].u = xa.data_ptr(); g[i].v = L.p; g[i].v_transposed = L.transposed; g[i].N = L.n; g[i].p1_transposed = 1;
        ws_g += hyc_lora_contract_workspace(T, L.n, r, 1, 1);
        ws_x += hyc_lora_contract_workspace(T, k, r, 1, 0);
    }
    if (x ? !(plain(*x) && x->size(-1) == k && x->numel() == T * k)
          : !(q && scale && bits_ok(bits) && packed(*q, T * k, bits) && aligned(*q) && vec(*scale, k) && (!zero || vec(*zero, k))))
        return std::nullopt;
    const Tensor& like = std::get<3>(members[0]);
    std::vector<std::tuple<Tensor, Tensor, Tensor>> out;
    for (size_t i = 0; i < count; ++i) {
        auto shape = like.sizes().vec();
        shape.back() = r;
        Tensor ga = at::empty({r, k}, like.options()), gb = at::empty({g[i].N, r}, like.options()), mid = at::empty(shape, like.options());
        g[i].p1 = gb.data_ptr();
        g[i].p2 = mid.data_ptr();
        s[i].u = mid.data_ptr(); s[i].p1 = ga.data_ptr(); s[i].N = k;
        out.emplace_back(ga.t(), gb.t(), mid);
    }
    if (x) s[0].x = x->data_ptr();
    else { s[0].q = q->data_ptr(); s[0].scale = scale->data_ptr(); s[0].zero_point = ptr(zero); }
    const int64_t bytes = std::max<int64_t>(std::max(ws_g, ws_x), 16);
    Tensor ws = at::empty({bytes}, like.options().dtype(at::kByte));
    check("hyc_lora_contract_group", hyc_lora_contract_group(g, (int)count, 0, 0, ws.data_ptr(), bytes, T, r, stream_of(like)));
    check("hyc_lora_contract_group", hyc_lora_contract_group(s, (int)count, 1, x ? 0 : (int)bits, ws.data_ptr(), bytes, T, r, stream_of(like)));
    return out;
}

// ---- products with a frozen weight --------------------------------------------------------------------------------
// Columns of a [rows, cols] product to hand to the library first (0: all in one call).  Its bf16 kernels work on 256 x 256 tiles,
// one per compute unit and round.  Where the tiles fill whole rounds and a remainder, one call spreads the remainder over all
// units along the contraction, which costs up to half of the time again; the whole rounds in one call and the remaining columns in
// another do not.  Measured with the frozen weight as it lies (forward) and transposed (backward), [rows, contraction] x cols,
// us:  4096 x 4096 x 11008: 413 -> 271 and 347 -> 307;  2048 x 4096 x 11008: 160 -> 148, 280 -> 176;  8192 x 4096 x 11008: 645 ->
// 506, 672 -> 579;  8192 x 5120 x 5120: 447 -> 302, 460 -> 339;  8192 x 5120 x 13824: 953 -> 786, 1008 -> 883;  4096 x 2048 x 5504: 90
// -> 78, 99 -> 99;  4096 x 4096 x 14336: 333 -> 335, 384 -> 378.  Left in one call: a single whole round with more than half of
// another behind it (2048 x 5120 x 13824: 207 -> 218, 232 -> 244), and row counts whose tiles do not divide a round (6144 x
// 4096 x 14336: 547 -> 668).
int64_t whole_rounds(int64_t rows, int64_t cols) {
    constexpr int64_t tile = 256, units = 256;
    const int64_t down = (rows + tile - 1) / tile, across = (cols + tile - 1) / tile;
    if (down <= 0 || units % down || down * across <= units) return 0;
    const int64_t rest = down * across % units;
    if (rest == 0 || (down * across < 2 * units && rest > units / 2)) return 0;
    return (across - rest / down) * tile;
}
// A few rows times a weight as it lies [K, N] (input gradients): this package's kernel where it is the faster one.  Measured
// against the library at 96 rows, contraction x outputs, us: 4096 x 1024 15 / 20, 4096 x 4096 19 / 35, 4096 x 11008 32 / 35,
// 5120 x 13824 47 / 48, 11008 x 4096 29 / 85, 13824 x 5120 46 / 114.  Left to the library: contractions under 4096 (2048 x 2048
// 14 / 13, 2048 x 5504 20 / 18).  Both are equally far from 64 bits: at 8 to 128 rows and these shapes 1 to 3 of 10000 results
// of the kernel are not the correctly rounded value, 1 to 5 of the library's.  Two more limits are neither for speed nor for
// accuracy, but because an order of the sums other than the library's moves results that are compared with it:
//  - 128 rows and more (4096 x 4096 21 / 39).  Gradients of layers on 128 tokens are held to an oracle that makes the library's
//    calls.  With the kernel one of them, a norm-weight gradient 8192 wide at 4 bits, leaves its bound: its largest error against
//    64 bits is 1.9e-2 of its largest entry, the oracle's 8.8e-3, the bound twice that (cosines 0.999969 and 0.999973; sums in
//    which the terms of a channel with an outlier nearly cancel);
//  - x W^T (4096 x 4096 18 / 22, 11008 x 4096 30 / 50): its last bits decide codes, so a step in another order has some other
//    codes, and its results move by 2.1 % instead of 0.6.
// (Other sums in an order of their own stay inside every bound: x A and the rank-R gradients move a step's results by 0.2 % at most, through
// the codes that a unit of x A changes now and then.  hyc_lora_gemm keeps the library's order.)
bool few_rows_is_faster(int64_t rows, int64_t k) { return rows < 128 && k >= 4096; }
OptT few_rows(const Tensor& x, const Tensor& w) {                  // x [.., K], w [K, N]
    if (!products_are_plain() || !plain(x) || x.dim() < 2 || x.numel() == 0 || !is_bf(w) || w.dim() != 2 || w.device() != x.device())
        return std::nullopt;
    const int64_t k = w.size(0), n = w.size(1);
    if (x.size(-1) != k || !aligned(w)) return std::nullopt;
    const int64_t rows = x.numel() / k;
    if (w.stride(1) != 1 || w.stride(0) != n || !few_rows_is_faster(rows, k)) return std::nullopt;
    const int64_t bytes = hyc_few_rows_workspace(rows, n, k);
    if (bytes == 0) return std::nullopt;
    auto shape = x.sizes().vec();
    shape.back() = n;
    Tensor out = at::empty(shape, x.options()), ws = at::empty({bytes}, x.options().dtype(at::kByte));
    check("hyc_few_rows", hyc_few_rows(x.data_ptr(), w.data_ptr(), 0, out.data_ptr(), ws.data_ptr(), bytes, rows, n, k, stream_of(x)));
    return out;
}
// x [.., K] times w [K, N], both bf16 and not to be differentiated, where one plain call of the library is not the way
OptT frozen_matmul(const Tensor& x, const Tensor& w) {
    if (!products_are_plain() || !is_bf(x) || !is_bf(w) || x.dim() < 1 || w.dim() != 2 || x.numel() == 0 || x.size(-1) != w.size(0))
        return std::nullopt;
    if (OptT done = few_rows(x, w)) return done;
    const int64_t k = w.size(0), n = w.size(1), rows = x.numel() / k, cut = whole_rounds(rows, n);
    if (cut == 0) return std::nullopt;
    auto shape = x.sizes().vec();
    shape.back() = n;
    const Tensor x2 = x.reshape({rows, k});
    Tensor out = at::empty({rows, n}, x.options());
    Tensor a = out.narrow(1, 0, cut), b = out.narrow(1, cut, n - cut);
    at::mm_out(a, x2, w.narrow(1, 0, cut));
    at::mm_out(b, x2, w.narrow(1, cut, n - cut));
    return out.view(shape);
}
Tensor frozen_product(const Tensor& x, const Tensor& w) {          // x [.., K] contiguous, w [K, N]
    if (OptT done = frozen_matmul(x, w)) return *done;
    auto shape = x.sizes().vec();
    shape.back() = w.size(1);
    return at::mm(x.view({-1, w.size(0)}), w).view(shape);
}
// The input gradient grad_y W of a frozen weight [out, in]
OptT frozen_input_grad(const Tensor& grad_y, const Tensor& w) {
    if (!products_are_plain() || !plain(grad_y) || grad_y.dim() < 2 || grad_y.numel() == 0 || !is_bf(w) || w.dim() != 2 || !w.is_contiguous() ||
        w.size(0) != grad_y.size(-1))
        return std::nullopt;
    return frozen_product(grad_y, w);
}
bool weight_ok(const Tensor& w, int64_t in) { return is_bf(w) && w.dim() == 2 && w.size(1) == in && w.is_contiguous(); }

// Whether x A of `members` adapters [k, r] is for this package's kernels.  Several adapters: always, x is read once ([2048, 4096] 10 / 16 and 12 / 24 us for
// two and three, [8192, 4096] 19 / 26 and 24 / 39).  One, this package / the library, us at 16 ranks:
//  - up to 4096 columns a workgroup has 16 rows to itself: one generation of workgroups, 4096 rows, is the shorter at every width ([4096, 768] 4.3 / 4.8,
//    [2048, 2048] 4.4 / 6.0, [4096, 4096] 7.4 / 12.6), a second is not ([8192, 768] 5.7 / 5.2, [6000, 2048] 7.0 / 6.8, [8192, 4096] 14.1 / 13.7).  Ranks
//    past 16 fill it with half the rows: 64 ranks, [2048, 1024] 5.9 / 6.8, [2048, 4096] 10 / 16, [4096, 2048] 11 / 8, [16384, 1024] 24 / 10;
//  - past that its partial planes cost a second pass, and the library is the shorter where it has its own splits of the contraction, which are
//    those of multiples of 512: [1536, 5120] 7.4 / 7.0, [1536, 8192] 8.7 / 8.8, [1536, 13824] 13.4 / 14.4, but [2048, 5120] 8.7 / 7.1, [2048, 13824] 16.0 /
//    14.8, [4096, 8192] 17 / 14.  Other widths: [4096, 5504] 14 / 21, [2048, 11008] 14 / 26, [4096, 11008] 21 / 28, [4096, 13056] 23 / 31 (6912: 15.7 / 18.9, and
//    16.0 / 13.8 at 4000 rows); 64 ranks [2048, 11008] 25 / 36, [4096, 11008] 40 / 40.
//  - an adapter that lies as [k, r] goes through the planes at any width: [1024, 768] 7.3 / 5.1, [1024, 2048] 7.0 / 6.9, [2048, 4096] 7.7 / 8.4, [2048, 8192] 10 / 14,
//    [2048, 13824] 16 / 18, [4096, 2048] 8.3 / 6.9, [4096, 13824] 24 / 21.
// A call of the library costs the host 10 us more.
bool adapters_are_ours(int64_t rows, int64_t k, int64_t r, bool lies_kr, size_t members) {
    if (k % 32) return false;
    if (members > 1) return true;
    if (lies_kr) return k >= 2048 && rows <= 2048;
    return rows <= (k > 4096 && k % 512 == 0 ? 1536 : r <= 16 ? 4096 : 2048);
}

// x A for one to three adapters [K, R] of one x, from one read of x, where that is the way
std::vector<Tensor> adapter_products(const Tensor& x, const std::vector<Tensor>& adapters) {
    TORCH_CHECK(plain(x) && x.dim() >= 2 && x.numel() > 0, "x must be a contiguous bfloat16 tensor on the GPU");
    const int64_t k = x.size(-1), rows = x.numel() / k;
    for (const Tensor& a : adapters) TORCH_CHECK(is_bf(a) && a.dim() == 2 && a.size(0) == k, "an adapter must be [", k, ", R] bfloat16, got ", a.sizes());
    hyc_contract_job jobs[3] = {};
    int64_t r = 0;
    bool group = !adapters.empty() && adapters.size() <= 3 &&
                 adapters_are_ours(rows, k, adapters[0].size(1), adapters[0].stride(1) == 1, adapters.size());
    for (size_t i = 0; group && i < adapters.size(); ++i) {
        const Tensor v = adapters[i].t();                          // [R, K]
        const Lora V(v);
        group = V.ok && V.n == k && V.r % 2 == 0 && V.r >= 2 && V.r <= (adapters.size() > 1 ? 16 : 64) && (i == 0 || V.r == r) &&
                v.device() == x.device() && (i == 0 || V.transposed == jobs[0].v_transposed);
        r = V.r;
        jobs[i].x = x.data_ptr(); jobs[i].v = V.p; jobs[i].v_transposed = V.transposed; jobs[i].N = k;
    }
    std::vector<Tensor> out;
    auto shape = x.sizes().vec();
    if (!group) {
        for (const Tensor& a : adapters) {
            shape.back() = a.size(1);
            out.push_back(at::mm(x.view({-1, k}), a).view(shape));
        }
        return out;
    }
    shape.back() = r;
    for (size_t i = 0; i < adapters.size(); ++i) {
        out.push_back(at::empty(shape, x.options()));
        jobs[i].p2 = out.back().data_ptr();
    }
    const int64_t bytes = std::max<int64_t>((int64_t)adapters.size() * hyc_lora_contract_workspace(rows, k, r, 0, 1), 16);
    Tensor ws = at::empty({bytes}, x.options().dtype(at::kByte));
    check("hyc_lora_contract_group", hyc_lora_contract_group(jobs, (int)adapters.size(), 1, 0, ws.data_ptr(), bytes, rows, r, stream_of(x)));
    return out;
}

// -> (x W^T, x A)
std::optional<std::tuple<Tensor, Tensor>> lora_parts(const Tensor& w, const Tensor& la, const Tensor& x, const OptT& xa) {
    if (!products_are_plain() || !plain(x) || x.dim() < 2 || x.numel() == 0 || !weight_ok(w, x.size(-1))) return std::nullopt;
    if (!is_bf(la) || la.dim() != 2 || la.size(0) != x.size(-1) || (xa && !is_bf(*xa))) return std::nullopt;
    Tensor main = frozen_product(x, w.t());
    return std::make_tuple(main, xa ? *xa : adapter_products(x, {la})[0]);
}

// -> (x W^T + (x A) B [+ residual], x W^T, x A)
std::optional<std::tuple<Tensor, Tensor, Tensor>> lora_forward(const Tensor& w, const Tensor& la, const Tensor& lb, const Tensor& x,
                                                               const OptT& residual, const OptT& xa) {
    const Lora L(lb);
    if (w.dim() != 2 || !L.fits(w.size(0)) || !plain(x) || x.dim() < 2 || x.numel() == 0 || !is_bf(la) || la.dim() != 2 || la.size(1) != L.r)
        return std::nullopt;
    auto shape = x.sizes().vec();
    const int64_t rows = x.numel() / shape.back();
    shape.back() = L.n;
    if ((residual && !(plain(*residual) && residual->sizes() == at::IntArrayRef(shape))) ||
        (xa && !(plain(*xa) && xa->size(-1) == L.r && xa->numel() == rows * L.r)))
        return std::nullopt;
    auto parts = lora_parts(w, la, x, xa);
    if (!parts) return std::nullopt;
    auto& [main, a] = *parts;
    OptT y = lora_add(main, a, lb, residual, false);
    TORCH_CHECK(y.has_value(), "LoRA operands do not match: x A is ", a.sizes(), ", B is ", lb.sizes(), ", x W^T is ", main.sizes());
    return std::make_tuple(*y, main, a);
}

// ---- projections in one pass, product included ----------------------------------------------------------------------
// Whether hyc_lora_gemm takes a weight W [n, k] (or, as an input gradient, [k, n]) for `rows` rows
bool gemm_weight(const Tensor& w, int64_t rows, int64_t n, int64_t k) {
    return is_bf(w) && w.dim() == 2 && w.is_contiguous() && aligned(w) && n % 128 == 0 && k % 64 == 0 && rows * k < int64_t{1} << 31 &&
           n * k < int64_t{1} << 31;
}
// The operands of one projection of the rows of x: W, B and x A
bool gemm_member(const Tensor& x, const Tensor& w, const Tensor& lb, const Tensor& xa, int64_t rows, int64_t n, int64_t k, const OptT& bias,
                 hyc_gemm_member& m) {
    if (!together(x, w, lb, xa, bias)) return false;
    const Lora L(lb);
    if (!gemm_weight(w, rows, n, k)) return false;
    if (!L.fits(n) || L.r > 16 || !plain(xa) || xa.size(-1) != L.r || xa.numel() != rows * L.r || (bias && !vec(*bias, n))) return false;
    m = {};
    m.w = w.data_ptr(); m.xa = xa.data_ptr(); m.b = L.p; m.b_transposed = L.transposed; m.bias = ptr(bias); m.N = n; m.K = k;
    return true;
}
// Where that kernel is the way: weights of up to 2^22 elements, an encoder's, and contractions of up to 4096.  On the device, us, this
// kernel / the library with the passes it replaces: input gradients [rows, k] x n  [4096, 768] x 768 15 / 22, [4096, 768] x 3072 38 / 41, [4096, 3072] x 768
// 40 / 44, [4096, 4096] x 1024 50 / 49, [2048, 2048] x 2048 31 / 33; projections with bias and codes  [4096, 768] x 3072 40 / 59, [4096, 3072] x 768 49 / 49,
// [4096, 2048] x 2048 50 / 62.  A workgroup walks the whole contraction, 0.65 us for 64 of it, which the library splits where tiles are few: under 192
// tiles of 128 x 128 a long one takes longer here (gradients [256, 768] x 768 14 / 12, [64, 2048] x 2048 27 / 18, [256, 3072] x 768 36 / 18,
// [256, 4096] x 1024 46 / 23; projections [256, 3072] x 768 45 / 25, [256, 4096] x 1024 55 / 32).  It is this kernel's all the same: steps of
// that size wait for the host, and the library's way costs a step 20 to 50 us for a gradient and 100 for a projection (whole steps, both ways
// in turn: encoder of 768 at 32 tokens 897 / 948, of 1024 at 512 tokens 939 / 1105, decoder of 2048 at 64 tokens 1211 / 1228).  Past 4096 it
// is more than that makes up for: [64, 8192] x 512 85 / 18.  The results are the library's bits, but for 3 of 10000 where the library splits the contraction;
// both are equally far from 64 bits.
bool gemm_is_faster(int64_t n, int64_t k) { return n * k <= int64_t{1} << 22 && k <= 4096; }
// Input gradients that few_rows takes, whose calls are as cheap for the host, are its: [96, 4096] x 1024 19 / 46
bool gemm_is_faster_gradient(int64_t rows, int64_t n, int64_t k) { return gemm_is_faster(n, k) && !few_rows_is_faster(rows, k); }

// (W, A, B, bias, steps) of projections of one x -> (y, x A, codes of the frozen part) each: bf16(main + (x A) B), main = bf16(x W^T [+
// bias]); gelu: of that; residual: added to it; steps (all members or none): the codes of main.  main_only: y = main, for a caller that
// needs it before its steps are known
using Projection = std::tuple<Tensor, Tensor, Tensor, OptT, OptT>;
std::optional<std::vector<std::tuple<Tensor, Tensor, OptT>>> lora_project(const Tensor& x, const std::vector<Projection>& members, int64_t bits, bool gelu,
                                                                          const OptT& residual, bool main_only) {
    if (!products_are_plain() || !plain(x) || x.dim() != 3 || x.numel() == 0 || members.empty() || members.size() > 3) return std::nullopt;
    const int64_t k = x.size(-1), rows = x.numel() / k;
    const bool codes = std::get<4>(members[0]).has_value();
    if ((codes && !bits_ok(bits)) || (main_only && (codes || gelu || residual))) return std::nullopt;
    std::vector<Tensor> adapters;
    for (const auto& [w, la, lb, bias, scale] : members) {
        if (!together(x, w, la, lb, bias, scale, residual)) return std::nullopt;
        if (w.dim() != 2 || w.size(1) != k || !gemm_weight(w, rows, w.size(0), k) || !gemm_is_faster(w.size(0), k) ||
            scale.has_value() != codes || (scale && !vec(*scale, w.size(0))))
            return std::nullopt;
        if (!is_bf(la) || la.dim() != 2 || la.size(0) != k || la.size(1) != lb.size(0) || lb.size(0) != std::get<2>(members[0]).size(0)) return std::nullopt;
        if (lb.size(0) > 16 || !Lora(lb).fits(w.size(0)) || (bias && !vec(*bias, w.size(0)))) return std::nullopt;
        adapters.push_back(la);
    }
    auto shape = x.sizes().vec();
    if (residual) {
        shape.back() = std::get<0>(members[0]).size(0);
        if (members.size() != 1 || !plain(*residual) || residual->sizes() != at::IntArrayRef(shape)) return std::nullopt;
    }
    const std::vector<Tensor> xa = adapter_products(x, adapters);
    hyc_gemm_member m[3];
    std::vector<std::tuple<Tensor, Tensor, OptT>> out;
    for (size_t i = 0; i < members.size(); ++i) {
        const auto& [w, la, lb, bias, scale] = members[i];
        if (!gemm_member(x, w, lb, xa[i], rows, w.size(0), k, bias, m[i])) return std::nullopt;
        shape.back() = w.size(0);
        Tensor y = at::empty(shape, x.options());
        OptT q;
        if (scale) {
            q = bytes_like(y, w.size(0), bits);
            m[i].q = q->data_ptr();
            m[i].scale = scale->data_ptr();
        }
        m[i].x = x.data_ptr(); m[i].residual = ptr(residual); m[i].y = y.data_ptr();
        if (main_only) m[i].xa = nullptr;
        out.emplace_back(y, xa[i], q);
    }
    check("hyc_lora_gemm", hyc_lora_gemm(m, (int)members.size(), 0, 0, codes ? (int)bits : 0, gelu, rows, std::get<2>(members[0]).size(0), stream_of(x)));
    return out;
}

// (grad_y, W, grad_y B^T, A^T) of projections that share their input -> the sum of their input gradients, each bf16(grad_y W + (grad_y
// B^T) A^T), in that order [+ residual]
using InputGrad = std::tuple<Tensor, Tensor, Tensor, Tensor>;
OptT lora_input_grad(const std::vector<InputGrad>& members, const OptT& residual) {
    if (!products_are_plain() || members.empty() || members.size() > 3) return std::nullopt;
    const Tensor& first = std::get<0>(members[0]);
    if (!plain(first) || first.dim() < 2 || first.numel() == 0) return std::nullopt;
    const int64_t rows = first.numel() / first.size(-1), n = std::get<1>(members[0]).size(1), r = std::get<3>(members[0]).size(0);
    hyc_gemm_member m[3];
    for (size_t i = 0; i < members.size(); ++i) {
        const auto& [g, w, mid, at_] = members[i];
        if (!together(first, g, residual)) return std::nullopt;
        if (!plain(g) || g.numel() != rows * g.size(-1) || w.dim() != 2 || w.size(0) != g.size(-1) || w.size(1) != n || at_.size(0) != r ||
            !gemm_is_faster_gradient(rows, n, w.size(0)) || !gemm_member(g, w, at_, mid, rows, n, w.size(0), std::nullopt, m[i]))
            return std::nullopt;
        m[i].x = g.data_ptr();
    }
    auto shape = first.sizes().vec();
    shape.back() = n;
    if (residual && !(plain(*residual) && residual->sizes() == at::IntArrayRef(shape))) return std::nullopt;
    Tensor y = at::empty(shape, first.options());
    m[0].y = y.data_ptr();
    m[0].residual = ptr(residual);
    check("hyc_lora_gemm", hyc_lora_gemm(m, (int)members.size(), 1, members.size() > 1, 0, 0, rows, r, stream_of(first)));
    return y;
}

// lora_backward of models/compute_utils.py: -> (grad A, grad B, grad x) or, deferred, (grad A, grad B, (grad_y W, grad_y B^T, A^T))
pybind11::object lora_backward(const Tensor& w, const Tensor& la, const Tensor& lb, const OptT& x, const OptT& q, const OptT& scale,
                               const OptT& zero, int64_t bits, const Tensor& xa, const Tensor& grad_y, const OptT& accumulate, bool defer) {
    const pybind11::object none = pybind11::none();
    const Lora L(lb);
    if (!products_are_plain() || !plain(grad_y) || grad_y.numel() == 0 || !is_bf(w) || w.dim() != 2 || !w.is_contiguous() ||
        w.size(0) != grad_y.size(-1) || !L.fits(w.size(0)) || !plain(xa) || !is_bf(la) || la.dim() != 2 || la.size(0) != w.size(1) ||
        la.size(1) != L.r || w.size(1) % 32)
        return none;
    const Tensor at_ = la.t();                                     // A^T [R, in]
    auto shape_x = grad_y.sizes().vec();
    shape_x.back() = w.size(1);
    if (!Lora(at_).fits(w.size(1)) || (accumulate && !(plain(*accumulate) && accumulate->sizes() == at::IntArrayRef(shape_x)))) return none;
    if (x ? !(plain(*x) && x->size(-1) == w.size(1)) : !(q && scale && vec(*scale, w.size(1)) && (!zero || vec(*zero, w.size(1))))) return none;
    auto both = contract(grad_y, std::nullopt, std::nullopt, std::nullopt, 0, xa, lb, w.size(0), true);
    if (!both) return none;
    const Tensor grad_b = std::get<0>(*both)->t(), grad_mid = *std::get<1>(*both);
    auto ga = x ? contract(x, std::nullopt, std::nullopt, std::nullopt, 0, grad_mid, std::nullopt, w.size(1), false)
                : contract(std::nullopt, q, scale, zero, bits, grad_mid, std::nullopt, w.size(1), false);
    if (!ga) return none;
    const Tensor grad_a = std::get<0>(*ga)->t();
    if (!defer)
        if (OptT done = lora_input_grad({{grad_y, w, grad_mid, at_}}, accumulate)) return pybind11::make_tuple(grad_a, grad_b, *done);
    Tensor grad_x = frozen_product(grad_y, w);
    if (defer) return pybind11::make_tuple(grad_a, grad_b, pybind11::make_tuple(grad_x, grad_mid, at_));
    OptT sum = lora_add(grad_x, grad_mid, at_, accumulate, true);
    TORCH_CHECK(sum.has_value(), "LoRA operands do not match: grad x is ", grad_x.sizes(), ", A^T is ", at_.sizes());
    return pybind11::make_tuple(grad_a, grad_b, *sum);
}

// ---- quantise / dequantise ----------------------------------------------------------------------------------------
std::optional<std::tuple<OptT, Tensor>> quantize(const Tensor& x, const Tensor& s, const OptT& z, const OptT& channel, int64_t bits) {
    if (!plain(x) || x.dim() != 3 || x.numel() == 0 || !bits_ok(bits)) return std::nullopt;
    const int64_t B = x.size(0), M = x.size(1), N = x.size(2);
    if (N % 32 || !vec(s, N) || (z && !vec(*z, N))) return std::nullopt;
    if (channel && !(channel->is_cuda() && channel->scalar_type() == at::kLong && channel->is_contiguous())) return std::nullopt;
    const int64_t k = channel ? channel->numel() : 0;
    Tensor q = bytes_like(x, N, bits);
    OptT kept;
    // a list position without a column reads as zeros: the kernel's work for lists of a usual length
    if (channel) kept = k <= HYC_OUTLIER_ZERO_MAX ? at::empty({B, M, k}, x.options()) : at::zeros({B, M, k}, x.options());
    check("hyc_quant_pack", hyc_quant_pack(x.data_ptr(), s.data_ptr(), ptr(z), q.data_ptr(), k ? (const int64_t*)channel->data_ptr() : nullptr, k,
                                           k ? kept->data_ptr() : nullptr, 0, B, M, N, M * N, N, N, 0, (int)bits, stream_of(x)));
    return std::make_tuple(kept, q);
}

OptT dequantize(const Tensor& q, const Tensor& s, const OptT& z, const OptT& kept, const OptT& channel, int64_t bits) {
    if (!bits_ok(bits) || q.dim() != 3 || q.numel() == 0 || s.dim() < 1) return std::nullopt;
    const int64_t B = q.size(0), M = q.size(1), N = s.size(-1);
    if (N % 32 || !packed(q, B * M * N, bits) || !aligned(q) || !vec(s, N) || (z && !vec(*z, N))) return std::nullopt;
    int64_t k = 0;
    if (channel) {
        k = channel->numel();
        if (!channel->is_cuda() || channel->scalar_type() != at::kLong || !channel->is_contiguous() || !kept || !is_bf(*kept) ||
            !kept->is_contiguous() || kept->dim() != 3 || kept->size(0) != B || kept->size(1) != M || kept->size(2) != k)
            return std::nullopt;
    }
    Tensor x = at::empty({B, M, N}, s.options());
    check("hyc_unpack_dequant", hyc_unpack_dequant(q.data_ptr(), s.data_ptr(), ptr(z), x.data_ptr(), k ? (const int64_t*)channel->data_ptr() : nullptr,
                                                   k, k ? kept->data_ptr() : nullptr, B, M, N, M * N, N, N, 0, (int)bits, stream_of(x)));
    return x;
}

// ---- norms --------------------------------------------------------------------------------------------------------
bool table_ok(const OptT& table, int64_t n) {
    return table && table->is_cuda() && table->scalar_type() == at::kShort && table->numel() == n && table->is_contiguous();
}

// -> (y, rstd, q_y, q_x, x_outlier, [y @ a]) of rmsnorm_forward_compress; k outlier channels, in `table`
using Normed = std::tuple<Tensor, Tensor, OptT, OptT, OptT, std::vector<Tensor>>;
std::optional<Normed> norm_compress(const Tensor& x, const Tensor& w, double eps, int64_t bits, const OptT& scale_y, const OptT& scale_x,
                                    const OptT& table, int64_t k, const std::vector<Tensor>& lora_a) {
    if (!plain(x) || x.dim() != 3 || x.numel() == 0 || !bits_ok(bits) || !plain(w)) return std::nullopt;
    const int64_t n = x.size(2), rows = x.numel() / n;
    if (n % 32 || n > 8192 || w.numel() != n || (scale_y && !vec(*scale_y, n)) || (scale_x && !vec(*scale_x, n))) return std::nullopt;
    if (!scale_x) k = 0;
    if (k && !table_ok(table, n)) return std::nullopt;
    const size_t g = lora_a.size();
    const void* weights[4];
    int64_t ranks[4], blocks = 0;
    if (g) {
        if (g > 4 || n % 512 || rows % 2) return std::nullopt;
        for (size_t i = 0; i < g; ++i) {
            const Tensor& a = lora_a[i];                           // the [N, R] view of a contiguous [R, N] weight
            if (!is_bf(a) || a.dim() != 2 || a.size(0) != n || a.stride(0) != 1 || a.stride(1) != n || a.size(1) < 1 || a.size(1) > 64 || !aligned(a))
                return std::nullopt;
            weights[i] = a.data_ptr();
            ranks[i] = a.size(1);
            blocks += (ranks[i] + 15) / 16;
        }
        if (blocks > 4) return std::nullopt;
    }
    Tensor y = at::empty_like(x), rstd = at::empty({rows}, x.options().dtype(at::kFloat));
    OptT qy, qx, kept;
    if (scale_y) qy = bytes_like(x, n, bits);
    if (scale_x) {
        qx = bytes_like(x, n, bits);
        kept = at::empty({x.size(0), x.size(1), k}, x.options());
    }
    const uint16_t* tab = k ? (const uint16_t*)table->data_ptr() : nullptr;
    void* kp = k ? kept->data_ptr() : nullptr;
    std::vector<Tensor> outs;
    if (g) {
        void* out_p[4];
        for (size_t i = 0; i < g; ++i) {
            outs.push_back(at::empty({x.size(0), x.size(1), ranks[i]}, x.options()));
            out_p[i] = outs.back().data_ptr();
        }
        check("hyc_rmsnorm_fwd_compress_lora",
              hyc_rmsnorm_fwd_compress_lora(x.data_ptr(), w.data_ptr(), y.data_ptr(), (float*)rstd.data_ptr(), rows, n, (float)eps, (int)bits,
                                            ptr(scale_y), ptr(qy), ptr(scale_x), ptr(qx), tab, k, kp, (int)g, weights, ranks, out_p, stream_of(x)));
    } else {
        check("hyc_rmsnorm_fwd_compress",
              hyc_rmsnorm_fwd_compress(x.data_ptr(), w.data_ptr(), 0, y.data_ptr(), (float*)rstd.data_ptr(), rows, n, (float)eps, (int)bits,
                                       ptr(scale_y), ptr(qy), ptr(scale_x), ptr(qx), tab, k, kp, stream_of(x)));
    }
    return Normed(y, rstd, qy, qx, kept, outs);
}

OptT norm_backward_codes(const Tensor& dy, const Tensor& q, const Tensor& scale, const OptT& kept, const OptT& table, int64_t k, int64_t bits,
                         const Tensor& w, const Tensor& rstd, const OptT& residual) {
    if (!plain(dy) || dy.numel() == 0 || !bits_ok(bits)) return std::nullopt;
    const int64_t n = dy.size(-1), rows = dy.numel() / n;
    if (n % 512 || n > 8192 || rows % 2 || !packed(q, rows * n, bits) || !vec(scale, n) || !plain(w) || w.numel() != n) return std::nullopt;
    if (!rstd.is_cuda() || rstd.scalar_type() != at::kFloat || !rstd.is_contiguous() || rstd.numel() != rows) return std::nullopt;
    if (k && (!table_ok(table, n) || !kept || !is_bf(*kept) || !kept->is_contiguous() || kept->numel() != rows * k)) return std::nullopt;
    if (residual && (!plain(*residual) || residual->sizes() != dy.sizes())) return std::nullopt;
    Tensor dx = at::empty_like(dy);
    check("hyc_rmsnorm_bwd_codes",
          hyc_rmsnorm_bwd_codes(dy.data_ptr(), q.data_ptr(), scale.data_ptr(), k ? (const uint16_t*)table->data_ptr() : nullptr, k,
                                k ? kept->data_ptr() : nullptr, (int)bits, w.data_ptr(), 0, (const float*)rstd.data_ptr(), ptr(residual),
                                dx.data_ptr(), rows, n, stream_of(dy)));
    return dx;
}

// ---- element-wise, rotation, gated product ------------------------------------------------------------------------
OptT binary(const std::string& name, const Tensor& a, const Tensor& b) {
    if (!plain(a) || !plain(b) || a.sizes() != b.sizes()) return std::nullopt;
    auto* fn = name == "hyc_silu_bwd" ? hyc_silu_bwd : name == "hyc_silu_mul" ? hyc_silu_mul : name == "hyc_silu_once_mul" ? hyc_silu_once_mul :
               name == "hyc_gelu_bwd" ? hyc_gelu_bwd : nullptr;
    if (!fn) return std::nullopt;
    Tensor o = at::empty_like(a);
    check(name.c_str(), fn(a.data_ptr(), b.data_ptr(), o.data_ptr(), a.numel(), stream_of(a)));
    return o;
}

OptT rope(const Tensor& x, const Tensor& cos, const Tensor& sin, bool backward) {
    if (!is_bf(x) || x.dim() != 4 || x.size(3) % 16 || x.stride(3) != 1 || x.stride(0) % 8 || x.stride(1) % 8 || x.stride(2) % 8 || !aligned(x))
        return std::nullopt;
    const Rope R(cos, sin, x.size(1), x.size(3) / 2);
    if (!R.ok) return std::nullopt;
    check("hyc_rope", hyc_rope(x.data_ptr(), R.cos.data_ptr(), R.sin.data_ptr(), R.fp32, x.size(0), x.size(1), x.size(2), x.size(3), x.stride(0),
                               x.stride(1), x.stride(2), R.cos.stride(0), R.sin.stride(0), backward, stream_of(x)));
    return x;
}

struct Gated {                                             // operands the fused gated product shares between its directions
    bool ok = false;
    int64_t rows = 0, n = 0, r = 0;
    const void *b1 = nullptr, *b2 = nullptr;
    int bt = 0;
    Gated(const Tensor& like, const Tensor& xa1, const Tensor& b1_, const Tensor& s1, const Tensor& xa2, const Tensor& b2_, const Tensor& s2) {
        if (!plain(like) || like.dim() != 3 || like.numel() == 0) return;
        n = like.size(2);
        rows = like.numel() / n;
        const Lora A(b1_), B(b2_);
        if (!A.fits(n) || !B.fits(n) || A.r != B.r || A.transposed != B.transposed) return;
        r = A.r;
        b1 = A.p; b2 = B.p; bt = A.transposed;
        ok = plain(xa1) && plain(xa2) && xa1.size(-1) == r && xa2.size(-1) == r && xa1.numel() == rows * r && xa2.numel() == rows * r && vec(s1, n) &&
             vec(s2, n);
    }
};
std::optional<std::tuple<Tensor, Tensor, Tensor>> gated_forward(const Tensor& xa1, const Tensor& b1, const Tensor& x1, const Tensor& s1,
                                                                const Tensor& xa2, const Tensor& b2, const Tensor& x2, const Tensor& s2, int64_t bits) {
    const Gated G(x1, xa1, b1, s1, xa2, b2, s2);
    if (!G.ok || !plain(x2) || x2.sizes() != x1.sizes() || !bits_ok(bits)) return std::nullopt;
    Tensor q1 = bytes_like(x1, G.n, bits), q2 = bytes_like(x1, G.n, bits), o = at::empty_like(x1);
    check("hyc_lora_silu_mul_fwd", hyc_lora_silu_mul_fwd(xa1.data_ptr(), G.b1, x1.data_ptr(), s1.data_ptr(), xa2.data_ptr(), G.b2, x2.data_ptr(),
                                                         s2.data_ptr(), q1.data_ptr(), q2.data_ptr(), o.data_ptr(), G.rows, G.n, G.r, (int)bits, G.bt,
                                                         stream_of(x1)));
    return std::make_tuple(q1, q2, o);
}
std::optional<std::tuple<Tensor, Tensor, Tensor>> gated_backward(const Tensor& xa1, const Tensor& b1, const Tensor& q1, const Tensor& s1,
                                                                 const Tensor& xa2, const Tensor& b2, const Tensor& q2, const Tensor& s2,
                                                                 const Tensor& grad_o, int64_t bits, bool once) {
    const Gated G(grad_o, xa1, b1, s1, xa2, b2, s2);
    if (!G.ok || !bits_ok(bits) || !packed(q1, G.rows * G.n, bits) || !packed(q2, G.rows * G.n, bits) || !aligned(q1) || !aligned(q2) ||
        q1.dim() != 3 || q1.size(0) != grad_o.size(0) || q1.size(1) != grad_o.size(1) || q2.sizes() != q1.sizes())
        return std::nullopt;
    Tensor o = at::empty_like(grad_o), gg = at::empty_like(grad_o), gu = at::empty_like(grad_o);
    auto* fn = once ? hyc_lora_silu_once_mul_bwd : hyc_lora_silu_mul_bwd;
    check(once ? "hyc_lora_silu_once_mul_bwd" : "hyc_lora_silu_mul_bwd",
          fn(xa1.data_ptr(), G.b1, q1.data_ptr(), s1.data_ptr(), xa2.data_ptr(), G.b2, q2.data_ptr(), s2.data_ptr(), grad_o.data_ptr(), o.data_ptr(),
             gg.data_ptr(), gu.data_ptr(), G.rows, G.n, G.r, (int)bits, G.bt, stream_of(grad_o)));
    return std::make_tuple(o, gg, gu);
}

// The gated product of layers that keep every activation as codes; `steps` of gate, up, fn and the product, in that order
std::optional<std::vector<Tensor>> silu_mul_codes(const Tensor& gate, const Tensor& up, const std::vector<Tensor>& steps, int64_t bits) {
    if (!plain(gate) || !plain(up) || !together(gate, up) || gate.dim() < 2 || gate.sizes() != up.sizes() || !bits_ok(bits) || steps.size() != 4 ||
        gate.numel() == 0)
        return std::nullopt;
    const int64_t n = gate.size(-1);
    if (n % 32) return std::nullopt;
    const void* s[4];
    void* q[4];
    std::vector<Tensor> out;
    for (const Tensor& step : steps)
        if (!together(gate, step) || !vec(step, n)) return std::nullopt;
    for (int k = 0; k < 4; ++k) {
        out.push_back(bytes_like(gate, n, bits));
        s[k] = steps[k].data_ptr();
        q[k] = out[k].data_ptr();
    }
    out.push_back(at::empty_like(gate));
    check("hyc_silu_mul_codes", hyc_silu_mul_codes(gate.data_ptr(), up.data_ptr(), s, q, out[4].data_ptr(), gate.numel() / n, n, (int)bits,
                                                   stream_of(gate)));
    return out;
}
std::optional<std::tuple<Tensor, Tensor>> silu_mul_bwd_codes(const std::vector<Tensor>& codes, const std::vector<Tensor>& steps, const Tensor& grad,
                                                             int64_t bits) {
    if (!plain(grad) || grad.dim() < 2 || grad.numel() == 0 || !bits_ok(bits) || codes.size() != 3 || steps.size() != 3) return std::nullopt;
    const int64_t n = grad.size(-1);
    if (n % 32) return std::nullopt;
    const void *s[3], *q[3];
    for (int k = 0; k < 3; ++k) {
        if (!together(grad, steps[k], codes[k]) || !vec(steps[k], n) || !packed(codes[k], grad.numel(), bits) || !aligned(codes[k])) return std::nullopt;
        s[k] = steps[k].data_ptr();
        q[k] = codes[k].data_ptr();
    }
    Tensor gg = at::empty_like(grad), gu = at::empty_like(grad);
    check("hyc_silu_mul_bwd_codes", hyc_silu_mul_bwd_codes(q, s, grad.data_ptr(), gg.data_ptr(), gu.data_ptr(), grad.numel() / n, n, (int)bits,
                                                           stream_of(grad)));
    return std::make_tuple(gg, gu);
}

// ---- NF4 weights --------------------------------------------------------------------------------------------------
OptT nf4_dequant(const Tensor& packed_w, const Tensor& absmax, const Tensor& code2, const Tensor& absmax2, const OptT& offset, const Tensor& table,
                 int64_t rows, int64_t cols, int64_t blocksize, int64_t blocksize2) {
    const int64_t n = rows * cols;
    auto f32 = [](const Tensor& t) { return t.is_cuda() && t.scalar_type() == at::kFloat && t.is_contiguous(); };
    auto u8 = [](const Tensor& t) { return t.is_cuda() && t.scalar_type() == at::kByte && t.is_contiguous(); };
    if (n <= 0 || blocksize <= 0 || blocksize2 <= 0 || !u8(packed_w) || packed_w.numel() * 2 != n || !u8(absmax) || !f32(code2) || code2.numel() != 256 ||
        !f32(absmax2) || !f32(table) || table.numel() != 16 || (offset && (!f32(*offset) || offset->numel() != 1)))
        return std::nullopt;
    const int64_t blocks = (n + blocksize - 1) / blocksize;
    if (absmax.numel() < blocks || absmax2.numel() < (blocks + blocksize2 - 1) / blocksize2) return std::nullopt;
    Tensor out = at::empty({rows, cols}, packed_w.options().dtype(at::kBFloat16));
    check("hyc_nf4_dequant", hyc_nf4_dequant(packed_w.data_ptr(), absmax.data_ptr(), 1, (const float*)code2.data_ptr(), (const float*)absmax2.data_ptr(),
                                             offset ? (const float*)offset->data_ptr() : nullptr, blocksize2, (const float*)table.data_ptr(), out.data_ptr(),
                                             n, blocksize, stream_of(packed_w)));
    return out;
}

}  // namespace

PYBIND11_MODULE(_native, m) {
    m.def("stream_of", [](const Tensor& t) { return (uintptr_t)stream_of(t); });
    m.def("lora_add", &lora_add);
    m.def("lora_add_sum", &lora_add_sum);
    m.def("lora_add_quant_group", &lora_add_quant_group);
    m.def("lora_add_restore_group", &lora_add_restore_group);
    m.def("contract", &contract);
    m.def("lora_products_shared", &lora_products_shared);
    m.def("adapter_products", &adapter_products);
    m.def("lora_project", &lora_project, pybind11::arg("x"), pybind11::arg("members"), pybind11::arg("bits"), pybind11::arg("gelu"),
          pybind11::arg("residual"), pybind11::arg("main_only") = false);
    m.def("lora_input_grad", &lora_input_grad);
    m.def("frozen_input_grad", &frozen_input_grad);
    m.def("whole_rounds", &whole_rounds);
    m.def("frozen_matmul", &frozen_matmul);
    m.def("lora_parts", &lora_parts);
    m.def("lora_forward", &lora_forward);
    m.def("lora_backward", &lora_backward);
    m.def("quantize", &quantize);
    m.def("dequantize", &dequantize);
    m.def("norm_compress", &norm_compress);
    m.def("norm_backward_codes", &norm_backward_codes);
    m.def("binary", &binary);
    m.def("rope", &rope);
    m.def("gated_forward", &gated_forward);
    m.def("gated_backward", &gated_backward);
    m.def("silu_mul_codes", &silu_mul_codes);
    m.def("silu_mul_bwd_codes", &silu_mul_bwd_codes);
    m.def("nf4_dequant", &nf4_dequant);
}
