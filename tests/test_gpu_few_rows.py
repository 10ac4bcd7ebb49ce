"""The product of a few rows with a frozen weight (csrc/few_rows.hip) against the product in 64 bits."""
import ctypes

import pytest
import torch

from hyclora_amd import _lib
from hyclora_amd.models.compute_utils import frozen_matmul


def few_rows(x, w, nk):
    (t, k), n = x.shape, w.shape[0 if nk else 1]
    ws = torch.empty(_lib.lib().hyc_few_rows_workspace(t, n, k), device=x.device, dtype=torch.uint8)
    out = torch.empty(t, n, device=x.device, dtype=torch.bfloat16)
    _lib.call("hyc_few_rows", x.data_ptr(), w.data_ptr(), int(nk), out.data_ptr(), ws.data_ptr(), ws.numel(), t, n, k, _lib.stream_of(out))
    return out


def check(out, x, w):
    """One rounding to bf16 (8 significant bits: 2^-8 relative) of a sum in 32 bits: at most k additions, 2^-24 of the magnitudes
    each."""
    ref, mag = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    assert out.dtype == torch.bfloat16
    assert ((out.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1.01 * x.shape[-1] * 2.0 ** -24 * mag).all()


# one step in all; a step per output block; blocks that start and end inside a workgroup's steps; the widths of the layers
SHAPES = [(128, 64), (640, 64), (128, 4096), (384, 832), (11008, 256), (1024, 4096), (4096, 11008)]


@pytest.mark.gpu
@pytest.mark.parametrize("nk", [True, False])
@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("t", [1, 31, 32, 33, 64, 65, 96, 97, 128])
def test_against_64_bits(t, n, k, nk):
    g = torch.Generator(device="cuda").manual_seed(t + n + k)
    x = torch.randn(t, k, generator=g, device="cuda").bfloat16()
    w = torch.randn((n, k) if nk else (k, n), generator=g, device="cuda").bfloat16()
    out = few_rows(x, w, nk)
    check(out, x, w.t() if nk else w)
    assert torch.equal(out, few_rows(x, w, nk))


@pytest.mark.gpu
@pytest.mark.parametrize("t,k,n,view", [(96, 4096, 4096, True), (96, 4096, 4096, False), (127, 4160, 4096, True), (128, 4096, 4096, False),
                                        (96, 4096, 4160, False), (96, 4100, 4096, False), (3, 11008, 4096, True)])
def test_frozen_matmul(t, k, n, view):
    """Shapes on both sides of the rule, entered as the layers enter them."""
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(1, t, k, generator=g, device="cuda").bfloat16()
    w = torch.randn((n, k) if view else (k, n), generator=g, device="cuda").bfloat16()
    w = w.t() if view else w
    with torch.no_grad():
        out = frozen_matmul(x, w)
    assert out.shape == (1, t, n)
    check(out[0], x[0], w)


def test_shapes_that_are_refused():
    h, fake = _lib.lib(), ctypes.c_void_p(0x1000)                      # nothing is launched
    for t, n, k in ((0, 128, 64), (129, 128, 64), (8, 64, 64), (8, 128, 32), (8, 128, 0), (8, 1 << 17, 1 << 14)):
        assert h.hyc_few_rows_workspace(t, n, k) == 0
        assert h.hyc_few_rows(fake, fake, 1, fake, fake, 1 << 40, t, n, k, None) == -3
    need = h.hyc_few_rows_workspace(8, 128, 64)
    assert h.hyc_few_rows(fake, fake, 1, fake, fake, need - 1, 8, 128, 64, None) < 0
    assert h.hyc_few_rows(ctypes.c_void_p(0x1008), fake, 1, fake, fake, need, 8, 128, 64, None) == -4
    assert h.hyc_few_rows(fake, None, 1, fake, fake, need, 8, 128, 64, None) == -1
