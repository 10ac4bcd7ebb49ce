"""Operands that lie on another GPU than the rest.  The native host side hands addresses to kernels where the library's products would refuse such
operands, so it has to see them: every function that takes several operands returns nothing, and the caller goes on to the
library call that raises.  Runs without a GPU: the tensors are host memory that says it is on cuda:0 or cuda:1, and nothing is launched."""
import pytest
import torch

BF16 = torch.bfloat16
_memory = []                                                 # the storages below do not own it


def on(device, *shape, dtype=BF16):
    host = torch.zeros(shape, dtype=dtype)
    _memory.append(host)
    nbytes = host.numel() * host.element_size()
    where = torch.device("cuda", device)
    storage = torch._C._construct_storage_from_data_pointer(host.data_ptr(), where, nbytes)
    meta = dict(size=tuple(shape), stride=host.stride(), dtype=dtype, device=where, storage_offset=0, nbytes=nbytes, data_ptr=host.data_ptr())
    return torch._C._construct_CUDA_Tensor_From_Storage_And_Metadata(meta, storage)


@pytest.fixture(scope="module")
def native():
    import hyclora_amd  # noqa: F401
    from hyclora_amd import _lib
    return _lib.native()


@pytest.fixture(autouse=True)
def no_grad():
    with torch.no_grad():
        yield


T, N, K, R = 8, 128, 64, 16
U8 = torch.uint8


def each_elsewhere(shapes):
    """Operands on cuda:0 but for one on cuda:1, every one in turn (not the first, whose device is the call's)."""
    for other in range(1, len(shapes)):
        yield other, [on(int(i == other), *shape, dtype=dtype) for i, (shape, dtype) in enumerate(shapes)]


def test_projection(native):
    shapes = [((1, T, K), BF16), ((N, K), BF16), ((R, K), BF16), ((N, R), BF16), ((N,), BF16), ((N,), BF16), ((1, T, N), BF16)]
    for other, (x, w, a, b, bias, scale, residual) in each_elsewhere(shapes):
        assert native.lora_project(x, [(w, a.t(), b.t(), bias, scale)], 4, False, residual) is None, other


def test_projections_of_several(native):
    x, w, a, b = on(0, 1, T, K), on(0, N, K), on(0, R, K), on(0, N, R)
    assert native.lora_project(x, [(w, a.t(), b.t(), None, None), (on(1, N, K), a.t(), b.t(), None, None)], 0, False, None) is None


def test_input_gradient(native):
    shapes = [((1, T, K), BF16), ((K, N), BF16), ((1, T, R), BF16), ((R, N), BF16), ((1, T, N), BF16)]
    for other, (g, w, mid, at, residual) in each_elsewhere(shapes):
        assert native.lora_input_grad([(g, w, mid, at)], residual) is None, other
        member = on(0, 1, T, K), on(0, K, N), on(0, 1, T, R), on(0, R, N)
        assert native.lora_input_grad([member, (g, w, mid, at)], residual) is None, other
    whole = tuple(on(1, *shape) for shape, _ in shapes[:4])                 # a member that is all elsewhere
    assert native.lora_input_grad([member, whole], None) is None


@pytest.mark.parametrize("q_bit", [0, 4])
def test_products_of_shared_input(native, q_bit):
    shapes = [((1, T, N), BF16), ((K, R), BF16), ((R, N), BF16), ((1, T, R), BF16)]
    shapes += [((1, T, K * q_bit // 8), U8), ((K,), BF16), ((K,), BF16)] if q_bit else [((1, T, K), BF16)]
    for other, (g, a, b, xa, *x) in each_elsewhere(shapes):
        x = (None, *x, q_bit) if q_bit else (x[0], None, None, None, 0)
        member = on(0, R, K).t(), on(0, R, N), on(0, 1, T, R), on(0, 1, T, N)
        assert native.lora_products_shared([member, (a, b, xa, g)], *x) is None, other
    x = (None, *(on(0, *s, dtype=d) for s, d in shapes[4:]), q_bit) if q_bit else (on(0, 1, T, K), None, None, None, 0)
    whole = on(1, R, K).t(), on(1, R, N), on(1, 1, T, R), on(1, 1, T, N)
    assert native.lora_products_shared([member, whole], *x) is None


def test_gated_codes(native):
    for other, ops in each_elsewhere([((1, T, K), BF16)] * 2 + [((K,), BF16)] * 4):
        assert native.silu_mul_codes(ops[0], ops[1], ops[2:], 4) is None, other
    for other, ops in each_elsewhere([((1, T, K), BF16)] + [((1, T, K // 2), U8)] * 3 + [((K,), BF16)] * 3):
        assert native.silu_mul_bwd_codes(ops[1:4], ops[4:], ops[0], 4) is None, other
