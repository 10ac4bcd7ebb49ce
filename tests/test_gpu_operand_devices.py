"""Operands left in host memory beside an activation on the GPU are refused before a launch: the kernels would take their host
address for one on the device."""
from types import SimpleNamespace

import pytest
import torch

import hyclora_amd  # noqa: F401
from hyclora_amd.operators import compress_function as cf
from hyclora_amd.operators import lora_kernels as lk
from hyclora_amd.operators import nf4
from hyclora_amd.operators import rmsnorm_kernels as rms

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
B, M, N, R = 2, 8, 512, 16


def refused(call, operands, *names):
    call(**operands)                                        # as they should be
    for name in names:
        with pytest.raises(RuntimeError, match="GPU only"):
            call(**{**operands, name: operands[name].cpu()})


def t(*shape, dtype=BF):
    return torch.zeros(*shape, device="cuda", dtype=dtype)


def test_rotary_tables():
    ops = dict(x=t(B, M, N), xa=t(B, M, R), b=t(R, N), s=t(1, N) + 1, cos=t(1, M, 128), sin=t(1, M, 128))
    refused(lambda x, xa, b, s, cos, sin: lk.lora_add_quant(x, xa, b, s, quantize_bit=4, rope=(cos, sin)), ops, "cos", "sin")
    refused(lambda x, xa, b, s, cos, sin: lk.lora_add_quant_group([dict(x_main=x, xa=xa, b=b, scale=s, rope=(cos, sin))], 4), ops, "cos", "sin")
    ops["x"] = t(B, M, N // 2, dtype=torch.uint8)
    refused(lambda x, xa, b, s, cos, sin: lk.lora_add_restore(x, s, xa, b, quantize_bit=4, rope=(cos, sin)), ops, "cos", "sin")
    refused(lambda x, xa, b, s, cos, sin: lk.lora_add_restore_group([dict(q=x, xa=xa, b=b, scale=s, rope=(cos, sin))], 4), ops, "cos", "sin")


@pytest.mark.parametrize("nested", [True, False])
def test_nf4_block_statistics(nested):
    state2 = SimpleNamespace(absmax=t(1, dtype=torch.float32), code=t(256, dtype=torch.float32), blocksize=256) if nested else None
    ops = dict(w=t(64, 1, dtype=torch.uint8), absmax=t(2, dtype=torch.uint8 if nested else torch.float32))
    refused(lambda w, absmax: nf4.dequantize_nf4(w, nf4.make_quant_state(absmax, (1, 128), state2=state2)), ops, "absmax")


def test_fused_norms():
    idx = torch.tensor([3, 200], device="cuda")
    ops = dict(x=t(B, M, N), w=t(N), sy=t(1, N) + 1, sx=t(1, N) + 1, table=rms.outlier_table(idx, N), a=t(16, N).T)
    refused(lambda x, w, sy, sx, table, a: rms.rmsnorm_forward_compress(x, w, 1e-5, 4, sy, sx, idx, table), ops, "w", "sy", "sx", "table")
    refused(lambda x, w, sy, sx, table, a: rms.rmsnorm_forward_compress(x, w, 1e-5, 4, sy, sx, idx, table, [a]), ops, "w", "sy", "sx", "table", "a")
    ops = dict(dy=t(B, M, N), q=t(B, M, N // 2, dtype=torch.uint8), s=t(1, N) + 1, xo=t(B, M, 2), w=t(N), rstd=t(B * M, dtype=torch.float32),
               table=rms.outlier_table(idx, N))
    refused(lambda dy, q, s, xo, w, rstd, table: rms.rmsnorm_backward_from_codes(dy, q, s, xo, idx, 4, w, rstd, table=table), ops, *ops)


def test_offsets_of_a_map():
    a = t(1, 1, 64, 64) + 1
    idx, val, seg = cf.compress_attention_map(a, 0.5)
    refused(lambda seg: cf.compress_attention_map(a, 0.5, seg), dict(seg=seg), "seg")
    refused(lambda seg: cf.restore_attention_map(idx, val, seg, a.shape), dict(seg=seg), "seg")
