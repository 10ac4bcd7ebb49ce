"""NF4 dequantisation at block sizes that are powers of two and not, and at element counts around a lane's, a workgroup's and no chunk."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 8, 10, 2046, 8192, 8198, 24576, 40002])
@pytest.mark.parametrize("blocksize,blocksize2", [(64, 256), (8, 2), (24, 256), (64, 100), (40, 7), (4096, 256)])
@pytest.mark.parametrize("nested", [False, True])
def test_block_sizes(n, blocksize, blocksize2, nested):
    import hyclora_amd  # noqa: F401
    from hyclora_amd.operators import nf4
    g = torch.Generator().manual_seed(n + blocksize)
    packed = torch.randint(0, 256, (n // 2, 1), generator=g, dtype=torch.uint8)
    blocks = -(-n // blocksize)
    table = torch.tensor(nf4.NF4_TABLE)
    if nested:
        absmax, code = torch.randint(0, 256, (blocks,), generator=g, dtype=torch.uint8), torch.linspace(-1, 1, 256)
        absmax2, offset = torch.rand(-(-blocks // blocksize2), generator=g), torch.tensor(0.7)
        qs = nf4.make_quant_state(absmax.cuda(), (n,), blocksize=blocksize, offset=offset.cuda(),
                                  state2=SimpleNamespace(absmax=absmax2.cuda(), code=code.cuda(), blocksize=blocksize2))
        scale = code[absmax.long()] * absmax2.repeat_interleave(blocksize2)[:blocks] + offset
    else:
        scale = torch.rand(blocks, generator=g)
        qs = nf4.make_quant_state(scale.cuda(), (n,), blocksize=blocksize)
    codes = torch.stack([packed[:, 0] >> 4, packed[:, 0] & 15], dim=1).flatten().long()
    want = (table[codes] * scale.repeat_interleave(blocksize)[:n]).to(torch.bfloat16)
    got = nf4.dequantize_nf4(packed.cuda(), qs)
    assert torch.equal(got.reshape(-1).cpu(), want)
