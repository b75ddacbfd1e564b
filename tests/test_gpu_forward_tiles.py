"""The forward whose key tiles come straight into LDS (head_dim 128, enough rows x heads that the split kernels do not take the call), at the
edges of its key tiles (32), rows per wave (32) and query tiles (128), against the float64 oracle on some heads (the bar of
test_gpu_parity.py) and bit for bit against itself; strided rows, attend_current, and with and without recorded products."""
import numpy as np
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import sb_attn_varlen
from test_gpu_parity import tol_check

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 161, 255, 256, 257]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("attend_current,token_major,grad", [(False, False, True), (True, True, False)])
def test_tile_edges_against_oracle(gpu_device, dtype, attend_current, token_major, grad):
    H, T = 48, sum(LENGTHS)
    assert T * H >= 64 << 10
    g = torch.Generator().manual_seed(T)
    host = [torch.randn(H, T, 128, generator=g).to(dtype) for _ in range(3)]
    dev = [(t.transpose(0, 1).contiguous().to(gpu_device).transpose(0, 1) if token_major else t.to(gpu_device)).requires_grad_(grad) for t in host]
    cu = torch.tensor(np.cumsum(LENGTHS), dtype=torch.int32)
    (o, rem), (o2, rem2) = (sb_attn_varlen(*dev, cu.to(gpu_device), max(LENGTHS), zero_start=False, attend_current=attend_current) for _ in range(2))
    assert torch.equal(o, o2) and torch.equal(rem, rem2)
    heads = [0, 1, H - 1]
    ref = orc.varlen_stream(*(t[heads] for t in host), cu, attend_current=attend_current, dtype=torch.float64)
    for name, a, r in zip(("o", "rem"), (o, rem), ref):
        tol_check(name, a.detach()[heads], r, dtype, f"forward tiles {dtype}")
