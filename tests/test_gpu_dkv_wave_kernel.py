"""The dK/dV kernel of head_dim up to 64 (a wave per 32 keys) on calls large enough to take it: lengths around its 32-row steps and
128-key tiles, waves whose keys lie beyond the sequence, rows no sequence covers, against the float64 oracle."""
import numpy as np
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import sb_attn_varlen
from test_gpu_parity import NAMES, tol_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("attend_current,add_remainder", [(False, False), (True, True)])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (64, torch.float16), (50, torch.bfloat16), (8, torch.float16)])
def test_lengths_around_the_tiles(gpu_device, D, dtype, attend_current, add_remainder):
    lengths, pad, H = [1, 31, 32, 33, 95, 96, 97, 127, 128, 129, 160, 257, 417], 40, 72
    T = sum(lengths)
    assert (T + pad) * H >= 100 << 10      # fewer rows x heads take the kernel that splits the rows
    g = torch.Generator().manual_seed(D)
    host = [torch.randn(H, T + pad, D, generator=g).to(dtype) for _ in range(4)] + [torch.randn(H, T + pad, generator=g).to(dtype)]
    q, k, v, do, drem = (t.to(gpu_device) for t in host)
    for t in (q, k, v):
        t.requires_grad_()
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
    o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False, attend_current=attend_current, add_remainder=add_remainder)
    got = (o, rem, *torch.autograd.grad([o, rem], [q, k, v], [do, drem]))
    heads = [0, 35, H - 1]
    d = [t[heads, :T].double() for t in host]
    if add_remainder:
        d[4] = orc.remainder_drem(d[3], d[4], d[2])
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, attend_current=attend_current, do=d[3], drem=d[4], dtype=torch.float64)
    if add_remainder:
        ref = orc.with_remainder(ref, d[2], d[3])
    for n, a, b in zip(NAMES, got, ref):
        tol_check(n, a[heads, :T], b, dtype, f"D={D}")
        assert (a[:, T:] == 0).all(), f"{n}: rows no sequence covers must be zero"
