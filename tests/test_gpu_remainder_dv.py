"""dV of o + rem * v: a key's share rem_j * d_o_j is taken from the first rows its tile sweeps, also where a tile's last key is seen by no row."""
import numpy as np
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import sb_attn_varlen
from test_gpu_parity import NAMES, tol_check

pytestmark = pytest.mark.gpu

# Tiles of 32 keys (up to head_dim 64), of 64 (above, short sequences) and of 128: lengths around a whole number of them and one key more.
SHORT, LONG = [1, 31, 32, 33, 64, 65, 127, 128, 129, 193, 321], [1537, 1281, 1025, 1152, 1153]


@pytest.mark.parametrize("attend_current", [False, True])
@pytest.mark.parametrize("H,D,lengths,dtype", [(5, 64, SHORT, torch.bfloat16), (5, 40, SHORT, torch.float16), (3, 128, SHORT, torch.float16),
                                               (3, 100, SHORT, torch.bfloat16), (25, 72, LONG, torch.bfloat16), (25, 105, LONG, torch.float16)])
def test_own_rows_and_last_keys(gpu_device, H, D, lengths, dtype, attend_current):
    T = sum(lengths)
    g = torch.Generator().manual_seed(T + D)
    host = [torch.randn(H, T, D, generator=g).to(dtype) for _ in range(4)] + [torch.randn(H, T, generator=g).to(dtype)]
    q, k, v, do, drem = (t.to(gpu_device) for t in host)
    for t in (q, k, v):
        t.requires_grad_()
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
    o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False, attend_current=attend_current, add_remainder=True)
    got = (o, rem, *torch.autograd.grad([o, rem], [q, k, v], [do, drem]))
    heads = [0, H - 1]
    d = [t[heads].double() for t in host]
    d[4] = orc.remainder_drem(d[3], d[4], d[2])
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, attend_current=attend_current, do=d[3], drem=d[4], dtype=torch.float64)
    for n, a, b in zip(NAMES, got, orc.with_remainder(ref, d[2], d[3])):
        tol_check(n, a[heads], b, dtype, f"H={H} D={D}")
