"""head_dims the 16-bit kernels pad, at the edges of the 8-column loads and of the kernels' widths: every row lies between NaN
columns, so a load that reaches past head_dim and a store that does show up; and full widths at odd addresses."""
import numpy as np
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import sb_attn_varlen
from test_gpu_parity import NAMES, tol_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,pad,add_remainder,save_carry", [(torch.bfloat16, 1, False, True), (torch.float16, 3, True, False)])
@pytest.mark.parametrize("D", [7, 8, 9, 15, 16, 33, 50, 63, 64, 65, 72, 96, 121, 127, 128])
def test_head_dim_between_nans_against_oracle(gpu_device, D, dtype, pad, add_remainder, save_carry):
    lengths, H = [1, 31, 64, 65, 129, 200], 3
    T = sum(lengths)
    g = torch.Generator().manual_seed(D)
    host = [torch.randn(H, T, D, generator=g).to(dtype) for _ in range(4)] + [torch.randn(H, T, generator=g).to(dtype)]
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)

    def between_nans(t):
        buf = torch.full((H, T, D + 2 * pad), float("nan"), dtype=dtype, device=gpu_device)
        buf[..., pad:-pad] = t.to(gpu_device)
        return buf[..., pad:-pad]

    q, k, v, do = (between_nans(t) for t in host[:4])
    for t in (q, k, v):
        t.requires_grad_()
    o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False, add_remainder=add_remainder, save_carry=save_carry)
    got = (o, rem, *torch.autograd.grad([o, rem], [q, k, v], [do, host[4].to(gpu_device)]))
    d = [t.double() for t in host]
    if add_remainder:
        d[4] = orc.remainder_drem(d[3], d[4], d[2])
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, do=d[3], drem=d[4], dtype=torch.float64)
    if add_remainder:
        ref = orc.with_remainder(ref, d[2], d[3])
    for n, a, b in zip(NAMES, got, ref):
        tol_check(n, a, b, dtype, f"D={D}")
