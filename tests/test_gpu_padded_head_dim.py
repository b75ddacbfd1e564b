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
@pytest.mark.parametrize("H,D", [(3, D) for D in (7, 8, 9, 15, 16, 33, 50, 63, 64, 65, 72, 96, 121, 127, 128)] +
                         [(80, D) for D in (9, 50, 65, 72, 96, 121, 127, 128)])
def test_head_dim_between_nans_against_oracle(gpu_device, H, D, dtype, pad, add_remainder, save_carry):
    """3 heads take the kernels that split the keys (and, above 64, key tiles of 64), 80 heads the wide ones."""
    lengths = [1, 31, 64, 65, 129, 200] if H == 3 else [1, 31, 64, 65, 129, 200, 833]
    T = sum(lengths)
    assert H == 3 or T * H >= 100 << 10
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
    heads = [0, H // 2, H - 1]
    assert all(torch.isfinite(t).all() for t in got)
    d = [t[heads].double() for t in host]
    if add_remainder:
        d[4] = orc.remainder_drem(d[3], d[4], d[2])
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, do=d[3], drem=d[4], dtype=torch.float64)
    if add_remainder:
        ref = orc.with_remainder(ref, d[2], d[3])
    for n, a, b in zip(NAMES, got, ref):
        tol_check(n, a[heads], b, dtype, f"H={H} D={D}")


@pytest.mark.parametrize("odd", ["none", "do", "all"])
def test_rows_off_16_bytes_where_the_one_kernel_backward_is_laid_out(gpu_device, odd):
    """A call the one-kernel backward takes if its rows allow it: with a gradient, or everything, at odd addresses the two kernels
    do (and the schedule the forward prepared fits, or is made again)."""
    lengths, H, D, dtype = [2600, 130], 8, 128, torch.bfloat16
    T = sum(lengths)
    g = torch.Generator().manual_seed(7)
    host = [torch.randn(H, T, D, generator=g).to(dtype) for _ in range(4)] + [torch.randn(H, T, generator=g).to(dtype)]

    def placed(t, shift):
        buf = torch.zeros(t.numel() + shift, dtype=dtype, device=gpu_device)
        buf[shift:] = t.to(gpu_device).flatten()
        return buf[shift:].view(t.shape)

    q, k, v = (placed(t, 1 if odd == "all" else 0).requires_grad_() for t in host[:3])
    do = placed(host[3], 0 if odd == "none" else 1)
    cu = torch.tensor(np.cumsum(lengths), dtype=torch.int32)
    o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False)
    got = (o, rem, *torch.autograd.grad([o, rem], [q, k, v], [do, host[4].to(gpu_device)]))
    d = [t[[0, 7]].double() for t in host]
    ref = orc.varlen_stream(d[0], d[1], d[2], cu, do=d[3], drem=d[4], dtype=torch.float64)
    for n, a, b in zip(NAMES, got, ref):
        tol_check(n, a[[0, 7]], b, dtype, f"odd: {odd}")
